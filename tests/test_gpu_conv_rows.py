"""causal_conv1d where its rows and reductions can go wrong: ends of the 8-step blocks and of the
32-step workgroups, channel counts that end inside a workgroup, every width class, the three types,
storage orders, and both splits of the weight gradient's final sum (1024 partial rows), against
torch in float64 on the CPU.

Tolerances: one rounding of the io type on y and dx (float32: sums of at most 8 products and the
SiLU factor, 1e-5); dweight and dbias sum B x L products of magnitude below 4 on average, each within
16 float32 roundings (the SiLU factor's included): 4e-6 B L, and 2e-5 for the largest of few products.
"""

import pytest
import torch
import torch.nn.functional as F

from ssm_scan.conv import causal_conv1d

pytestmark = pytest.mark.gpu


def _ref(x, w, b, act, dy):
    leaves = [t.double().cpu().requires_grad_() for t in (x, w, b)]
    y = F.conv1d(F.pad(leaves[0].transpose(1, 2), (w.shape[1] - 1, 0)), leaves[1].unsqueeze(1), leaves[2],
                 groups=w.shape[0]).transpose(1, 2)
    y = F.silu(y) if act else y
    return [y.detach()] + list(torch.autograd.grad(y, leaves, dy.double().cpu()))


def _view(g, B, L, D, dtype, form, dev):
    """A (B, L, D) tensor in the storage `form` names."""
    if form == "split":       # the first half of an in_proj output
        return torch.randn(B, L, 2 * D, generator=g).to(dev, dtype)[..., :D]
    if form == "offset":      # rows that start at an odd element
        return torch.randn(B, L, D + 2, generator=g).to(dev, dtype)[..., 1:D + 1]
    if form == "odd_rows":    # an odd row stride
        return torch.randn(B, L, D + 1, generator=g).to(dev, dtype)[..., :D]
    if form == "channel":     # (B, D, L) storage
        return torch.randn(B, D, L, generator=g).to(dev, dtype).transpose(1, 2)
    if form == "expanded":    # one row for every batch and step
        return torch.randn(1, 1, D, generator=g).to(dev, dtype).expand(B, L, D)
    if form == "scalar":      # the gradient of a sum
        return torch.ones((), device=dev, dtype=dtype).expand(B, L, D)
    return torch.randn(B, L, D, generator=g).to(dev, dtype)


def _check(dev, B, L, D, W, dtype, act=True, form="split", dform="dense"):
    g = torch.Generator().manual_seed(B + L + D + W)
    x = _view(g, B, L, D, dtype, form, dev)
    w, b = torch.randn(D, W, generator=g).to(dev) * 0.5, torch.randn(D, generator=g).to(dev) * 0.1
    dy = _view(g, B, L, D, dtype, dform, dev)
    leaves = [x.requires_grad_(), w.requires_grad_(), b.requires_grad_()]
    y = causal_conv1d(*leaves, activation=act)
    got = [y.detach()] + list(torch.autograd.grad(y, leaves, dy))
    eps = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for name, a, r in zip(("y", "dx", "dw", "db"), got, _ref(x.detach(), w.detach(), b.detach(), act, dy)):
        a, wsum = a.double().cpu(), name in ("dw", "db")
        err = (a - r).abs()
        assert bool(torch.isfinite(a).all()), name
        lim = 2e-5 + 4e-6 * B * L if wsum else 1e-5 + 1.1 * eps * r.abs()
        assert bool((err <= lim).all()), (name, float(err.max()))


@pytest.mark.parametrize("L", [1, 7, 8, 9, 31, 32, 33, 67])
@pytest.mark.parametrize("D", [64, 65, 190])
def test_block_ends(dev, L, D):
    _check(dev, 3, L, D, 4, torch.float32)


@pytest.mark.parametrize("B", [1023, 1024])
@pytest.mark.parametrize("D,W", [(3, 4), (67, 8)])
def test_final_sum_splits(dev, B, D, W):
    _check(dev, B, 9, D, W, torch.float32)


@pytest.mark.parametrize("W", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_widths_and_types(dev, W, dtype):
    _check(dev, 5, 70, 130, W, dtype, act=W != 2)


@pytest.mark.parametrize("form,dform", [("offset", "dense"), ("odd_rows", "dense"), ("channel", "dense"),
                                        ("split", "offset"), ("split", "channel"), ("expanded", "expanded"),
                                        ("split", "scalar")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_storage_forms(dev, form, dform, dtype):
    _check(dev, 3, 100, 128, 4, dtype, form=form, dform=dform)


def test_infinite_input_stays_within_its_taps(dev):
    """Steps past the end and before the start are dropped, not multiplied by zero."""
    x = torch.randn(64, 131, 256, generator=torch.Generator().manual_seed(1)).to(dev)
    x[:, 130] = float("inf")
    x[:, 0] = float("inf")
    y = causal_conv1d(x, torch.ones(256, 4, device=dev), None, activation=False)
    assert bool(torch.isfinite(y[:, 4:130]).all()) and bool(torch.isinf(y[:, :4]).all())


def test_more_columns_than_a_grid_row_has_threads(dev):
    """2^26 channels x 4 taps and the bias: 16 threads for each of their sums are more than 2^32."""
    D = 1 << 26
    x = torch.arange(D, device=dev, dtype=torch.float32).remainder_(251.0).view(1, 1, D).requires_grad_()
    w, b = torch.ones(D, 4, device=dev).requires_grad_(), torch.zeros(D, device=dev).requires_grad_()
    y = causal_conv1d(x, w, b, activation=False)
    dw, db = torch.autograd.grad(y, (w, b), torch.full_like(y, 2.0))
    assert torch.equal(dw[:, 3], 2 * x.detach().view(D)) and not bool(dw[:, :3].any())
    assert bool((db == 2).all())
