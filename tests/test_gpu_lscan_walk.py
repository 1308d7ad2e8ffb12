"""GPU: the tiled walk of the linear scans at the edges of its tiles -- lengths around one and two
tiles (128 steps; 64 for hillis_steele and for the forward walk with 4 row lanes), widths that
fill no 64-recurrence workgroup, both sides of the chunked algorithm's one-pass rule, the adjoint
with and without h0, strided views, both directions -- against the recurrence in float64."""

import pytest
import torch

from parity import close
from ssm_scan import scan as S

pytestmark = pytest.mark.gpu
ALGOS = list(S.SCANS)


def _ref(a, b, h0, dh, reverse):
    """h, da, db, dh0 of the recurrence, step by step in float64."""
    a, b, dh = (t.double().flip(1) if reverse else t.double() for t in (a, b, dh))
    h = torch.zeros_like(a[:, 0]) if h0 is None else h0.double()
    hp, hs = [], []
    for t in range(a.shape[1]):
        hp.append(h)
        h = a[:, t] * h + b[:, t]
        hs.append(h)
    lam, mu = [], torch.zeros_like(h)
    for t in reversed(range(a.shape[1])):
        lam.append(dh[:, t] + mu)
        mu = a[:, t] * lam[-1]
    lam = torch.stack(lam[::-1], 1)
    out = [torch.stack(hs, 1), lam * torch.stack(hp, 1), lam]
    return [t.flip(1) if reverse else t for t in out] + [mu]


# (B, L, M): one workgroup; ragged; 160 workgroups and one fewer; 512 and 1,024 (4 and 8 row lanes)
# ... and the lengths and widths that change the row lanes: 16, 32 and 64 steps (8, 16 and 32 for
# hillis_steele), 48, 64 and 96 (sequential's one-wavefront forward; 70 columns are not its own), 512
# steps at 512 and 1,024 workgroups
SHORT = [(2, L, M) for L in (3, 8, 9, 16, 17, 31, 32, 33, 48, 49, 64, 65, 96, 97) for M in (64, 70)] + [
    (1, 40, 65600), (4, 80, 8192), (1, 512, 32832), (3, 513, 10944), (1, 130, 98368)]
SHAPES = [(1, 1, 1), (1, 15, 64), (2, 64, 65), (1, 127, 63), (2, 128, 64), (1, 129, 130), (1, 257, 70),
          (1, 63, 10240), (1, 130, 10177), (1, 66, 10176), (2, 70, 16384), (4, 33, 16384)]


@pytest.mark.parametrize("shape", SHAPES + SHORT, ids=str)
@pytest.mark.parametrize("algo", ALGOS)
def test_walk_edges(algo, shape):
    B, L, M = shape
    g = torch.Generator(device="cuda").manual_seed(L * 7 + M)
    a = torch.rand(B, L, M, generator=g, device="cuda") * 0.5 + 0.5
    b, dh = (torch.randn(B, L, M, generator=g, device="cuda") for _ in range(2))
    for h0, reverse in ((torch.randn(B, M, generator=g, device="cuda"), False), (None, True)):
        leaves = [t.detach().requires_grad_() for t in (a, b) + ((h0,) if h0 is not None else ())]
        h = S._scan(algo, *leaves, reverse=reverse)
        grads = torch.autograd.grad(h, leaves, dh)
        refs = _ref(a, b, h0, dh, reverse)
        # da = lambda h_prev: each factor within a few ulps of its largest magnitude, times the other
        da_atol = max(1e-5, 16 * 2.0 ** -24 * refs[0].abs().max().item() * refs[2].abs().max().item())
        for name, got, ref in zip(("h", "da", "db", "dh0"), (h.detach(), *grads), refs):
            close(got, ref, name=name, **({"atol": da_atol} if name == "da" else {}))


@pytest.mark.parametrize("algo", ALGOS)
def test_walk_strided_and_float64(algo):
    g = torch.Generator(device="cuda").manual_seed(3)
    B, L, M = 2, 131, 37
    a = (torch.rand(B, M, L, generator=g, device="cuda", dtype=torch.float64) * 0.5 + 0.5).transpose(1, 2)
    b, dh = (torch.randn(B, L, 2 * M, generator=g, device="cuda", dtype=torch.float64)[..., ::2] for _ in range(2))
    leaves = [t.detach().requires_grad_() for t in (a, b)]
    h = S._scan(algo, *leaves)
    grads = torch.autograd.grad(h, leaves, dh)
    for got, ref in zip((h.detach(), *grads), _ref(a, b, None, dh, False)):
        torch.testing.assert_close(got, ref, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("M", [159 * 64, 159 * 64 + 1])     # three launches and one pass
@pytest.mark.parametrize("chunk", [1, 7, 300])
def test_chunk_sizes_on_both_sides_of_the_one_pass_rule(M, chunk):
    g = torch.Generator(device="cuda").manual_seed(chunk)
    a = torch.rand(1, 67, M, generator=g, device="cuda") * 0.5 + 0.5
    b, dh = (torch.randn(1, 67, M, generator=g, device="cuda") for _ in range(2))
    h0 = torch.randn(1, M, generator=g, device="cuda")
    leaves = [t.detach().requires_grad_() for t in (a, b, h0)]
    h = S.scan_chunked(*leaves, chunk_size=chunk)
    refs = _ref(a, b, h0, dh, False)
    da_atol = max(1e-5, 16 * 2.0 ** -24 * refs[0].abs().max().item() * refs[2].abs().max().item())  # as above
    for name, got, ref in zip(("h", "da", "db", "dh0"), (h.detach(), *torch.autograd.grad(h, leaves, dh)), refs):
        close(got, ref, name=name, **({"atol": da_atol} if name == "da" else {}))


@pytest.mark.parametrize("algo", ["sequential", "blelloch"])
def test_width_cut_into_launches(algo):
    """2^29 recurrences of 8 wavefronts per 64 are 2^32 threads, more than a launch has; they are walked in
    several, 2^28 each: columns around the cuts, with h0."""
    L, M = 3, (1 << 29) + 65
    a = torch.full((1, 1, 1), 0.5, device="cuda").expand(1, L, M)
    b = torch.arange(M, device="cuda", dtype=torch.float32).remainder_(127.0).expand(1, L, M)
    h0 = (torch.arange(M, device="cuda", dtype=torch.float32).remainder_(61.0) - 30).view(1, M).requires_grad_()
    ad = a.detach().requires_grad_()
    h = S.LinearScanFn.apply(ad, b, h0, S._SCAN_ALGO[algo], 0, False)
    da, dh0 = torch.autograd.grad(h, (ad, h0), torch.ones(1, 1, 1, device="cuda").expand(1, L, M))
    cols = torch.cat([torch.arange(70), torch.arange((1 << 28) - 70, (1 << 28) + 70), torch.arange((1 << 29) - 70, M)]).cuda()
    refs = _ref(a[..., cols], b[..., cols], h0.detach()[:, cols], torch.ones(1, L, len(cols), device="cuda"), False)
    for got, ref in ((h.detach()[..., cols], refs[0]), (da[..., cols], refs[1]), (dh0[:, cols], refs[3])):
        torch.testing.assert_close(got.double(), ref, rtol=1e-6, atol=1e-6)   # a few float32 roundings
