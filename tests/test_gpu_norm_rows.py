"""RMSNorm at the edges of its row splits: the widths where the lanes per row change, rows that end
inside a pass, more rows than one pass of the backward's workgroups holds, and operands whose
alignment or strides send them to the one-column kernels, against float64 on the same values.

y and dx: a few float32 roundings of sums over C <= 1024 terms kept per lane (1e-5 relative, 2e-6 of
the row's scale).  dw sums R products; a product's factors carry up to 7 float32 roundings (rstd's sum,
division, root and reciprocal, the product), the lane's sum of its rows up to 8 more here and the
partial row one, all of one sign where rows repeat: 16 of 6e-8, 1e-6 of the sum of the magnitudes.
"""

import pytest
import torch

from ssm_scan import norm

pytestmark = pytest.mark.gpu


def _check(x, w, dy, eps=1e-5):
    x, w = x.detach().requires_grad_(), w.detach().requires_grad_()
    y = norm.rms_norm(x, w, eps)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    x64, w64 = x.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    r = torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + eps)
    y64 = x64 * r * w64
    dx64, dw64 = torch.autograd.grad(y64, (x64, w64), dy.double())
    torch.testing.assert_close(y.detach().double(), y64.detach(), rtol=1e-5, atol=2e-6)
    scale = float((r * dy.double() * w64).detach().abs().max())
    torch.testing.assert_close(dx.double(), dx64, rtol=1e-5, atol=2e-6 * max(scale, 1.0))
    mag = (dy.double() * x64 * r).abs().reshape(-1, x.shape[-1]).sum(0)
    assert bool(((dw.double() - dw64).abs() <= 1e-6 * mag + 1e-7).all())


def _draw(dev, R, C, seed=0):
    g = torch.Generator(device=dev).manual_seed(R * 1031 + C + seed)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    return 2.0 * r(R, C), 1.0 + 0.3 * r(C), r(R, C)


@pytest.mark.parametrize("C", [1, 4, 28, 32, 36, 64, 65, 68, 128, 132, 200, 256, 260, 511, 512, 516, 1020, 1023, 1024])
@pytest.mark.parametrize("R", [1, 5, 16, 131])
def test_widths_and_row_ends(dev, R, C):
    _check(*_draw(dev, R, C))


@pytest.mark.parametrize("R,C", [(131072 + 5, 32), (16384 + 3, 256), (8192 + 1, 512), (4096 + 3, 1024), (16384 + 1, 63),
                                 (4096 + 1, 1001)])
def test_more_rows_than_one_pass(dev, R, C):
    _check(*_draw(dev, R, C))


@pytest.mark.parametrize("C", [64, 256, 1024])
def test_alignment_and_strides(dev, C):
    x, w, dy = _draw(dev, 37, C + 4)
    for o, n in ((1, C), (4, C), (0, C)):                  # column slices: unaligned and aligned rows
        _check(x[:, o:o + n], w[:n], dy[:, o:o + n])
    _check(x[:, :C], w[1:C + 1], dy[:, :C])                # an unaligned weight
    xo = torch.randn(37, C + 1, device=dev)                # an odd row stride
    _check(xo[:, :C], w[:C], dy[:, :C])
    _check(x[:, :C], w[:C], xo[:, :C])
    _check(x[:1, :C].expand(37, C), w[:C], dy[:1, :C].expand(37, C))
    _check(x[:, :C], w[:C], torch.ones((), device=dev).expand(37, C))
