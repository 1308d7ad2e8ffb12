"""GPU: the composed selective scan's kernels at their edges -- lengths around one time tile (64
steps; 16 for float64 Hillis-Steele) and one row lane (8), every state padding and state counts
that fill none, channels that fill no workgroup, storage orders, a broadcast A, channel tiles of
the backward -- against the float64 oracle."""

import pytest
import torch

import ctypes

import ssm_scan
from ssm_scan import _abi
from ssm_scan import scan as S
from test_gpu_scan import ALGOS, _oracle_sel, close, sel_inputs

pytestmark = pytest.mark.gpu


def _run(scan, method, ins, dy, dlast, dtype, d_block=None, prep=lambda name, t: t):
    names = ("x", "delta", "A", "Bm", "Cm", "h0")
    leaves = [None if t is None else prep(n, t.to("cuda", dtype)).detach().requires_grad_()
              for n, t in zip(names, ins)]
    y, last = S.selective_scan(*leaves, method=method, scan=scan, d_block=d_block)
    live = [t for t in leaves if t is not None]
    grads = torch.autograd.grad((y, last), live, (prep("dy", dy.to("cuda", dtype)), dlast.to("cuda", dtype)))
    ry, rlast, rg = _oracle_sel(ins, method, dy, dlast, dtype)
    close(y.detach(), ry, dtype, "y")
    close(last.detach(), rlast, dtype, "last")
    for name, g in zip(("dx", "ddelta", "dA", "dB", "dC", "dh0"), grads):
        close(g, rg[name], dtype, name)


def _problem(B, L, D, N, h0, seed):
    g = torch.Generator().manual_seed(seed)
    return (sel_inputs(B=B, L=L, D=D, N=N, seed=seed, h0=h0), torch.randn(B, L, D, generator=g, dtype=torch.float64),
            torch.randn(B, D, N, generator=g, dtype=torch.float64))


# (L, D, N): L around the row lane and the tile; N of every padding (8, 16, 32, 64) and between; D
# below, at and past the 64 / NP channels of a workgroup
EDGES = [(1, 1, 1), (7, 5, 3), (8, 8, 8), (9, 9, 5), (63, 4, 16), (64, 3, 16), (65, 5, 12), (15, 2, 32), (16, 3, 32),
         (17, 1, 20), (64, 2, 64), (66, 1, 40), (129, 33, 16)]


@pytest.mark.parametrize("edge", EDGES, ids=str)
@pytest.mark.parametrize("scan", ALGOS)
def test_edges_float64(scan, edge):
    L, D, N = edge
    for method, h0 in (("zoh", True), ("bilinear", False), ("euler", True)):
        _run(scan, method, *_problem(2, L, D, N, h0, L + N), torch.float64)


@pytest.mark.parametrize("scan", ALGOS)
@pytest.mark.parametrize("shape", [(3, 70, 6, 16), (1, 150, 17, 8), (2, 65, 4, 48)], ids=str)
def test_edges_float32(scan, shape):
    _run(scan, "zoh", *_problem(*shape, True, 11), torch.float32)


@pytest.mark.parametrize("scan", ALGOS)
def test_storage_orders_and_channel_tiles(scan):
    ins, dy, dlast = _problem(2, 75, 21, 16, True, 5)
    ins = list(ins)
    ins[2] = ins[2][:, :1].expand(-1, 16)       # one decay per channel shared by the states

    def prep(name, t):
        if name in ("x", "dy", "Bm"):            # (B, C, L) storage
            return t.transpose(1, 2).contiguous().transpose(1, 2)
        if name in ("delta", "Cm"):              # a view into a wider row
            return torch.stack([t, t], -1).flatten(2)[..., ::2]
        return t[:, :1].expand(-1, t.shape[1]) if name == "A" else t

    _run(scan, "zoh", ins, dy, dlast, torch.float64, d_block=6, prep=prep)


def _close_norm(got, ref, name):
    """float32 sums of a few hundred terms: 2-norm of the difference within 2e-5 of the result's."""
    got, ref = got.detach().double().cpu(), torch.as_tensor(ref)
    assert bool(torch.isfinite(got).all()), f"{name} is not finite"
    assert float((got - ref).norm()) <= 2e-5 * float(ref.norm()) + 1e-30, (name, float((got - ref).norm()), float(ref.norm()))


def _check_all(scan, method, ins, dy, dlast, ref_ins=None):
    leaves = [None if t is None else t.float().cuda().requires_grad_() for t in ins]
    y, last = S.selective_scan(*leaves, method=method, scan=scan)
    grads = torch.autograd.grad((y, last), [t for t in leaves if t is not None], (dy.float().cuda(), dlast.float().cuda()))
    ry, rlast, rg = _oracle_sel(ref_ins or ins, method, dy, dlast, torch.float32)
    _close_norm(y, ry, "y")
    _close_norm(last, rlast, "last")
    for name, g in zip(("dx", "ddelta", "dA", "dB", "dC", "dh0"), grads):
        _close_norm(g, rg[name], name)


@pytest.mark.parametrize("N", [5, 12, 20, 33])
@pytest.mark.parametrize("scan", ALGOS)
def test_pad_states_with_negative_steps(scan, N):
    """A > 0 and delta < 0 decay; a pad lane of its own decay would grow past float32 within 8 steps."""
    ins, dy, dlast = _problem(2, 75, 6, N, True, N)
    ins = list(ins)
    g = torch.Generator().manual_seed(N)
    ins[1] = -10 - 4 * torch.rand(2, 75, 6, generator=g, dtype=torch.float64)
    ins[2] = 0.005 + 0.015 * torch.rand(6, N, generator=g, dtype=torch.float64)
    _check_all(scan, "zoh", ins, dy, dlast)


@pytest.mark.parametrize("scan", ALGOS)
def test_infinite_input_with_pad_states(scan):
    """An infinite x makes its channel infinite from its step on (all B, C > 0), and nothing else."""
    ins, _, _ = _problem(2, 75, 6, 12, True, 3)
    x, delta, A, Bm, Cm, h0 = (t.float().cuda() for t in ins)
    Bm, Cm, delta = Bm.abs() + 0.1, Cm.abs() + 0.1, delta * 0.1
    want, _ = S.selective_scan(x, delta, A, Bm, Cm, h0, scan=scan)
    x[1, 40, 2] = float("inf")
    y, last = S.selective_scan(x, delta, A, Bm, Cm, h0, scan=scan)
    assert bool(torch.isposinf(y[1, 40:, 2]).all()) and bool(torch.isposinf(last[1, 2]).all())
    want[1, 40:, 2] = y[1, 40:, 2]
    assert torch.equal(y, want)


@pytest.mark.parametrize("L", [70, 128])
@pytest.mark.parametrize("scan", ALGOS)
def test_infinite_decay(scan, L):
    """A = -inf (-exp of a large A_log): the state forgets at once and adds nothing, also where the
    sequence ends inside a time tile.  The oracle takes the largest decays float32 holds for it."""
    ins, dy, dlast = _problem(2, L, 6, 12, True, 9)
    ins, ref = list(ins), list(ins)
    ins[2], ref[2] = ins[2].clone(), ins[2].clone()
    ins[2][1, 3], ins[2][4] = -float("inf"), -float("inf")
    ref[2][1, 3], ref[2][4] = -1e38, -1e38
    _check_all(scan, "zoh", ins, dy, dlast, ref)


def test_operand_spans_up_to_2_gib():
    """64 steps of a batch row may span up to 2^31 bytes, the last elements included; a view that spans
    more is copied."""
    ins, dy, dlast = _problem(1, 64, 3, 5, False, 21)
    x, delta, A, Bm, Cm, _ = (None if t is None else t.float().cuda() for t in ins)
    store = torch.empty((1 << 29) + 1, device="cuda")
    for s2 in (134217726, 134217727, 134217728):   # one B for every step; its last state starts 32,
        Bs = store[:4 * s2 + 1].as_strided((1, 64, 5), (0, 0, s2))  # 16 and 0 bytes below 2^31
        store[:4 * s2 + 1:s2] = Bm[0, 0]
        res = []
        for v in (Bm[:, :1].expand(1, 64, 5).contiguous(), Bs):
            leaves = [x.clone().requires_grad_(), v.detach().requires_grad_()]
            y, last = S.selective_scan(leaves[0], delta, A, leaves[1], Cm, scan="chunked")
            res.append((y, last, *torch.autograd.grad((y, last), leaves, (dy.float().cuda(), dlast.float().cuda()))))
        for got, want in zip(res[1], res[0]):
            assert torch.equal(got, want)


# Time segments of the chunked algorithm (from 1024 steps, up to 256 workgroups): whole and ragged last
# segments, segments shorter than their eight wavefronts' shares, the most segments, every padding
SEGS = [(1, 1024, 3, 16), (2, 1025, 5, 12), (1, 1087, 9, 3), (3, 1100, 4, 33), (1, 16384, 1, 2), (1, 4200, 70, 16)]


@pytest.mark.parametrize("shape", SEGS, ids=str)
def test_time_segments_float64(shape):
    for method, h0 in (("zoh", True), ("euler", False), ("bilinear", True)):
        _run("chunked", method, *_problem(*shape, h0, 31), torch.float64)


@pytest.mark.parametrize("shape", SEGS, ids=str)
def test_time_segments_float32(shape):
    _check_all("chunked", "zoh", *_problem(*shape, True, 32))


def test_forward_without_workspace_walks_time_whole():
    """ssm_cscan_fwd splits time only with its workspace; without, the sequence is one segment."""
    ins, _, _ = _problem(1, 1300, 5, 16, True, 33)
    x, delta, A, Bm, Cm, h0 = (t.float().cuda() for t in ins)
    y, last = S.selective_scan(x, delta, A, Bm, Cm, h0, scan="chunked")
    y1, last1 = torch.empty_like(y), torch.empty_like(last)
    a = _abi.CscanArgs()
    a.batch, a.seqlen, a.dim, a.dstate, a.algo = 1, 1300, 5, 16, 4
    for name, t in (("x", x), ("delta", delta), ("A", A), ("Bm", Bm), ("Cm", Cm), ("h0", h0), ("y", y1), ("last", last1)):
        setattr(a, name, _abi.view(t))
    lib = _abi.lib()
    assert lib.ssm_cscan_fwd_workspace_bytes(ctypes.byref(a)) > 0
    _abi.check(lib.ssm_cscan_fwd(ctypes.byref(a), _abi.stream_handle(x.device)), "ssm_cscan_fwd")
    _close_norm(y1, y.double().cpu(), "y")
    _close_norm(last1, last.double().cpu(), "last")


@pytest.mark.parametrize("scan", ["chunked", "sequential"])
def test_backward_cuts_channels_to_its_workspace(scan):
    """Without d_block a launch takes the channels whose partials fit 256 MiB: here 64 of 70."""
    ins, dy, dlast = _problem(1, 8192, 70, 64, True, 34)
    leaves = [t.float().cuda().requires_grad_() for t in ins]
    out = []
    for d_block in (None, 16):
        y, last = S.selective_scan(*leaves, scan=scan, d_block=d_block)
        with ssm_scan.KernelTimer() as t:
            out.append(torch.autograd.grad((y, last), leaves, (dy.float().cuda(), dlast.float().cuda())))
        assert len(t.records["ssm_cscan_bwd"]) == (2 if d_block is None else 5)
    for name, got, ref in zip(("dx", "ddelta", "dA", "dB", "dC", "dh0"), *out):
        _close_norm(got, ref.double().cpu(), name)


def test_more_partials_than_a_launch_has_threads():
    """2^25 steps of 33 states are 2^32 sums of dB and dC.  Only the last 64 steps carry anything."""
    ins, dy, _ = _problem(1, 64, 1, 33, False, 35)
    x, delta, A, Bm, Cm = (t.float().cuda() for t in ins[:5])
    dy, L = dy.float().cuda(), 1 << 25

    def tail(t):
        out = torch.zeros(1, L, 1, device="cuda")
        out[:, L - 64:] = t
        return out

    got = []
    for ops, g in (((x, delta, Bm[:, :1].expand(1, 64, 33), Cm[:, :1].expand(1, 64, 33)), dy),
                   ((tail(x), tail(delta), Bm[:, :1].expand(1, L, 33), Cm[:, :1].expand(1, L, 33)), tail(dy))):
        leaves = [t.detach().requires_grad_() for t in (ops[0], ops[1], A, ops[2], ops[3])]
        y, _ = S.selective_scan(*leaves, scan="chunked")
        got.append(torch.autograd.grad(y, leaves, g))
    small, large = got
    for name, a, b in zip(("dx", "ddelta", "dB", "dC"), (small[i] for i in (0, 1, 3, 4)), (large[i] for i in (0, 1, 3, 4))):
        _close_norm(b[:, L - 64:], a.double().cpu(), name)
    _close_norm(large[2], small[2].double().cpu(), "dA")
    assert not bool(large[3][:, :L - 64].any()) and not bool(large[4][:, :L - 64].any())
