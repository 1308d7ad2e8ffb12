"""The reference's scan module (models/scan.py) on the HIP engine.

Same names, signatures, dispatch strings and error classes as models/scan.py, so callers such
as models/mamba.py:120-121 switch by changing the import:

  discretize        models/scan.py:39-55     materialized (a, b) from the ssm_disc kernels
  zoh_matrix        models/scan.py:58-62     dense test helper (torch.linalg on the device)
  scan_sequential   models/scan.py:70-76     \
  scan_hillis_steele models/scan.py:87-98     | ssm_lscan kernels, one per algorithm, each
  scan_blelloch     models/scan.py:101-135    | differentiable through ssm_lscan_bwd
  scan_chunked      models/scan.py:142-165   /
  SCANS, default_chunk, SCAN_ELEMENT_BUDGET, _blocks   models/scan.py:138-190
  SelectiveScanFn   models/scan.py:193-255   discretize -> scan -> contract in one kernel per
                                             direction, backward by recompute + reverse scan
  selective_scan_reference  models/scan.py:264-274   the time loop; runs on the fused engine,
                                             which walks the same recurrence step by step
  selective_scan    models/scan.py:277-299   dispatcher ('triton' and 'auto' select the fused
                                             engine, ssm_scan.hip_scan)

Everything runs on ROCm tensors; a CPU tensor raises RuntimeError (there is no CPU path).
"""

import ctypes

import torch

from . import _abi, plan, profiling
from .hip_scan import METHODS, FusedSelectiveScanFn, _require_gpu, check_operands

DISCRETIZATIONS = ("zoh", "euler", "bilinear")      # models/scan.py:36
SCAN_ELEMENT_BUDGET = plan.SCAN_ELEMENT_BUDGET       # models/scan.py:182
_SCAN_ALGO = {"sequential": 1, "hillis_steele": 2, "blelloch": 3, "chunked": 4}


def default_chunk(L):
    """max(4, 2^ceil(log2 sqrt(L))) (models/scan.py:138-139), computed in exact integers."""
    return plan.default_chunk(L)


def _blocks(shape_bld, N, d_block):
    """The reference's channel tiles of SelectiveScanFn (models/scan.py:185-190); here they plan nothing."""
    return plan.blocks(shape_bld, N, d_block)


def _ct(*ts):
    dt = torch.float32
    for t in ts:
        if t is not None:
            dt = torch.promote_types(dt, t.dtype)
    return dt


def _launch(name, fn, args, dev):
    with _abi.on_device(dev):
        stream = _abi.stream_handle(dev)
        timer = profiling.active()
        end = None if timer is None else timer.begin(name)
        rc = fn(ctypes.byref(args), stream)
        if end is not None:
            end.record()
    _abi.check(rc, name)


# ------------------------------------------------------------------ discretization
class DiscretizeFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, delta, A, Bm, x, method):
        ct = delta.dtype
        Bsz, L, D = x.shape
        N = A.shape[1]
        a = torch.empty((Bsz, L, D, N), dtype=ct, device=x.device)
        b = torch.empty_like(a)
        args = _disc_args(delta, A, Bm, x, method)
        args.a, args.b = a.data_ptr(), b.data_ptr()
        _launch("ssm_disc_fwd", _abi.lib().ssm_disc_fwd, args, x.device)
        ctx.save_for_backward(delta, A, Bm, x)
        ctx.method = method
        return a, b

    @staticmethod
    def backward(ctx, da, db):
        delta, A, Bm, x = ctx.saved_tensors
        dev = x.device
        shape = (*x.shape, A.shape[1])
        if da is None:
            da = torch.zeros(shape, dtype=delta.dtype, device=dev)
        if db is None:
            db = torch.zeros(shape, dtype=delta.dtype, device=dev)
        da, db = da.contiguous(), db.contiguous()
        ddelta, dx = torch.empty_like(delta), torch.empty_like(x)
        dA, dB = torch.empty_like(A), torch.empty_like(Bm)
        args = _disc_args(delta, A, Bm, x, ctx.method)
        args.da, args.db = da.data_ptr(), db.data_ptr()
        args.ddelta, args.dx, args.dA, args.dBm = (_abi.view(t) for t in (ddelta, dx, dA, dB))
        lib = _abi.lib()
        nbytes = lib.ssm_disc_workspace_bytes(ctypes.byref(args))
        if nbytes < 0:
            _abi.check(lib.ssm_disc_check(ctypes.byref(args)), "ssm_disc_bwd")
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
        args.workspace, args.workspace_bytes = ws.data_ptr(), nbytes
        _launch("ssm_disc_bwd", lib.ssm_disc_bwd, args, dev)
        return ddelta, dA, dB, dx, None


def _disc_args(delta, A, Bm, x, method):
    Bsz, L, D = x.shape
    args = _abi.DiscArgs()
    args.batch, args.seqlen, args.dim, args.dstate = Bsz, L, D, A.shape[1]
    args.method = METHODS[method]
    args.dtype = _abi.DTYPE_CODE[delta.dtype]
    args.delta, args.x, args.A, args.Bm = (_abi.view(t) for t in (delta, x, A, Bm))
    return args


def discretize(delta, A, Bm, x, method="zoh"):
    """delta, x: (B, L, D); A: (D, N) with A < 0; Bm: (B, L, N) -> a, b: (B, L, D, N).

    zoh a = exp(dA), b = expm1(dA)/A * B x; euler b = delta B x; bilinear (Tustin)
    a = (1 + dA/2)/(1 - dA/2), b = delta/(1 - dA/2) B x (models/scan.py:39-55).
    Differentiable in all four tensors."""
    if method not in DISCRETIZATIONS:
        raise ValueError(f"unknown discretization {method!r}")
    check_operands(x, delta, A, Bm, Bm, None, None, None, None)  # the kernels index by (B, L, D, N)
    ct = _ct(delta, A, Bm, x)
    return DiscretizeFn.apply(delta.to(ct), A.to(ct), Bm.to(ct), x.to(ct), method)


def zoh_matrix(A, B, delta):
    """Dense ZOH (models/scan.py:58-62): Ad = expm(A delta), Bd = A^{-1}(Ad - I) B.
    A test helper for general (non-diagonal) A; uses the device's linear-algebra library."""
    Ad = torch.matrix_exp(A * delta)
    eye = torch.eye(A.shape[0], dtype=A.dtype, device=A.device)
    return Ad, torch.linalg.solve(A, (Ad - eye) @ B)


# ------------------------------------------------------------------ linear scans
class LinearScanFn(torch.autograd.Function):
    """h = scan(a, b, h0) on (B, L, M) with a chosen algorithm; backward via ssm_lscan_bwd."""

    @staticmethod
    def forward(ctx, a, b, h0, algo, chunk, reverse):
        cfg = (algo, int(chunk or 0), bool(reverse))
        h = _abi.host().lscan_forward(a, b, h0, *cfg, profiling.active())
        ctx.save_for_backward(a, h0, h)
        ctx.cfg = cfg
        return h

    @staticmethod
    def backward(ctx, dh):
        a, h0, h = ctx.saved_tensors
        da, db, dh0 = _abi.host().lscan_backward(a, h0, h, dh, *ctx.cfg, ctx.needs_input_grad[2], profiling.active())
        return da, db, dh0, None, None, None


def _scan(name, a, b, h0=None, chunk_size=None, reverse=False):
    """a, b (B, L, *rest), h0 (B, *rest) -> h (B, L, *rest) by the named algorithm."""
    _require_gpu(a, b, h0)
    if a.shape != b.shape or a.dim() < 2:
        raise ValueError(f"a and b must share a (B, L, ...) shape, got {tuple(a.shape)} and {tuple(b.shape)}")
    if h0 is not None and (tuple(h0.shape) != (a.shape[0],) + tuple(a.shape[2:])):
        raise ValueError(f"h0 must have shape {(a.shape[0],) + tuple(a.shape[2:])}, got {tuple(h0.shape)}")
    shape = a.shape
    Bsz, L = shape[:2]
    M = 1
    for s in shape[2:]:
        M *= s
    ct = _ct(a, b, h0)
    a3 = a.to(ct).reshape(Bsz, L, M)
    b3 = b.to(ct).reshape(Bsz, L, M)
    h03 = None if h0 is None else h0.to(ct).reshape(Bsz, M)
    h = LinearScanFn.apply(a3, b3, h03, _SCAN_ALGO[name], chunk_size, reverse)
    return h.reshape(shape).to(b.dtype)


def scan_sequential(a, b, h0=None):
    """h_t = a_t h_{t-1} + b_t, one lane per recurrence (models/scan.py:70-76)."""
    return _scan("sequential", a, b, h0)


def scan_hillis_steele(a, b, h0=None):
    """Recursive-doubling inclusive scan (models/scan.py:87-98)."""
    return _scan("hillis_steele", a, b, h0)


def scan_blelloch(a, b, h0=None):
    """Work-efficient up-sweep / down-sweep scan (models/scan.py:101-135)."""
    return _scan("blelloch", a, b, h0)


def scan_chunked(a, b, h0=None, chunk_size=None):
    """Two-level scan (models/scan.py:142-165).

    Below 160 groups of 64 recurrences the chunks of C = chunk_size or default_chunk(L) steps are spread
    over the GPU (three launches; the workspace holds three values per chunk and recurrence).  From
    there on one launch walks every recurrence in chunks of 16 steps and chunk_size changes
    nothing.  The result is the same to rounding either way."""
    return _scan("chunked", a, b, h0, chunk_size)


SCANS = {
    "sequential": scan_sequential,
    "hillis_steele": scan_hillis_steele,
    "blelloch": scan_blelloch,
    "chunked": scan_chunked,
}


def _scan_algo(name):
    """Algorithm id for a SCANS name; KeyError otherwise (models/scan.py:258-261)."""
    SCANS[name]
    return _SCAN_ALGO[name]


# ------------------------------------------------------------------ composed selective scan
class SelectiveScanFn(torch.autograd.Function):
    """y, last = selective scan by a named algorithm (models/scan.py:193-255).

    One kernel discretizes, scans and contracts with C tile by tile in time (ssm_cscan), so no
    (B, L, D, N) tensor exists; saved for the backward are x, delta, A, Bm, Cm, h0 and the state
    entering every time tile.  The backward recomputes the states tile by tile, runs the adjoint
    scan lambda_t = g_t + a_{t+1} lambda_{t+1} with the same algorithm and maps (da, db) =
    (lambda h_{t-1}, lambda) back through the discretization, in channel tiles of d_block (default:
    as many channels as keep the workspace within 256 MiB).  d_block bounds that workspace only (the
    forward has none to speak of), and chunk_size changes nothing: it is the chunk of a linear scan over
    materialized tensors, where here a chunk is a wavefront's part of a time tile."""

    @staticmethod
    def forward(ctx, x, delta, A, Bm, Cm, h0, method, scan_name, d_block, chunk_size):
        algo = _scan_algo(scan_name)
        if method not in DISCRETIZATIONS:
            raise ValueError(f"unknown discretization {method!r}")
        chunk = int(chunk_size or 0)
        if not 0 <= chunk < 1 << 30:
            raise ValueError(f"chunk={chunk} out of range")
        y, last, Bm, Cm, saved = _abi.host().cscan_forward(x, delta, A, Bm, Cm, h0, algo, METHODS[method],
                                                           any(ctx.needs_input_grad[:6]), profiling.active())
        ctx.save_for_backward(x, delta, A, Bm, Cm, h0, saved)
        ctx.set_materialize_grads(False)   # an unused output passes None (no zero fill)
        ctx.cfg = (algo, METHODS[method], int(d_block or 0))
        return y, last

    @staticmethod
    def backward(ctx, dy, dlast):
        grads = _abi.host().cscan_backward(*ctx.saved_tensors, *ctx.cfg, dy, dlast, profiling.active())
        return (*grads, None, None, None, None)


def selective_scan_reference(x, delta, A, Bm, Cm, h0=None, method="zoh"):
    """The step-by-step recurrence of models/scan.py:264-274, returning (y, h_last).

    Runs on the fused engine, which walks h_t = a_t h_{t-1} + b_t one time step at a time
    in every lane -- the same recurrence as the reference's loop, without storing the states."""
    if method not in DISCRETIZATIONS:
        raise ValueError(f"unknown discretization {method!r}")
    check_operands(x, delta, A, Bm, Cm, None, None, None, h0)
    return FusedSelectiveScanFn.apply(x, delta, A, Bm, Cm, None, None, None, h0, METHODS[method], False)


def selective_scan(x, delta, A, Bm, Cm, h0=None, method="zoh", scan="chunked",
                   d_block=None, chunk_size=None):
    """Returns (y, h_last) (models/scan.py:277-299).

    scan = 'reference' | 'sequential' | 'hillis_steele' | 'blelloch' | 'chunked'
           | 'triton' (the fused engine) | 'auto' (fused when N is a power of two, else chunked)
    d_block: channels per launch of the backward of the four named algorithms (bounds its workspace);
    chunk_size is accepted for the reference's signature and changes nothing (SelectiveScanFn).
    Computes in promote(dtype, float32); y is returned in x's dtype, h_last in the compute
    dtype.  KeyError for an unknown scan, ValueError for an unknown method."""
    _require_gpu(x, delta, A, Bm, Cm, h0)
    if scan == "auto":
        scan = plan.resolve_scan("auto", x.is_cuda, method, A.shape[1])
    elif scan not in _abi.SCAN_IDS:
        raise KeyError(scan)
    dtype = x.dtype
    ct = torch.promote_types(dtype, torch.float32)
    with torch.autocast(device_type=x.device.type, enabled=False):
        if scan == "triton":
            from .hip_scan import selective_scan_hip
            # the engine reads low-precision inputs directly and computes in ct
            y, last = selective_scan_hip(x, delta, A.to(ct), Bm, Cm, None if h0 is None else h0.to(ct),
                                         method=method, d_block=d_block)
            return y.to(dtype), last
        args = [t.to(ct) if t is not None else None for t in (x, delta, A, Bm, Cm, h0)]
        if scan == "reference":
            y, last = selective_scan_reference(*args, method=method)
        else:
            check_operands(*args[:5], None, None, None, args[5])
            y, last = SelectiveScanFn.apply(*args, method, scan, d_block, chunk_size)
    return y.to(dtype), last
