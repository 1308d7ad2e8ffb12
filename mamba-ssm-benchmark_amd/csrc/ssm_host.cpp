// Python binding of the launches (module ssm_scan._ssmhost): operand checks, output and workspace
// allocation and the argument structs of the C ABI in one call per launch.  The same work done from
// Python -- a ctypes struct of up to 25 views, 5-10 torch.empty calls, device and stream lookups --
// took 15-45 us per launch, more than the kernels of a short scan, a conv or a norm: rms_norm
// forward + backward (8192 x 256) 120 us against 18 us of kernels.
//
// Nothing here is numerical and nothing is kept between calls but a DecodePlan's weight tensors.
// Errors of the C ABI become the exception classes of ssm_scan._abi.check.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <optional>
#include <sstream>
#include <vector>

#include "../../include/ssm_scan.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

// ------------------------------------------------------------------ helpers
ssm_tensor view(const Tensor &t) {
  ssm_tensor v{};
  if (!t.defined()) return v;
  TORCH_CHECK_VALUE(t.dim() <= 3, "expected a tensor of at most 3 dims, got ", t.dim());
  v.data = t.data_ptr();
  for (int64_t i = 0; i < t.dim(); ++i) v.stride[i] = t.stride(i);
  return v;
}
Tensor get(const OptTensor &t) { return t.has_value() ? *t : Tensor(); }
py::object out(const Tensor &t) { return t.defined() ? py::cast(t) : py::none(); }

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return SSM_F32;
    case at::kBFloat16: return SSM_BF16;
    case at::kHalf: return SSM_F16;
    case at::kDouble: return SSM_F64;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t);
  }
}
bool io_type(at::ScalarType t) {
  return t == at::kFloat || t == at::kBFloat16 || t == at::kHalf || t == at::kDouble;
}

void check(int rc, const char *what) {
  if (rc == SSM_OK) return;
  TORCH_CHECK_VALUE(rc != SSM_EINVAL && rc != SSM_ESPACE, what, ": ", ssm_last_error());
  TORCH_CHECK(false, what, ": ", ssm_last_error());
}
// A *_bytes query: the check behind it names what is wrong.
#define SSM_BYTES(var, query, checkfn, args, what) \
  const int64_t var = query(&args);                \
  if (var < 0) {                                   \
    check(checkfn(&args), what);                   \
    check(SSM_EINVAL, what);                       \
  }

void require_gpu(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    TORCH_CHECK(!t->defined() || t->is_cuda(), "ssm_scan runs on ROCm GPU tensors only; got a tensor on ",
                t->device().str(), " (there is no CPU path)");
}

std::string shape_str(at::IntArrayRef s) {
  std::ostringstream o;
  o << "(";
  for (size_t i = 0; i < s.size(); ++i) o << (i ? ", " : "") << s[i];
  o << (s.size() == 1 ? ",)" : ")");
  return o.str();
}
void want(const char *name, const Tensor &t, at::IntArrayRef shape) {
  if (t.defined())
    TORCH_CHECK_VALUE(t.sizes() == shape, name, " must have shape ", shape_str(shape), ", got ", shape_str(t.sizes()));
}

Tensor cast(const Tensor &t, at::ScalarType dt) { return !t.defined() || t.scalar_type() == dt ? t : t.to(dt); }
// Output buffer with t's layout when t is dense (e.g. channel-major views), else contiguous.
Tensor like(const Tensor &t, at::ScalarType dt) {
  const auto o = t.options().dtype(dt);
  return t.is_non_overlapping_and_dense() ? at::empty_like(t, o, at::MemoryFormat::Preserve) : at::empty(t.sizes(), o);
}
Tensor empty(at::IntArrayRef s, const Tensor &ref, at::ScalarType dt) { return at::empty(s, ref.options().dtype(dt)); }
Tensor bytes(int64_t n, const Tensor &ref) { return at::empty({std::max<int64_t>(n, 1)}, ref.options().dtype(at::kByte)); }

// The engine launches on the current device and on torch's current stream there.
struct Launch {
  c10::DeviceGuard guard;
  void *stream;
  explicit Launch(const Tensor &t)
      : guard(t.device()), stream((void *)c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
  // One launch, without the GIL: it blocks while the device's queue is full, and other Python threads
  // run on.  `timer` (a profiling.KernelTimer, or None) records its events right around it: the operand
  // checks, casts and allocations of the call are outside.
  template <typename Args>
  void run(const char *what, int (*fn)(const Args *, void *), const Args &args, const py::object &timer = py::none()) const {
    const py::object end = timer.is_none() ? timer : timer.attr("begin")(what);
    int rc;
    {
      py::gil_scoped_release release;
      rc = fn(&args, stream);
    }
    if (!end.is_none()) end.attr("record")();
    check(rc, what);
  }
};

// ------------------------------------------------------------------ fused scan
void scan_checks(const Tensor &x, const OptTensor &delta_, const Tensor &A, const Tensor &Bm, const Tensor &Cm,
                 const OptTensor &D_, const OptTensor &z_, const OptTensor &bias_, const OptTensor &h0_,
                 const OptTensor &proj_) {
  const Tensor delta = get(delta_), D = get(D_), z = get(z_), bias = get(bias_), h0 = get(h0_), proj = get(proj_);
  require_gpu({&x, &delta, &A, &Bm, &Cm, &D, &z, &bias, &h0, &proj});
  TORCH_CHECK_VALUE(x.dim() == 3, "x must be (B, L, D), got ", shape_str(x.sizes()));
  const int64_t B = x.size(0), L = x.size(1), Dm = x.size(2);
  TORCH_CHECK_VALUE(A.dim() == 2 && A.size(0) == Dm, "A must be (D, N) = (", Dm, ", N), got ", shape_str(A.sizes()));
  const int64_t N = A.size(1);
  int64_t dd = Dm;
  if (proj.defined()) {
    TORCH_CHECK_VALUE(proj.dim() == 2 && proj.size(0) == Dm, "delta_proj must be (D, R) = (", Dm, ", R), got ",
                      shape_str(proj.sizes()));
    dd = proj.size(1);
  }
  want("delta", delta, {B, L, dd});
  want("Bm", Bm, {B, L, N});
  want("Cm", Cm, {B, L, N});
  want("D", D, {Dm});
  want("z", z, {B, L, Dm});
  want("delta_bias", bias, {Dm});
  want("h0", h0, {B, Dm, N});
}

template <typename Args>
void fill_scan(Args &a, const Tensor &x, const Tensor &delta, const Tensor &A, const Tensor &Bm, const Tensor &Cm,
               const Tensor &D, const Tensor &z, const Tensor &bias, const Tensor &h0, const Tensor &proj, int method,
               bool softplus, bool a_log, int segments) {
  memset(&a, 0, sizeof(a));
  a.batch = x.size(0); a.seqlen = x.size(1); a.dim = x.size(2); a.dstate = A.size(1);
  a.method = method;
  a.dtype = dtype_code(x.scalar_type());
  a.x = view(x); a.delta = view(delta); a.A = view(A); a.Bm = view(Bm); a.Cm = view(Cm);
  a.Dskip = view(D); a.z = view(z); a.delta_bias = view(bias); a.h0 = view(h0);
  a.delta_softplus = softplus;
  a.segments = segments;
  if (proj.defined()) {
    a.delta_proj = view(proj);
    a.delta_rank = proj.size(1);
  }
  a.A_is_log = a_log;
}

// (out in the io dtype, last, the tensors scan_backward needs)
py::tuple scan_forward(const Tensor &x, const Tensor &delta, const Tensor &A, const Tensor &Bm, const Tensor &Cm,
                       const OptTensor &D_, const OptTensor &z_, const OptTensor &bias_, const OptTensor &h0_, int method,
                       bool softplus, int segments, const OptTensor &proj_, bool a_log, bool need_saved, const py::object &timer) {
  at::ScalarType ct = c10::promoteTypes(x.scalar_type(), at::kFloat), io = at::kFloat;
  const Tensor z = get(z_);
  if (ct == at::kDouble) {
    io = ct;
  } else {
    ct = at::kFloat;
    bool same = io_type(x.scalar_type());
    for (const Tensor *t : {&delta, &Bm, &Cm, &z}) same = same && (!t->defined() || t->scalar_type() == x.scalar_type());
    if (same) io = x.scalar_type();
  }
  const Tensor xs = cast(x, io), ds = cast(delta, io), Bs = cast(Bm, io), Cs = cast(Cm, io), zs = cast(z, io);
  const Tensor As = cast(A, ct), Dv = cast(get(D_), ct), bv = cast(get(bias_), ct), h0 = cast(get(h0_), ct),
               W = cast(get(proj_), ct);
  const Tensor o = like(xs, io), last = empty({x.size(0), x.size(2), A.size(1)}, x, ct);
  ssm_fwd_args a;
  fill_scan(a, xs, ds, As, Bs, Cs, Dv, zs, bv, h0, W, method, softplus, a_log, segments);
  a.out = view(o);
  a.last = view(last);
  SSM_BYTES(wbytes, ssm_fwd_workspace_bytes, ssm_fwd_check, a, "ssm_fwd");
  Tensor ws, saved;
  if (wbytes) {
    ws = bytes(wbytes, x);
    a.workspace = ws.data_ptr();
    a.workspace_bytes = wbytes;
  }
  if (need_saved) {
    SSM_BYTES(sbytes, ssm_fwd_saved_bytes, ssm_fwd_check, a, "ssm_fwd_saved_bytes");
    saved = bytes(sbytes, x);
    a.saved = saved.data_ptr();
  }
  const Launch l(x);
  l.run("ssm_fwd", ssm_fwd, a, timer);
  return py::make_tuple(o, last, py::make_tuple(xs, ds, As, Bs, Cs, out(Dv), out(zs), out(bv), out(h0), out(W), out(saved)));
}

py::tuple scan_backward(const Tensor &xs, const Tensor &ds, const Tensor &As, const Tensor &Bs, const Tensor &Cs,
                        const OptTensor &Dv_, const OptTensor &zs_, const OptTensor &bv_, const OptTensor &h0_,
                        const OptTensor &W_, const Tensor &saved, int method, bool softplus, bool a_log, int segments,
                        const OptTensor &dout_, const OptTensor &dlast_, const OptTensor &dz_, const OptTensor &dB_,
                        const OptTensor &dC_, const py::object &timer) {
  const Tensor Dv = get(Dv_), zs = get(zs_), bv = get(bv_), h0 = get(h0_), W = get(W_);
  const at::ScalarType io = xs.scalar_type(), ct = As.scalar_type();
  const Tensor dout = dout_ ? cast(*dout_, io) : at::zeros(xs.sizes(), xs.options());
  const Tensor dlast = cast(get(dlast_), ct);
  const int64_t B = xs.size(0), Dm = xs.size(2), N = As.size(1);
  const Tensor dx = like(xs, io), dd = like(W.defined() ? xs : ds, io), dA = empty({Dm, N}, xs, ct);
  const Tensor dB = dB_ ? *dB_ : like(Bs, io), dC = dC_ ? *dC_ : like(Cs, io);
  const Tensor dz = dz_ ? *dz_ : zs.defined() ? like(zs, io) : Tensor();
  const Tensor dD = Dv.defined() ? empty({Dm}, xs, ct) : Tensor(), db = bv.defined() ? empty({Dm}, xs, ct) : Tensor();
  const Tensor dh0 = h0.defined() ? empty({B, Dm, N}, xs, ct) : Tensor();
  ssm_bwd_args a;
  fill_scan(a, xs, ds, As, Bs, Cs, Dv, zs, bv, h0, W, method, softplus, a_log, segments);
  a.saved = saved.data_ptr();
  a.dout = view(dout); a.dlast = view(dlast);
  a.dx = view(dx); a.ddelta = view(dd); a.dA = view(dA);
  a.dBm = view(dB); a.dCm = view(dC); a.dD = view(dD);
  a.dz = view(dz); a.ddelta_bias = view(db); a.dh0 = view(dh0);
  SSM_BYTES(n, ssm_bwd_workspace_bytes, ssm_bwd_check, a, "ssm_bwd");
  const Tensor ws = bytes(n, xs);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = n;
  const Launch l(xs);
  l.run("ssm_bwd", ssm_bwd, a, timer);
  return py::make_tuple(dx, dd, dA, dB, dC, out(dD), out(dz), out(db), out(dh0));
}

// ------------------------------------------------------------------ conv
ssm_conv_args conv_args(const Tensor &x, const Tensor &w, const Tensor &bias, bool act) {
  ssm_conv_args a;
  memset(&a, 0, sizeof(a));
  a.batch = x.size(0); a.seqlen = x.size(1); a.dim = x.size(2); a.width = w.size(1);
  a.dtype = dtype_code(x.scalar_type());
  a.silu = act;
  a.x = view(x); a.weight = view(w); a.bias = view(bias);
  return a;
}

Tensor conv_forward(const Tensor &x, const Tensor &w, const OptTensor &bias, bool act, const OptTensor &state) {
  const Tensor o = at::empty(x.sizes(), x.options());
  ssm_conv_args a = conv_args(x, w, get(bias), act);
  a.out = view(o);
  if (state) a.state_in = a.state_out = view(*state);
  const Launch l(x);
  l.run("ssm_conv_fwd", ssm_conv_fwd, a);
  return o;
}

py::tuple conv_backward(const Tensor &x, const Tensor &w, const OptTensor &bias_, const Tensor &dout_, bool act,
                        const OptTensor &dx_) {
  const Tensor bias = get(bias_), dout = cast(dout_, x.scalar_type());
  const Tensor dx = dx_ ? *dx_ : at::empty(x.sizes(), x.options()), dw = at::empty_like(w);
  const Tensor db = bias.defined() ? at::empty_like(bias) : Tensor();
  ssm_conv_args a = conv_args(x, w, bias, act);
  a.dout = view(dout); a.dx = view(dx); a.dweight = view(dw); a.dbias = view(db);
  SSM_BYTES(n, ssm_conv_workspace_bytes, ssm_conv_check, a, "ssm_conv_bwd");
  const Tensor ws = bytes(n, x);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = n;
  const Launch l(x);
  l.run("ssm_conv_bwd", ssm_conv_bwd, a);
  return py::make_tuple(dx, dw, out(db));
}

// ------------------------------------------------------------------ RMSNorm
ssm_norm_args norm_args(const Tensor &x2, const Tensor &w, double eps) {
  ssm_norm_args a;
  memset(&a, 0, sizeof(a));
  a.rows = x2.size(0);
  a.dim = x2.size(1);
  a.dtype = dtype_code(x2.scalar_type());
  a.eps = eps;
  a.x = view(x2);
  a.weight = view(w);
  return a;
}
Tensor rows(const Tensor &t, int64_t C) {
  const Tensor r = t.reshape({-1, C});
  return r.stride(1) == 1 ? r : r.contiguous();
}

// (out, x as rows, weight, rstd)
py::tuple norm_forward(const Tensor &x, const Tensor &weight, double eps) {
  const Tensor x2 = rows(x, x.size(-1)), w = weight.contiguous();
  const Tensor o = at::empty(x2.sizes(), x.options()), rstd = at::empty({x2.size(0)}, x.options());
  ssm_norm_args a = norm_args(x2, w, eps);
  a.out = view(o);
  a.rstd = rstd.data_ptr();
  const Launch l(x);
  l.run("ssm_norm_fwd", ssm_norm_fwd, a);
  return py::make_tuple(o.view(x.sizes()), x2, w, rstd);
}

py::tuple norm_backward(const Tensor &x2, const Tensor &w, const Tensor &rstd, const Tensor &dout, double eps) {
  const Tensor dy = rows(cast(dout, x2.scalar_type()), x2.size(1));
  const Tensor dx = at::empty(x2.sizes(), x2.options()), dw = at::empty(w.sizes(), w.options());
  ssm_norm_args a = norm_args(x2, w, eps);
  a.rstd = rstd.data_ptr();
  a.dout = view(dy);
  a.dx = view(dx);
  a.dweight = dw.data_ptr();
  SSM_BYTES(n, ssm_norm_workspace_bytes, ssm_norm_check, a, "ssm_norm_bwd");
  const Tensor ws = bytes(n, x2);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = n;
  const Launch l(x2);
  l.run("ssm_norm_bwd", ssm_norm_bwd, a);
  return py::make_tuple(dx.view(dout.sizes()), dw);
}

// ------------------------------------------------------------------ linear scans
template <typename Args>
void fill_lscan(Args &args, const Tensor &a, int algo, int64_t chunk, bool reverse) {
  memset(&args, 0, sizeof(args));
  args.batch = a.size(0); args.seqlen = a.size(1); args.width = a.size(2);
  args.algo = algo;
  args.dtype = dtype_code(a.scalar_type());
  args.reverse = reverse;
  args.chunk = chunk;
}

Tensor lscan_forward(const Tensor &a, const Tensor &b, const OptTensor &h0, int algo, int64_t chunk, bool reverse,
                     const py::object &timer) {
  const Tensor h = at::empty(a.sizes(), a.options());
  ssm_lscan_args args;
  fill_lscan(args, a, algo, chunk, reverse);
  args.a = view(a); args.b = view(b); args.h0 = view(get(h0)); args.h = view(h);
  SSM_BYTES(n, ssm_lscan_workspace_bytes, ssm_lscan_check, args, "ssm_lscan");
  Tensor ws;
  if (n) {
    ws = bytes(n, a);
    args.workspace = ws.data_ptr();
    args.workspace_bytes = n;
  }
  const Launch l(a);
  l.run("ssm_lscan", ssm_lscan, args, timer);
  return h;
}

py::tuple lscan_backward(const Tensor &a, const OptTensor &h0_, const Tensor &h, const Tensor &dh, int algo, int64_t chunk,
                         bool reverse, bool need_dh0, const py::object &timer) {
  const Tensor h0 = get(h0_);
  const Tensor da = at::empty_like(h), db = at::empty_like(h);
  const Tensor dh0 = h0.defined() && need_dh0 ? at::empty_like(h0) : Tensor();
  ssm_lscan_bwd_args args;
  fill_lscan(args, a, algo, chunk, reverse);
  args.a = view(a); args.h0 = view(h0); args.h = view(h); args.dh = view(dh);
  args.da = view(da); args.db = view(db); args.dh0 = view(dh0);
  SSM_BYTES(n, ssm_lscan_bwd_workspace_bytes, ssm_lscan_bwd_check, args, "ssm_lscan_bwd");
  Tensor ws;
  if (n) {
    ws = bytes(n, a);
    args.workspace = ws.data_ptr();
    args.workspace_bytes = n;
  }
  const Launch l(a);
  l.run("ssm_lscan_bwd", ssm_lscan_bwd, args, timer);
  return py::make_tuple(da, db, out(dh0));
}

// ------------------------------------------------------------------ composed scan
constexpr int64_t kCscanWorkspace = 1LL << 28;  // bytes of dB / dC partials per backward launch
constexpr int64_t kCscanChannels = 1LL << 21;   // channels per launch

// t, or a contiguous copy where 64 steps of a batch row span 2 GiB (the kernels' offsets).
Tensor steps_fit(const Tensor &t) {
  const int64_t span = (t.stride(2) * (t.size(2) - 1) + 63 * t.stride(1) + 1) * t.element_size();
  return span < (1LL << 31) ? t : t.contiguous();
}
Tensor chans(const Tensor &t, int64_t dim, int64_t i, int64_t n) {
  return !t.defined() || (i == 0 && n == t.size(dim)) ? t : t.narrow(dim, i, n);
}

ssm_cscan_args cscan_args(const Tensor &x, const Tensor &delta, const Tensor &A, const Tensor &Bm, const Tensor &Cm,
                          const Tensor &h0, const Tensor &saved, int64_t i, int64_t n, int algo, int method) {
  ssm_cscan_args a;
  memset(&a, 0, sizeof(a));
  a.batch = x.size(0); a.seqlen = x.size(1); a.dim = n; a.dstate = A.size(1);
  a.algo = algo;
  a.method = method;
  a.dtype = dtype_code(x.scalar_type());
  a.x = view(x); a.delta = view(delta); a.A = view(chans(A, 0, i, n)); a.Bm = view(Bm); a.Cm = view(Cm);
  a.h0 = view(chans(h0, 1, i, n));
  if (saved.defined()) {  // (B, tiles, D, N), states consecutive
    a.saved.data = (char *)saved.data_ptr() + i * saved.stride(2) * saved.element_size();
    for (int k = 0; k < 3; ++k) a.saved.stride[k] = saved.stride(k);
  }
  return a;
}

// (y, last, Bm, Cm, saved)
py::tuple cscan_forward(const Tensor &x, const Tensor &delta, const Tensor &A, const Tensor &Bm_, const Tensor &Cm_,
                        const OptTensor &h0_, int algo, int method, bool need_saved, const py::object &timer) {
  const Tensor Bm = steps_fit(Bm_), Cm = steps_fit(Cm_), h0 = get(h0_);
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2), N = A.size(1);
  const Tensor y = at::empty_like(x), last = at::empty({B, D, N}, x.options());
  Tensor saved;
  if (need_saved) {
    const int64_t tile = ssm_cscan_tile(algo, dtype_code(x.scalar_type()));
    saved = at::empty({B, (L + tile - 1) / tile, D, N}, x.options());
  }
  const Launch l(x);
  for (int64_t i = 0; i < D || i == 0; i += kCscanChannels) {
    const int64_t n = std::min(D - i, kCscanChannels);
    const Tensor xb = steps_fit(chans(x, 2, i, n)), db = steps_fit(chans(delta, 2, i, n));
    ssm_cscan_args a = cscan_args(xb, db, A, Bm, Cm, h0, saved, i, n, algo, method);
    a.y = view(chans(y, 2, i, n));
    a.last = view(chans(last, 1, i, n));
    SSM_BYTES(nb, ssm_cscan_fwd_workspace_bytes, ssm_cscan_check, a, "ssm_cscan_fwd");
    Tensor ws;
    if (nb) {
      ws = bytes(nb, x);
      a.workspace = ws.data_ptr();
      a.workspace_bytes = nb;
    }
    l.run("ssm_cscan_fwd", ssm_cscan_fwd, a, timer);
  }
  return py::make_tuple(y, last, Bm, Cm, out(saved));
}

// Channel tiles of d_block, else all channels at once up to kCscanChannels and as many as keep the
// partials (2 x L x NP per 64 / NP channels and batch row) within kCscanWorkspace.
py::tuple cscan_backward(const Tensor &x, const Tensor &delta, const Tensor &A, const Tensor &Bm, const Tensor &Cm,
                         const OptTensor &h0_, const Tensor &saved, int algo, int method, int64_t d_block,
                         const OptTensor &dy_, const OptTensor &dlast_, const py::object &timer) {
  const Tensor h0 = get(h0_), dlast = get(dlast_);
  const Tensor dy = dy_ ? *dy_ : at::zeros_like(x);
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2), N = A.size(1);
  int64_t step = kCscanChannels;
  if (d_block > 0) {
    step = std::min(step, d_block);
  } else {
    const int64_t NP = N <= 8 ? 8 : N <= 16 ? 16 : N <= 32 ? 32 : 64;
    step = std::min(step, std::max<int64_t>(1, kCscanWorkspace / (B * L * 2 * NP * x.element_size())) * (64 / NP));
  }
  const Tensor dx = at::empty_like(x), dd = at::empty_like(delta), dA = at::empty_like(A);
  const Tensor dh0 = h0.defined() ? at::empty_like(h0) : Tensor();
  Tensor dB, dC;
  const Launch l(x);
  for (int64_t i = 0; i < D; i += step) {
    const int64_t n = std::min(D - i, step);
    const Tensor gB = at::empty_like(Bm), gC = at::empty_like(Cm);
    const Tensor xb = steps_fit(chans(x, 2, i, n)), db = steps_fit(chans(delta, 2, i, n)), yb = steps_fit(chans(dy, 2, i, n));
    ssm_cscan_args a = cscan_args(xb, db, A, Bm, Cm, h0, saved, i, n, algo, method);
    a.dy = view(yb); a.dlast = view(chans(dlast, 1, i, n));
    a.dx = view(chans(dx, 2, i, n)); a.ddelta = view(chans(dd, 2, i, n)); a.dA = view(chans(dA, 0, i, n));
    a.dBm = view(gB); a.dCm = view(gC); a.dh0 = view(chans(dh0, 1, i, n));
    SSM_BYTES(nb, ssm_cscan_workspace_bytes, ssm_cscan_check, a, "ssm_cscan_bwd");
    const Tensor ws = bytes(nb, x);
    a.workspace = ws.data_ptr();
    a.workspace_bytes = nb;
    l.run("ssm_cscan_bwd", ssm_cscan_bwd, a, timer);
    if (!dB.defined()) {
      dB = gB;
      dC = gC;
    } else {
      dB.add_(gB);
      dC.add_(gC);
    }
  }
  return py::make_tuple(dx, dd, dA, dB, dC, out(dh0));
}

// ------------------------------------------------------------------ decode
// The weights of a block stack's token step, laid out once; a step brings tokens and states.
struct DecodePlan {
  struct Block {
    Tensor w_in4, conv_w, conv_b, x_proj_wt, dt_proj_w, dt_bias, A_log, Dskip, w_out4;
    double eps;
  };
  std::vector<Block> blocks;
  Tensor head_w4;
  int64_t dm, dim, N, W, R, V;

  DecodePlan(const std::vector<std::pair<std::vector<Tensor>, double>> &layers, Tensor head, int64_t dm_, int64_t dim_,
             int64_t N_, int64_t W_, int64_t R_, int64_t V_)
      : head_w4(std::move(head)), dm(dm_), dim(dim_), N(N_), W(W_), R(R_), V(V_) {
    for (const auto &l : layers) {
      const auto &t = l.first;
      TORCH_CHECK_VALUE(t.size() == 9, "a decode block has 9 weights");
      blocks.push_back({t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], l.second});
    }
  }

  // Host-side checks before any launch: the kernels size every state buffer from the token count
  // and the model's dimensions.
  void check_states(const Tensor &tok, const std::vector<Tensor> &conv, const std::vector<Tensor> &ssm) const {
    const Tensor &w = blocks.at(0).w_in4;
    require_gpu({&w, &tok});
    for (size_t i = 0; i < conv.size(); ++i) require_gpu({&conv[i], &ssm[i]});
    const int64_t B = tok.numel();
    const auto dev = w.device();
    TORCH_CHECK_VALUE(tok.device() == dev, "tokens on ", tok.device().str(), ", the model on ", dev.str());
    TORCH_CHECK_VALUE(conv.size() == blocks.size(), conv.size(), " states for ", blocks.size(), " blocks");
    for (size_t i = 0; i < conv.size(); ++i) {
      const Tensor &c = conv[i], &s = ssm[i];
      const std::vector<int64_t> ws{B, dim, N}, wc{B, dim, W - 1};
      TORCH_CHECK_VALUE(s.sizes() == at::IntArrayRef(ws) && c.sizes() == at::IntArrayRef(wc), "block ", i, ": states ",
                        shape_str(s.sizes()), " / ", shape_str(c.sizes()), ", expected ", shape_str(ws), " / ",
                        shape_str(wc), " for ", B, " tokens");
      TORCH_CHECK_VALUE(s.device() == dev && c.device() == dev, "block ", i, ": states on ", s.device().str(), " / ",
                        c.device().str(), ", the model on ", dev.str());
      TORCH_CHECK_VALUE(c.is_contiguous() && s.is_contiguous() && s.scalar_type() == at::kFloat &&
                            (c.scalar_type() == at::kFloat || c.scalar_type() == at::kBFloat16),
                        "decode states must be contiguous: ssm float32, conv float32 or bf16");
    }
  }

  void fill(ssm_decode_stack_args &a, int64_t B) const {
    memset(&a, 0, sizeof(a));
    a.batch = B; a.dim = dim; a.dstate = N; a.width = W; a.dt_rank = R; a.d_model = dm;
    a.n_blocks = (int32_t)blocks.size();
    a.vocab = V;
  }
  int64_t workspace_bytes(int64_t B) const {
    ssm_decode_stack_args a;
    fill(a, B);
    return ssm_decode_stack_workspace_bytes(&a);
  }
  int64_t status_offset(int64_t B) const {
    ssm_decode_stack_args a;
    fill(a, B);
    return ssm_decode_stack_status_offset(&a);
  }

  // The whole token step in one call; returns the logits.  The discretization and the final norm's eps
  // are settings of the model, not weights: they come with each step.
  Tensor step(const Tensor &tok_, const std::vector<Tensor> &conv, const std::vector<Tensor> &ssm, const Tensor &embed,
              const Tensor &ws, int method, double head_eps) const {
    for (const Tensor &c : conv)
      TORCH_CHECK_VALUE(c.scalar_type() == conv[0].scalar_type(),
                        "the stack path needs one conv state dtype for every block");
    const Tensor tok = tok_.reshape({-1}).to(at::kLong).contiguous();  // a strided view of ids is copied
    const int64_t B = tok.numel();
    const auto f = head_w4.options();
    const Tensor u = at::empty({B, dm}, f), logits = at::empty({B, V}, f);
    std::vector<ssm_decode_block> k(blocks.size());
    auto p = [](const Tensor &t) { return (const float *)t.data_ptr(); };
    for (size_t i = 0; i < k.size(); ++i) {
      const Block &b = blocks[i];
      memset(&k[i], 0, sizeof(k[i]));
      k[i].w_in4 = p(b.w_in4); k[i].conv_w = p(b.conv_w); k[i].conv_b = p(b.conv_b); k[i].x_proj_wt = p(b.x_proj_wt);
      k[i].dt_proj_w = p(b.dt_proj_w); k[i].dt_bias = p(b.dt_bias); k[i].A_log = p(b.A_log); k[i].Dskip = p(b.Dskip);
      k[i].w_out4 = p(b.w_out4);
      k[i].conv_state = conv[i].data_ptr();
      k[i].ssm_state = (float *)ssm[i].data_ptr();
      k[i].eps = (float)b.eps;
    }
    ssm_decode_stack_args a;
    fill(a, B);
    a.method = method;
    a.head_eps = (float)head_eps;
    a.conv_state_dtype = dtype_code(conv[0].scalar_type());
    a.blocks = k.data();
    a.u = (float *)u.data_ptr();
    a.tokens = (const int64_t *)tok.data_ptr();
    a.embed = p(embed);
    a.head_w4 = p(head_w4);
    a.logits = (float *)logits.data_ptr();
    a.workspace = ws.data_ptr();
    a.workspace_bytes = ws.numel();
    const Launch l(u);
    l.run("ssm_decode_stack", ssm_decode_stack, a);
    return logits;
  }
};

}  // namespace

PYBIND11_MODULE(_ssmhost, m) {
  m.def("scan_checks", torch::wrap_pybind_function(scan_checks));
  m.def("scan_forward", torch::wrap_pybind_function(scan_forward));
  m.def("scan_backward", torch::wrap_pybind_function(scan_backward));
  m.def("conv_forward", torch::wrap_pybind_function(conv_forward));
  m.def("conv_backward", torch::wrap_pybind_function(conv_backward));
  m.def("norm_forward", torch::wrap_pybind_function(norm_forward));
  m.def("norm_backward", torch::wrap_pybind_function(norm_backward));
  m.def("lscan_forward", torch::wrap_pybind_function(lscan_forward));
  m.def("lscan_backward", torch::wrap_pybind_function(lscan_backward));
  m.def("cscan_forward", torch::wrap_pybind_function(cscan_forward));
  m.def("cscan_backward", torch::wrap_pybind_function(cscan_backward));
  m.attr("ABI_VERSION") = SSM_ABI_VERSION;  // of the header the argument structs above were compiled from
  py::class_<DecodePlan>(m, "DecodePlan")
      .def(py::init<const std::vector<std::pair<std::vector<Tensor>, double>> &, Tensor, int64_t, int64_t, int64_t, int64_t,
                    int64_t, int64_t>())
      .def("check_states", torch::wrap_pybind_function(&DecodePlan::check_states))
      .def("workspace_bytes", &DecodePlan::workspace_bytes)
      .def("status_offset", &DecodePlan::status_offset)
      .def("step", torch::wrap_pybind_function(&DecodePlan::step));
}
