// The host side of the path's calls in one native module (_gpic_host): output allocation and the C-ABI calls of a cast
// group, a GEMM, a weight gradient, and the whole forward or backward of a phase-3 linear, without a Python frame, a
// ctypes conversion and a tensor constructor for each piece. A linear of a few hundred rows is bound by that host time,
// not by its kernels (~40 us of Python for 25 us of kernels in a sampler's proj).
//
// Every function takes tensors of the usual form only (on the current device, contiguous, 16-byte aligned, the types
// the C ABI takes) and returns None for any other, for which the caller runs its general form. Outputs are ordinary
// tensors of torch's allocator on the current stream, as the general form's. dev, ws, stream: the current device, its
// current stream's cast workspace (0 for the calls that cast nothing) and that stream. The GIL is released while a call
// allocates and launches, as ctypes and torch's own operations release it: a launch waits where the queue is full.
#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <string>

#include "../../include/gpic_fp8.h"

namespace py = pybind11;

namespace {

constexpr auto kE4 = at::kFloat8_e4m3fn;

void check(int status, const char *what) {
  if (status != GPIC_OK)
    throw std::runtime_error(std::string(what) + " failed: " + gpic_fp8_status_string(status) + " (status " +
                             std::to_string(status) + ")");
}

bool plain(const at::Tensor &t, int dev) {
  return t.is_cuda() && t.get_device() == dev && t.layout() == at::kStrided && t.is_contiguous() &&
         (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
}
bool castable(const at::Tensor &t, int dev) {
  return (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat) && plain(t, dev);
}
// A contiguous [rows, cols] e4m3 operand with 16-byte rows, and its scale
bool operand(const at::Tensor &t, const at::Tensor &s, int dev) {
  return t.scalar_type() == kE4 && t.dim() == 2 && t.size(1) % 16 == 0 && plain(t, dev) && s.scalar_type() == at::kFloat &&
         s.dim() == 1 && s.size(0) == 1 && s.is_cuda() && s.get_device() == dev;
}
int dtype_code(const at::Tensor &t) { return t.scalar_type() == at::kFloat ? GPIC_DTYPE_F32 : GPIC_DTYPE_BF16; }
template <class T>
T *ptr(const at::Tensor &t) {
  return static_cast<T *>(t.data_ptr());
}
at::Tensor make(const at::Tensor &like, at::IntArrayRef size, at::ScalarType ty) {
  return at::empty(size, like.options().dtype(ty).requires_grad(false));
}

struct Scratch {   // a GEMM's split-K workspace, when its plan has one
  at::Tensor t;
  size_t bytes;
  Scratch(const at::Tensor &like, int64_t M, int64_t N, int64_t K) : bytes(gpic_fp8_gemm_workspace_bytes(M, N, K)) {
    if (bytes) t = make(like, {(int64_t)bytes}, at::kByte);
  }
  void *p() const { return bytes ? t.data_ptr() : nullptr; }
};

enum { kFlat = 0, kBoth = 1, kTransposed = 2 };
constexpr int kMost = 8;

struct Casts {
  at::Tensor q[kMost], qt[kMost], s[kMost];
};
// xs[i]: castable; kind kBoth / kTransposed: 2-D with a multiple of 16 columns
void cast_group(int n, const at::Tensor *const *xs, const int *kinds, void *ws, void *stream, Casts &o) {
  const void *x[kMost];
  int dt[kMost];
  int64_t rows[kMost], cols[kMost], ldt[kMost];
  uint8_t *q[kMost], *qt[kMost];
  float *s[kMost];
  for (int i = 0; i < n; i++) {
    const at::Tensor &t = *xs[i];
    const bool flat = kinds[i] == kFlat;
    rows[i] = flat ? 1 : t.size(0);
    cols[i] = flat ? t.numel() : t.size(1);
    ldt[i] = flat ? 0 : (rows[i] + 15) / 16 * 16;
    o.q[i] = kinds[i] == kTransposed ? make(t, {0}, kE4) : make(t, t.sizes(), kE4);
    o.qt[i] = flat ? make(t, {0}, kE4) : make(t, {cols[i], ldt[i]}, kE4);
    o.s[i] = make(t, {1}, at::kFloat);
    x[i] = t.data_ptr();
    dt[i] = dtype_code(t);
    q[i] = kinds[i] == kTransposed ? nullptr : ptr<uint8_t>(o.q[i]);
    qt[i] = flat ? nullptr : ptr<uint8_t>(o.qt[i]);
    s[i] = ptr<float>(o.s[i]);
  }
  check(gpic_fp8_cast_group(n, x, dt, rows, cols, q, qt, ldt, s, ws, stream), "gpic_fp8_cast_group");
}

bool bias_ok(const std::optional<at::Tensor> &b, int64_t N, int dev) {
  return !b || (castable(*b, dev) && b->dim() == 1 && b->size(0) == N);
}
// a [M, K], b [N, K] -> bf16(sa sb a b^T) (+ bias) [M, N]
at::Tensor gemm_tn(const at::Tensor &a, const at::Tensor &sa, const at::Tensor &b, const at::Tensor &sb,
                   const std::optional<at::Tensor> &bias, void *stream) {
  const int64_t M = a.size(0), K = a.size(1), N = b.size(0);
  at::Tensor c = make(a, {M, N}, at::kBFloat16);
  const Scratch w(a, M, N, K);
  if (bias && bias->scalar_type() == at::kFloat) {
    check(gpic_fp8_gemm_bias32(ptr<uint8_t>(a), K, ptr<float>(sa), ptr<uint8_t>(b), K, ptr<float>(sb), ptr<float>(*bias),
                               ptr<uint16_t>(c), N, M, N, K, w.p(), w.bytes, stream),
          "gpic_fp8_gemm_bias32");
    return c;
  }
  check(gpic_fp8_gemm(ptr<uint8_t>(a), K, ptr<float>(sa), ptr<uint8_t>(b), K, ptr<float>(sb),
                      bias ? ptr<uint16_t>(*bias) : nullptr, ptr<uint16_t>(c), N, M, N, K, 1, w.p(), w.bytes, stream),
        "gpic_fp8_gemm");
  return c;
}
bool wgrad_ok(const at::Tensor &a, const at::Tensor &b) {
  return a.size(0) == b.size(0) && a.size(0) * std::max(a.size(1), b.size(1)) < (int64_t(1) << 31) &&
         b.size(1) < (1 << 21);
}
// a [K, M], b [K, N] -> bf16(sa sb a^T b) [M, N], as fp32 when f32
at::Tensor gemm_mn(const at::Tensor &a, const at::Tensor &sa, const at::Tensor &b, const at::Tensor &sb, bool f32,
                   void *stream) {
  const int64_t K = a.size(0), M = a.size(1), N = b.size(1);
  at::Tensor c = make(a, {M, N}, f32 ? at::kFloat : at::kBFloat16);
  const Scratch w(a, M, N, K);
  if (f32)
    check(gpic_fp8_gemm_mn_f32(ptr<uint8_t>(a), M, ptr<float>(sa), ptr<uint8_t>(b), N, ptr<float>(sb), ptr<float>(c), N,
                               M, N, K, w.p(), w.bytes, stream),
          "gpic_fp8_gemm_mn_f32");
  else
    check(gpic_fp8_gemm_mn(ptr<uint8_t>(a), M, ptr<float>(sa), ptr<uint8_t>(b), N, ptr<float>(sb), nullptr,
                           ptr<uint16_t>(c), N, M, N, K, w.p(), w.bytes, stream),
          "gpic_fp8_gemm_mn");
  return c;
}

at::Tensor bias_grad(const at::Tensor &dy, bool f32, void *stream) {
  const int64_t M = dy.size(0), N = dy.size(1);
  const size_t bytes = gpic_fp8_bias_grad_workspace_bytes(M, N);
  at::Tensor part = make(dy, {std::max<int64_t>((int64_t)bytes, 16)}, at::kByte);
  at::Tensor db = make(dy, {N}, f32 ? at::kFloat : at::kBFloat16);
  check(gpic_fp8_bias_grad(ptr<uint16_t>(dy), N, M, N, db.data_ptr(), f32 ? GPIC_DTYPE_F32 : GPIC_DTYPE_BF16,
                           part.data_ptr(), bytes, stream),
        "gpic_fp8_bias_grad");
  return db;
}

typedef uintptr_t handle;
void *vp(handle h) { return reinterpret_cast<void *>(h); }
typedef py::gil_scoped_release NoGil;

py::object casts(const std::vector<at::Tensor> &xs, const std::vector<int> &kinds, int dev, handle ws, handle stream) {
  const int n = (int)xs.size();
  if (n < 1 || n > kMost) return py::none();
  const at::Tensor *p[kMost];
  for (int i = 0; i < n; i++) {
    if (!castable(xs[i], dev) || (kinds[i] != kFlat && (xs[i].dim() != 2 || xs[i].size(1) % 16))) return py::none();
    p[i] = &xs[i];
  }
  Casts o;
  {
    NoGil no_gil;
    cast_group(n, p, kinds.data(), vp(ws), vp(stream), o);
  }
  py::list out;
  for (int i = 0; i < n; i++) {
    out.append(o.q[i]);
    out.append(o.qt[i]);
    out.append(o.s[i]);
  }
  return out;
}

py::object gemm(const at::Tensor &a, const at::Tensor &sa, const at::Tensor &b, const at::Tensor &sb,
                const std::optional<at::Tensor> &bias, int dev, handle, handle stream) {
  if (!operand(a, sa, dev) || !operand(b, sb, dev) || a.size(1) != b.size(1) || b.size(0) % 16 ||
      !bias_ok(bias, b.size(0), dev))
    return py::none();
  at::Tensor c;
  {
    NoGil no_gil;
    c = gemm_tn(a, sa, b, sb, bias, vp(stream));
  }
  return py::cast(c);
}

py::object wgrad(const at::Tensor &a, const at::Tensor &sa, const at::Tensor &b, const at::Tensor &sb, bool f32, int dev,
                 handle, handle stream) {
  if (!operand(a, sa, dev) || !operand(b, sb, dev) || !wgrad_ok(a, b)) return py::none();
  at::Tensor c;
  {
    NoGil no_gil;
    c = gemm_mn(a, sa, b, sb, f32, vp(stream));
  }
  return py::cast(c);
}

// x [M, K] bf16, w [N, K], bias [N] or None -> y [M, N], and x's and w's casts: (y, xq, sx, wqt, sw), w's
// transposed bytes only when `both` (else an empty tensor)
py::object linear_fwd(const at::Tensor &x, const at::Tensor &w, const std::optional<at::Tensor> &bias, bool both, int dev,
                      handle ws, handle stream) {
  if (x.dim() != 2 || w.dim() != 2 || x.size(1) != w.size(1) || x.size(1) % 16 || w.size(0) % 16 ||
      !castable(x, dev) || !castable(w, dev) || !bias_ok(bias, w.size(0), dev))
    return py::none();
  const at::Tensor *p[2] = {&x, &w};
  const int kinds[2] = {kFlat, both ? kBoth : kFlat};
  Casts o;
  at::Tensor y;
  {
    NoGil no_gil;
    cast_group(2, p, kinds, vp(ws), vp(stream), o);
    y = gemm_tn(o.q[0], o.s[0], o.q[1], o.s[1], bias, vp(stream));
  }
  return py::make_tuple(y, o.q[0], o.s[0], o.qt[1], o.s[1]);
}

// dy [M, N] bf16, the forward's xq [M, K] and wqt [K, N] -> (dx [M, K], dw [N, K], db [N] or None); dw and db fp32
// (holding bf16 values) when f32, else bf16
py::object linear_bwd(const at::Tensor &dy, const at::Tensor &xq, const at::Tensor &sx, const at::Tensor &wqt,
                      const at::Tensor &sw, bool has_bias, bool f32, int dev, handle ws, handle stream) {
  if (dy.dim() != 2 || dy.scalar_type() != at::kBFloat16 || !plain(dy, dev) || dy.size(1) % 16 ||
      !operand(xq, sx, dev) || !operand(wqt, sw, dev) || wqt.size(0) % 16 || wqt.size(1) != dy.size(1) ||
      xq.size(0) != dy.size(0) || !wgrad_ok(dy, xq))
    return py::none();
  const at::Tensor *p[1] = {&dy};
  const int kinds[1] = {kFlat};
  at::Tensor dx, dw, db;
  {
    NoGil no_gil;
    Casts o;
    cast_group(1, p, kinds, vp(ws), vp(stream), o);
    const at::Tensor &dyq = o.q[0], &sdy = o.s[0];
    dx = gemm_tn(dyq, sdy, wqt, sw, std::nullopt, vp(stream));
    dw = gemm_mn(dyq, sdy, xq, sx, f32, vp(stream));
    if (has_bias) db = bias_grad(dy, f32, vp(stream));
  }
  if (!has_bias) return py::make_tuple(dx, dw, py::none());
  return py::make_tuple(dx, dw, db);
}

}  // namespace

PYBIND11_MODULE(_gpic_host, m) {   // (wrapped: torch's own errors, out of memory among them, stay what they are)
  m.def("casts", torch::wrap_pybind_function(&casts));
  m.def("gemm", torch::wrap_pybind_function(&gemm));
  m.def("wgrad", torch::wrap_pybind_function(&wgrad));
  m.def("linear_fwd", torch::wrap_pybind_function(&linear_fwd));
  m.def("linear_bwd", torch::wrap_pybind_function(&linear_bwd));
}
