// Native entry of the torch-facing ops (hxmi.py) for their plain form: every
// tensor an ordinary strided GPU tensor on one device, already in the layout
// the C ABI takes.  Each function checks exactly that, allocates the result
// (a split-K workspace comes from hxmi.py's own cache) and calls the C ABI on
// the current stream; for anything else, and for a call the library rejects,
// it returns None and the Python form of the op runs, which converts what it
// can and names what it cannot.  A launch costs the host 2.7 us; the Python form of these ops took
// 8.2-17.4 us a call (arguments, checks, allocation, ctypes), which is what
// a decode projection or a norm took eagerly whatever its kernel did.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "../../include/hxmi.h"

namespace {

using at::Tensor;

constexpr int kEpiNone = HXMI_EPI_NONE, kEpiBias = HXMI_EPI_BIAS, kEpiSiluMul = HXMI_EPI_SILU_MUL,
              kEpiBiasGelu = HXMI_EPI_BIAS_GELU_TANH;

// Ordinary dispatch: no torch dispatch or function mode, no functorch or
// tracing layer (they see the torch calls of the Python form).
bool ordinary_dispatch() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty();
}

// The operands of one call: plain GPU tensors of one device.
struct Operands {
  bool ok = ordinary_dispatch();
  c10::DeviceIndex device = -1;

  // The tensor in o, or null for None (only where it may be absent).
  const Tensor* get(PyObject* o, bool optional = false) {
    if (o == Py_None) {
      if (!optional) ok = false;
      return nullptr;
    }
    if (!ok || !THPVariable_CheckExact(o)) {
      ok = false;
      return nullptr;
    }
    static const uint64_t plain = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView,
                                                       c10::DispatchKey::AutogradCUDA,
                                                       c10::DispatchKey::AutocastCUDA})
                                      .raw_repr();
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || (t.key_set().raw_repr() & ~plain) || !t.is_cuda() || !t.has_storage() ||
        (device >= 0 && t.get_device() != device)) {
      ok = false;
      return nullptr;
    }
    device = t.get_device();
    return &t;
  }

  void* stream() const { return (void*)c10::hip::getCurrentHIPStream(device).stream(); }
};

bool half_type(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool bf16(const Tensor& t) { return t.scalar_type() == at::kBFloat16; }

// Rows over the last two dimensions, with unit last stride and no elements in
// common; their leading dimension (a single row may have any stride).
bool lead(const Tensor& t, int64_t& ld) {
  const int64_t d = t.dim(), stride = t.stride(d - 2), width = t.size(d - 1);
  if ((t.stride(d - 1) != 1 && width > 1) || (t.size(d - 2) > 1 && stride < width)) return false;
  ld = std::max<int64_t>({stride, t.size(d - 2) > 1 ? 1 : width, 1});
  return true;
}

// A 2-D view of such rows.
bool rows(const Tensor& t, int64_t& ld) { return t.dim() == 2 && lead(t, ld); }

// A contiguous vector of n elements.
bool vec(const Tensor* t, int64_t n, at::ScalarType type) {
  return !t || (t->dim() == 1 && t->size(0) == n && t->scalar_type() == type && t->is_contiguous());
}

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// The value of a Python float or int; false, with no Python error left, for
// anything else (which the Python form converts or names).
bool number(PyObject* o, long& v) {
  if (!PyLong_Check(o)) return false;
  v = PyLong_AsLong(o);
  if (v != -1 || !PyErr_Occurred()) return true;
  PyErr_Clear();  // (out of range)
  return false;
}
bool number(PyObject* o, double& v) {
  long i;
  if (PyFloat_Check(o)) v = PyFloat_AS_DOUBLE(o);
  else if (number(o, i)) v = (double)i;
  else return false;
  return true;
}

template <typename F>
int unlocked(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f();
  Py_END_ALLOW_THREADS;
  return rc;
}

PyObject* result(int rc, const Tensor& out) {
  if (rc != HXMI_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
}

Tensor like(const Tensor& t, at::IntArrayRef shape) { return at::empty(shape, t.options()); }

#define NOT_PLAIN_UNLESS(cond) \
  do {                         \
    if (!(cond)) Py_RETURN_NONE; \
  } while (0)

// The split-K workspace of one call: hxmi.py's _workspace(bytes, device), which
// keeps one per stream and per graph capture.
PyObject* g_workspace = nullptr;

struct Workspace {
  PyObject* tensor = nullptr;
  void* data = nullptr;
  int64_t bytes = 0;
  bool ok = true;  // false: a Python error is set

  Workspace(int64_t need, const Tensor& like) {
    if (need <= 0) return;
    PyObject* const device = g_workspace ? THPDevice_New(like.device()) : nullptr;
    tensor = device ? PyObject_CallFunction(g_workspace, "LO", (long long)need, device) : nullptr;
    Py_XDECREF(device);
    ok = tensor && THPVariable_Check(tensor);
    if (!ok) return;
    const Tensor& t = THPVariable_Unpack(tensor);
    data = t.data_ptr();
    bytes = t.nbytes();
  }
  ~Workspace() { Py_XDECREF(tensor); }
};

PyObject* set_workspace(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XDECREF(g_workspace);
  g_workspace = fn;
  Py_RETURN_NONE;
}

// gemm(a, b, nt, epilogue, bias, alpha, out)
PyObject* op_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 7);
  Operands in;
  const Tensor *a = in.get(args[0]), *b = in.get(args[1]), *bias = in.get(args[4], true), *o = in.get(args[6], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*a) && b->scalar_type() == a->scalar_type());
  const int nt = PyObject_IsTrue(args[2]);
  long epi;
  double alpha;
  NOT_PLAIN_UNLESS(number(args[3], epi) && number(args[5], alpha));
  int64_t lda, ldb, ldc;
  NOT_PLAIN_UNLESS(rows(*a, lda) && rows(*b, ldb));
  const int64_t M = a->size(0), K = a->size(1), N = b->size(nt ? 0 : 1);
  const int64_t nout = epi == kEpiSiluMul ? N / 2 : N;
  const bool takes_bias = epi == kEpiBias || epi == kEpiBiasGelu;
  NOT_PLAIN_UNLESS(b->size(nt ? 1 : 0) == K && takes_bias == (bias != nullptr) && vec(bias, N, a->scalar_type()));
  NOT_PLAIN_UNLESS(!o || (o->dim() == 2 && o->size(0) == M && o->size(1) == nout &&
                          o->scalar_type() == a->scalar_type()));
  const Tensor out = o ? *o : like(*a, {M, nout});
  NOT_PLAIN_UNLESS(rows(out, ldc));
  const auto fn = bf16(*a) ? hxmi_gemm_bf16 : hxmi_gemm_f16;
  const Workspace ws(hxmi_gemm_workspace_bytes(M, N, K, nt, epi), *a);
  if (!ws.ok) return nullptr;
  void* s = in.stream();
  return result(unlocked([&] {
                  return fn(ptr(a), ptr(b), ptr(&out), ptr(bias), M, N, K, lda, ldb, ldc, nt, (int)epi, (float)alpha,
                            ws.data, ws.bytes, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// bgemm(a, b, nt, epilogue, bias, alpha, out)
PyObject* op_bgemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 7);
  Operands in;
  const Tensor *a = in.get(args[0]), *b = in.get(args[1]), *bias = in.get(args[4], true), *o = in.get(args[6], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*a) && b->scalar_type() == a->scalar_type() && a->dim() == 3 && b->dim() == 3);
  const int nt = PyObject_IsTrue(args[2]);
  long epi;
  double alpha;
  NOT_PLAIN_UNLESS(number(args[3], epi) && number(args[5], alpha));
  int64_t lda, ldb, ldc;
  const int64_t batch = a->size(0), M = a->size(1), K = a->size(2), N = b->size(nt ? 1 : 2);
  const int64_t nout = epi == kEpiSiluMul ? N / 2 : N;
  const bool takes_bias = epi == kEpiBias || epi == kEpiBiasGelu;
  NOT_PLAIN_UNLESS(lead(*a, lda) && lead(*b, ldb) && b->size(0) == batch && b->size(nt ? 2 : 1) == K &&
                   takes_bias == (bias != nullptr) && vec(bias, N, a->scalar_type()));
  NOT_PLAIN_UNLESS(!o || (o->dim() == 3 && o->size(0) == batch && o->size(1) == M && o->size(2) == nout &&
                          o->scalar_type() == a->scalar_type()));
  const Tensor out = o ? *o : like(*a, {batch, M, nout});
  NOT_PLAIN_UNLESS(lead(out, ldc));
  const auto fn = bf16(*a) ? hxmi_bgemm_bf16 : hxmi_bgemm_f16;
  void* s = in.stream();
  return result(unlocked([&] {
                  return fn(ptr(a), ptr(b), ptr(&out), ptr(bias), batch, M, N, K, lda, ldb, ldc, a->stride(0),
                            b->stride(0), out.stride(0), nt, (int)epi, (float)alpha, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// x as rows of its last dimension: contiguous of any rank, or a 2-D view.
bool as_rows(const Tensor& x, int64_t& M, int64_t& K, int64_t& ld) {
  if (x.dim() == 2) {
    M = x.size(0);
    K = x.size(1);
    return rows(x, ld);
  }
  if (x.dim() < 1 || !x.is_contiguous() || x.numel() == 0) return false;
  K = x.size(-1);
  M = x.numel() / K;
  ld = K;
  return true;
}

Tensor rows_like(const Tensor& x, int64_t width) {
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = width;
  return like(x, shape);
}

// linear(x, w, bias, epilogue, out): y = x . w^T, no out of another rank
PyObject* op_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 5);
  Operands in;
  const Tensor *x = in.get(args[0]), *w = in.get(args[1]), *bias = in.get(args[2], true), *o = in.get(args[4], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*x) && w->scalar_type() == x->scalar_type());
  long epi;
  NOT_PLAIN_UNLESS(number(args[3], epi));
  int64_t M, K, ldx, ldw, ldy;
  NOT_PLAIN_UNLESS(as_rows(*x, M, K, ldx) && rows(*w, ldw) && w->size(1) == K);
  const int64_t N = w->size(0), nout = epi == kEpiSiluMul ? N / 2 : N;
  const bool takes_bias = epi == kEpiBias || epi == kEpiBiasGelu;
  NOT_PLAIN_UNLESS(takes_bias == (bias != nullptr) && vec(bias, N, x->scalar_type()));
  NOT_PLAIN_UNLESS(!o || (o->dim() == 2 && o->size(0) == M && o->size(1) == nout &&
                          o->scalar_type() == x->scalar_type() && rows(*o, ldy)));
  const Tensor out = o ? *o : rows_like(*x, nout);
  if (!o) ldy = std::max<int64_t>(nout, 1);
  const auto fn = bf16(*x) ? hxmi_gemm_bf16 : hxmi_gemm_f16;
  const Workspace ws(hxmi_gemm_workspace_bytes(M, N, K, 1, epi), *x);
  if (!ws.ok) return nullptr;
  void* s = in.stream();
  return result(unlocked([&] {
                  return fn(ptr(x), ptr(w), ptr(&out), ptr(bias), M, N, K, ldx, ldw, ldy, 1, epi, 1.f, ws.data,
                            ws.bytes, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// rms_norm_linear(x, w, eps, epilogue, rscale_out, rscale_in, bias): no out
PyObject* op_rms_norm_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 7);
  Operands in;
  const Tensor *x = in.get(args[0]), *w = in.get(args[1]), *rs_out = in.get(args[4], true),
               *rs_in = in.get(args[5], true), *bias = in.get(args[6], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*x) && w->scalar_type() == x->scalar_type());
  double eps;
  long epi;
  NOT_PLAIN_UNLESS(number(args[2], eps) && number(args[3], epi));
  int64_t M, K, ldx, ldw;
  NOT_PLAIN_UNLESS(as_rows(*x, M, K, ldx) && rows(*w, ldw) && w->size(1) == K);
  const int64_t N = w->size(0), nout = epi == kEpiSiluMul ? N / 2 : N;
  NOT_PLAIN_UNLESS(!(rs_out && rs_in) && vec(rs_out, M, at::kFloat) && vec(rs_in, M, at::kFloat) &&
                   vec(bias, N, x->scalar_type()) && (epi == kEpiNone || (epi == kEpiSiluMul && !bias)));
  if (bias) epi = kEpiBias;
  const Tensor out = rows_like(*x, nout);
  const auto fn = bf16(*x) ? hxmi_rmsnorm_linear_bf16 : hxmi_rmsnorm_linear_f16;
  void* s = in.stream();
  return result(unlocked([&] {
                  return fn(ptr(x), ptr(w), ptr(&out), ptr(bias), M, N, K, ldx, ldw, std::max<int64_t>(nout, 1), epi,
                            (float)eps, (float*)ptr(rs_out), (const float*)ptr(rs_in), s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// gemv(x, w, bias, out)
PyObject* op_gemv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 4);
  Operands in;
  const Tensor *x = in.get(args[0]), *w = in.get(args[1]), *bias = in.get(args[2], true), *o = in.get(args[3], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*x) && w->scalar_type() == x->scalar_type());
  int64_t ldx, ldw, ldy;
  NOT_PLAIN_UNLESS(rows(*x, ldx) && rows(*w, ldw) && w->size(1) == x->size(1));
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  NOT_PLAIN_UNLESS(vec(bias, N, x->scalar_type()));
  NOT_PLAIN_UNLESS(!o || (o->dim() == 2 && o->size(0) == M && o->size(1) == N &&
                          o->scalar_type() == x->scalar_type()));
  const Tensor out = o ? *o : like(*x, {M, N});
  NOT_PLAIN_UNLESS(rows(out, ldy));
  const auto fn = bf16(*x) ? hxmi_gemv_bf16 : hxmi_gemv_f16;
  const Workspace ws(hxmi_gemv_workspace_bytes(M, N, K), *x);
  if (!ws.ok) return nullptr;
  void* s = in.stream();
  return result(unlocked([&] {
                  return fn(ptr(x), ptr(w), ptr(bias), ptr(&out), M, N, K, ldx, ldw, ldy, ws.data, ws.bytes, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// w8a16_linear(x, wq, scale, bias, out)
PyObject* op_w8a16_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 5);
  Operands in;
  const Tensor *x = in.get(args[0]), *w = in.get(args[1]), *scale = in.get(args[2]), *bias = in.get(args[3], true),
               *o = in.get(args[4], true);
  NOT_PLAIN_UNLESS(in.ok && x->scalar_type() == at::kHalf && w->scalar_type() == at::kChar);
  int64_t ldx, ldw, ldy;
  NOT_PLAIN_UNLESS(rows(*x, ldx) && rows(*w, ldw) && w->size(1) == x->size(1));
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  NOT_PLAIN_UNLESS(vec(scale, N, at::kHalf) && vec(bias, N, at::kHalf));
  NOT_PLAIN_UNLESS(!o || (o->dim() == 2 && o->size(0) == M && o->size(1) == N && o->scalar_type() == at::kHalf));
  const Tensor out = o ? *o : like(*x, {M, N});
  NOT_PLAIN_UNLESS(rows(out, ldy));
  const Workspace ws(hxmi_w8a16_workspace_bytes(M, N, K), *x);
  if (!ws.ok) return nullptr;
  void* s = in.stream();
  return result(unlocked([&] {
                  return hxmi_gemv_w8a16(ptr(x), (const int8_t*)ptr(w), ptr(scale), ptr(bias), ptr(&out), M, N, K, ldx,
                                         ldw, ldy, ws.data, ws.bytes, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

// rms_norm(x, weight, eps, out)
PyObject* op_rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 4);
  Operands in;
  const Tensor *x = in.get(args[0]), *w = in.get(args[1]), *o = in.get(args[3], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*x) && x->is_contiguous() && x->dim() >= 1 && x->numel() > 0);
  double eps;
  NOT_PLAIN_UNLESS(number(args[2], eps));
  const int64_t cols = x->size(-1), nrows = x->numel() / cols;
  NOT_PLAIN_UNLESS(w && vec(w, cols, x->scalar_type()));
  NOT_PLAIN_UNLESS(!o || (o->sizes() == x->sizes() && o->scalar_type() == x->scalar_type() && o->is_contiguous()));
  const Tensor out = o ? *o : like(*x, x->sizes());
  const auto fn = bf16(*x) ? hxmi_rmsnorm_bf16 : hxmi_rmsnorm_f16;
  void* s = in.stream();
  return result(
      unlocked([&] { return fn(ptr(x), ptr(w), ptr(&out), nrows, cols, cols, cols, (float)eps, s); }), out);
  END_HANDLE_TH_ERRORS
}

// softmax(x, scale, out)
PyObject* op_softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 3);
  Operands in;
  const Tensor *x = in.get(args[0]), *o = in.get(args[2], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*x) && x->is_contiguous() && x->dim() >= 1 && x->numel() > 0);
  double scale;
  NOT_PLAIN_UNLESS(number(args[1], scale));
  const int64_t cols = x->size(-1), nrows = x->numel() / cols;
  NOT_PLAIN_UNLESS(!o || (o->sizes() == x->sizes() && o->scalar_type() == x->scalar_type() && o->is_contiguous()));
  const Tensor out = o ? *o : like(*x, x->sizes());
  const auto fn = bf16(*x) ? hxmi_softmax_bf16 : hxmi_softmax_f16;
  void* s = in.stream();
  return result(unlocked([&] { return fn(ptr(x), ptr(&out), nrows, cols, cols, cols, (float)scale, s); }), out);
  END_HANDLE_TH_ERRORS
}

// The leading dimensions of [..., S, D] as one: rows ld apart, slices `slice`
// apart, all rows on the 16-byte grid.
bool slices(const Tensor& t, int64_t& ld, int64_t& slice) {
  const int64_t d = t.dim();
  if (t.stride(d - 1) != 1) return false;
  int64_t next = -1;  // stride the next outer dimension (of more than one slice) must have
  slice = 0;
  for (int64_t i = d - 3; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (t.stride(i) <= 0) return false;  // (expanded)
    if (next < 0) slice = t.stride(i);
    else if (t.stride(i) != next) return false;
    next = t.stride(i) * t.size(i);
  }
  ld = t.size(d - 2) == 1 ? t.size(d - 1) : t.stride(d - 2);
  if (slice == 0) slice = t.size(d - 2) * ld;
  return ld >= t.size(d - 1) && slice >= 0 && ld % 8 == 0 && slice % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0 &&
         (t.size(d - 2) - 1) * ld + t.size(d - 1) <= int64_t(1) << 30;
}

// An additive fp16 mask with q's leading dimensions (or 1 in their place, or
// none of the outer ones): rows ld apart, `group` query slices a mask slice, those `slice` apart.
bool mask_slices(const Tensor& m, const Tensor& q, int64_t Skv, int64_t& ld, int64_t& slice, int64_t& group) {
  const int64_t r = q.dim(), off = r - m.dim();
  if (m.scalar_type() != at::kHalf || off < 0 || off > r - 2 || m.size(-1) != Skv || m.size(-2) != q.size(-2) ||
      (m.stride(-1) != 1 && Skv > 1) || (uintptr_t)m.data_ptr() % 2)
    return false;
  ld = m.stride(-2);
  slice = 0;
  group = 1;
  int64_t next = -1;  // stride the next outer dimension must have
  bool broadcast = false;
  for (int64_t i = r - 3; i >= 0; --i) {
    const int64_t sz = i < off ? 1 : m.size(i - off);
    if (sz != 1 && sz != q.size(i)) return false;
    if (q.size(i) == 1) continue;
    const int64_t st = sz == 1 ? 0 : m.stride(i - off);
    if (st == 0 && next < 0) {  // (the innermost ones only)
      group *= q.size(i);
      broadcast = true;
      continue;
    }
    if (st <= 0 || (next >= 0 && st != next)) return false;
    if (next < 0) slice = st;
    next = st * q.size(i);
  }
  if (next < 0 && broadcast) group = 1;  // one slice for all
  return ld >= Skv;
}

// Whether the address ranges of two tensors' elements meet (neither is empty).
bool overlap(const Tensor& a, const Tensor& b) {
  const auto end = [](const Tensor& t) {
    int64_t last = 0;
    for (int64_t i = 0; i < t.dim(); ++i) last += (t.size(i) - 1) * t.stride(i);
    return (uintptr_t)t.data_ptr() + (last + 1) * t.element_size();
  };
  return (uintptr_t)a.data_ptr() < end(b) && (uintptr_t)b.data_ptr() < end(a);
}

// attention(q, k, v, scale or None, causal, mask or None, out or None)
PyObject* op_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NOT_PLAIN_UNLESS(n == 7);
  Operands in;
  const Tensor *q = in.get(args[0]), *k = in.get(args[1]), *v = in.get(args[2]), *m = in.get(args[5], true),
               *o = in.get(args[6], true);
  NOT_PLAIN_UNLESS(in.ok && half_type(*q) && k->scalar_type() == q->scalar_type() &&
                   v->scalar_type() == q->scalar_type());
  const int64_t r = q->dim();
  NOT_PLAIN_UNLESS(r >= 3 && k->dim() == r && v->sizes() == k->sizes() && q->numel() > 0 && k->numel() > 0);
  const int64_t S = q->size(-2), Skv = k->size(-2), D = q->size(-1), H = q->size(-3), Hkv = k->size(-3);
  NOT_PLAIN_UNLESS(k->size(-1) == D && D % 8 == 0 && D <= 128 && H % Hkv == 0 &&
                   q->sizes().slice(0, r - 3) == k->sizes().slice(0, r - 3));
  double scale = 1.0 / std::sqrt((double)D);
  long causal;
  NOT_PLAIN_UNLESS((args[3] == Py_None || number(args[3], scale)) && number(args[4], causal));
  NOT_PLAIN_UNLESS(scale > 0 && std::isfinite((float)scale) && causal >= 0 && causal <= 2);
  int64_t ldq, ldk, ldv, sq, sk, sv;
  NOT_PLAIN_UNLESS(slices(*q, ldq, sq) && slices(*k, ldk, sk) && slices(*v, ldv, sv));
  int64_t ldm = 0, sm = 0, mg = 1;
  NOT_PLAIN_UNLESS(!m || mask_slices(*m, *q, Skv, ldm, sm, mg));
  int64_t ldo = D, so = S * D;
  NOT_PLAIN_UNLESS(!o || (o->sizes() == q->sizes() && o->scalar_type() == q->scalar_type() && slices(*o, ldo, so) &&
                          ((!bf16(*q) && (D == 64 || D == 128)) ||
                           (o->is_contiguous() && !overlap(*o, *k) && !overlap(*o, *v) && !(m && overlap(*o, *m)) &&
                            (!overlap(*o, *q) || (q->data_ptr() == o->data_ptr() && q->is_contiguous()))))));
  const Tensor out = o ? *o : like(*q, q->sizes());
  void* s = in.stream();
  return result(unlocked([&] {
                  return hxmi_attention_ex(bf16(*q), ptr(q), ptr(k), ptr(v), ptr(&out), q->numel() / (S * D), S, Skv, D,
                                           ldq, ldk, ldv, ldo, sq, sk, sv, so, H / Hkv, ptr(m), ldm, sm, mg, (int)causal,
                                           (float)scale, s);
                }),
                out);
  END_HANDLE_TH_ERRORS
}

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))op_##name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {ENTRY(gemm),         ENTRY(bgemm),    ENTRY(linear),  ENTRY(rms_norm_linear), ENTRY(gemv),
                          ENTRY(w8a16_linear), ENTRY(rms_norm), ENTRY(softmax), ENTRY(attention),
                          {"set_workspace", set_workspace, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "hxmi_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_hxmi_torch(void) { return PyModule_Create(&kModule); }
