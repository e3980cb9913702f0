// Native host path of the torch wrappers.
//
// A decode step calls its norms, projections and attention on tensors so small
// that the call is bound by the host: checking the arguments in Python,
// allocating through torch's Python bindings and building ctypes arguments
// took 8-15 us per call, against 3-4 us for the launch itself.  The functions
// here do the same for the usual case of each op -- plain GPU tensors on the
// current device in layouts that need no copy or cast -- and return None for
// anything else (other layouts, dtypes or devices, tensor subclasses, function
// modes, wrong arguments), which the wrapper then serves or rejects in Python.
// The kernels and their arguments are those of the Python path, but for a
// softmax of a single row (see there).
// add_rms_norm bf16 (8, 4096) 15.1 -> 5.65 us per call, silu of a few rows 7.1
// -> 4.4, softmax 10.7 -> 4.6.
//
// Entry points of the kernel library are handed over by address (init), so
// both paths call the one loaded library.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/DispatchKeySet.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../../../include/ntops_amd.h"

namespace {

decltype(&ntops_unary) f_unary;
decltype(&ntops_softmax) f_softmax;
decltype(&ntops_rms_norm) f_rms_norm;
decltype(&ntops_layer_norm) f_layer_norm;
decltype(&ntops_add_rms_norm) f_add_rms_norm;
decltype(&ntops_rope_qk) f_rope_qk;
decltype(&ntops_gemm_ws) f_gemm_ws;
decltype(&ntops_gemm_workspace) f_gemm_workspace;
decltype(&ntops_sdpa_ws) f_sdpa_ws;
decltype(&ntops_sdpa_workspace) f_sdpa_workspace;
decltype(&ntops_copy2) f_copy2;
bool ready = false;
PyObject* get_device = nullptr;  // torch._C._cuda_getDevice
PyObject* get_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

// The dtype's code in the C ABI (F32 / F16 / BF16), else -1.
int code16_32(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return NTOPS_F32;
    case at::kHalf: return NTOPS_F16;
    case at::kBFloat16: return NTOPS_BF16;
    default: return -1;
  }
}

// The tensor of a torch.Tensor or Parameter that is an ordinary dense GPU
// tensor -- no subclass, wrapper of a transform, or lazily applied operation;
// else null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const uint64_t allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA,
                           c10::DispatchKey::AutocastCUDA})
          .raw_repr();
  if (!t.defined() || !t.is_cuda() || (t.key_set().raw_repr() & ~allowed) != 0) return nullptr;
  return &t;
}

// Current device and its current stream; false on any error (cleared).
bool current(int64_t& device, void*& stream) {
  PyObject* d = PyObject_CallNoArgs(get_device);
  if (!d) {
    PyErr_Clear();
    return false;
  }
  PyObject* s = PyObject_CallOneArg(get_stream, d);
  device = PyLong_AsLongLong(d);
  Py_DECREF(d);
  if (!s) {
    PyErr_Clear();
    return false;
  }
  stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool usable() { return ready && at::impl::PythonTorchFunctionTLS::stack_len() == 0; }

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

at::Tensor new_like(const at::Tensor& t, c10::IntArrayRef sizes) {
  return at::empty(sizes, at::TensorOptions().dtype(t.dtype()).device(t.device()));
}
at::Tensor workspace(const at::Tensor& t, int64_t bytes) {
  return at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(t.device()));
}

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }
PyObject* wrap2(const at::Tensor& a, const at::Tensor& b) {
  PyObject* x = wrap(a);
  PyObject* y = x ? wrap(b) : nullptr;
  PyObject* r = y ? PyTuple_Pack(2, x, y) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  return r;
}
PyObject* none() { Py_RETURN_NONE; }

// The interpreter is free while a call allocates and launches (either may wait
// for the device), as it is in torch's own allocations and in ctypes calls;
// no Python object is touched inside.
class NoGil {
 public:
  NoGil() : state_(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(state_); }
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;

 private:
  PyThreadState* state_;
};

// A Python float or int (not a bool) as a double.
bool number(PyObject* o, double& v) {
  if (PyFloat_CheckExact(o)) {
    v = PyFloat_AS_DOUBLE(o);
    return true;
  }
  if (PyLong_CheckExact(o)) {
    v = PyLong_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    return true;
  }
  return false;
}

// Elements of the normalized dims when `shape` (an int, or a tuple or list of
// ints) names the input's last dims; else -1.
int64_t norm_cols(const at::Tensor& x, PyObject* shape) {
  const auto sizes = x.sizes();
  const int64_t nd = static_cast<int64_t>(sizes.size());
  if (PyLong_CheckExact(shape)) {
    const int64_t n = PyLong_AsLongLong(shape);
    if (n == -1 && PyErr_Occurred()) PyErr_Clear();
    return nd >= 1 && sizes[nd - 1] == n ? n : -1;
  }
  if (!PyTuple_Check(shape) && !PyList_CheckExact(shape)) return -1;
  const Py_ssize_t k = PySequence_Fast_GET_SIZE(shape);
  if (k < 1 || k > nd) return -1;
  int64_t cols = 1;
  for (Py_ssize_t i = 0; i < k; ++i) {
    PyObject* v = PySequence_Fast_GET_ITEM(shape, i);
    if (!PyLong_CheckExact(v)) return -1;
    const int64_t n = PyLong_AsLongLong(v);
    if (n == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return -1;
    }
    if (sizes[nd - k + i] != n) return -1;
    cols *= n;
  }
  return cols;
}

// A norm's weight or bias as one contiguous row of the normalized dims, of the
// input's dtype or fp32; `o` None leaves p null.  False: the Python path.
bool norm_param(PyObject* o, const at::Tensor& x, int64_t cols, int dev, const at::Tensor*& p) {
  p = nullptr;
  if (o == Py_None) return true;
  p = plain(o);
  if (!p || p->get_device() != dev || !p->is_contiguous() || p->numel() != cols) return false;
  if (p->scalar_type() != x.scalar_type() && p->scalar_type() != at::kFloat) return false;
  const auto ps = p->sizes(), xs = x.sizes();
  if (ps.size() > xs.size()) return false;
  for (size_t i = 0; i < ps.size(); ++i)
    if (ps[i] != xs[xs.size() - ps.size() + i]) return false;
  return true;
}

// Whatever goes wrong (out of memory, say) is left to the Python path, which
// meets it again and raises what it always has.
#define NTOPS_TRY try {
#define NTOPS_END       \
  }                     \
  catch (...) {         \
    PyErr_Clear();      \
    return none();      \
  }

// unary(op, input): a contiguous floating input into empty_like(input)
PyObject* unary(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  if (n != 2 || !usable()) return none();
  const at::Tensor* x = plain(a[1]);
  int64_t dev;
  void* st;
  if (!x || code16_32(*x) < 0 || !x->is_contiguous() || x->dim() > 16 || !current(dev, st) || x->get_device() != dev)
    return none();
  const int op = static_cast<int>(PyLong_AsLong(a[0]));
  at::Tensor y;
  int rc;
  {
    NoGil free;
    y = at::empty_like(*x);
    rc = f_unary(op, code16_32(*x), static_cast<int>(x->dim()), x->sizes().data(), x->data_ptr(), x->strides().data(),
                 y.data_ptr(), y.strides().data(), st);
  }
  return rc == NTOPS_OK ? wrap(y) : none();
  NTOPS_END
}

// softmax(input, dim).  A single row has its length as the row stride here,
// where the Python path's merged strides give 1: it takes the row kernels (bf16
// (1, 131072) 70.6 -> 18.6 us), whose sums round in another order.
PyObject* softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  if (n != 2 || !usable() || !PyLong_CheckExact(a[1])) return none();
  const at::Tensor* x = plain(a[0]);
  int64_t dev;
  void* st;
  if (!x || code16_32(*x) < 0 || !x->is_contiguous() || x->dim() < 1 || !current(dev, st) || x->get_device() != dev)
    return none();
  int64_t dim = PyLong_AsLongLong(a[1]);
  if (dim == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  if (dim < -x->dim() || dim >= x->dim()) return none();
  if (dim < 0) dim += x->dim();
  int64_t outer = 1, inner = 1;
  for (int64_t i = 0; i < dim; ++i) outer *= x->size(i);
  for (int64_t i = dim + 1; i < x->dim(); ++i) inner *= x->size(i);
  const int64_t size = x->size(dim);
  const int64_t strides[3] = {size * inner, inner, 1};
  at::Tensor y;
  int rc;
  {
    NoGil free;
    y = new_like(*x, x->sizes());
    rc = f_softmax(code16_32(*x), code16_32(*x), outer, size, inner, x->data_ptr(), strides, y.data_ptr(), strides, st);
  }
  return rc == NTOPS_OK ? wrap(y) : none();
  NTOPS_END
}

// rms_norm(input, normalized_shape, weight, eps)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  double eps;
  if (n != 4 || !usable() || !number(a[3], eps)) return none();
  const at::Tensor* x = plain(a[0]);
  const at::Tensor* w;
  int64_t dev;
  void* st;
  if (!x || code16_32(*x) < 0 || !x->is_contiguous() || !aligned16(*x) || x->numel() == 0 || !current(dev, st) ||
      x->get_device() != dev)
    return none();
  const int64_t cols = norm_cols(*x, a[1]);
  if (cols <= 0 || !norm_param(a[2], *x, cols, static_cast<int>(dev), w)) return none();
  at::Tensor y;
  int rc;
  {
    NoGil free;
    y = new_like(*x, x->sizes());
    rc = f_rms_norm(code16_32(*x), x->numel() / cols, cols, x->data_ptr(), cols, w ? w->data_ptr() : nullptr, 0,
                    w ? code16_32(*w) : code16_32(*x), eps, y.data_ptr(), cols, st);
  }
  return rc == NTOPS_OK ? wrap(y) : none();
  NTOPS_END
}

// layer_norm(input, normalized_shape, weight, bias, eps)
PyObject* layer_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  double eps;
  if (n != 5 || !usable() || !number(a[4], eps)) return none();
  const at::Tensor* x = plain(a[0]);
  const at::Tensor *w, *b;
  int64_t dev;
  void* st;
  if (!x || code16_32(*x) < 0 || !x->is_contiguous() || !aligned16(*x) || x->numel() == 0 || !current(dev, st) ||
      x->get_device() != dev)
    return none();
  const int64_t cols = norm_cols(*x, a[1]);
  if (cols <= 0 || !norm_param(a[2], *x, cols, static_cast<int>(dev), w) ||
      !norm_param(a[3], *x, cols, static_cast<int>(dev), b))
    return none();
  int code = code16_32(*x);
  if (w) code = code16_32(*w);
  if (b) {
    if (w && b->scalar_type() != w->scalar_type()) return none();
    code = code16_32(*b);
  }
  at::Tensor y;
  int rc;
  {
    NoGil free;
    y = new_like(*x, x->sizes());
    rc = f_layer_norm(code16_32(*x), x->numel() / cols, cols, x->data_ptr(), cols, w ? w->data_ptr() : nullptr,
                      b ? b->data_ptr() : nullptr, 0, code, eps, y.data_ptr(), cols, st);
  }
  return rc == NTOPS_OK ? wrap(y) : none();
  NTOPS_END
}

// add_rms_norm(input, residual, normalized_shape, weight, eps)
PyObject* add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  double eps;
  if (n != 5 || !usable() || !number(a[4], eps)) return none();
  const at::Tensor *x = plain(a[0]), *r = plain(a[1]);
  const at::Tensor* w;
  int64_t dev;
  void* st;
  if (!x || !r || code16_32(*x) < 0 || !x->is_contiguous() || !r->is_contiguous() || !aligned16(*x) || !aligned16(*r) ||
      x->numel() == 0 || r->scalar_type() != x->scalar_type() || r->sizes() != x->sizes() || !current(dev, st) ||
      x->get_device() != dev || r->get_device() != dev)
    return none();
  const int64_t cols = norm_cols(*x, a[2]);
  if (cols <= 0 || !norm_param(a[3], *x, cols, static_cast<int>(dev), w)) return none();
  at::Tensor y, h;
  int rc;
  {
    NoGil free;
    y = new_like(*x, x->sizes());
    h = new_like(*x, x->sizes());
    rc = f_add_rms_norm(code16_32(*x), x->numel() / cols, cols, x->data_ptr(), cols, r->data_ptr(), cols,
                        w ? w->data_ptr() : nullptr, 0, w ? code16_32(*w) : code16_32(*x), eps, y.data_ptr(), cols,
                        h.data_ptr(), cols, st);
  }
  return rc == NTOPS_OK ? wrap2(y, h) : none();
  NTOPS_END
}

// rope_qk(q, k, sin, cos, interleaved)
PyObject* rope_qk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  if (n != 5 || !usable() || !PyBool_Check(a[4])) return none();
  const at::Tensor* t[4];
  int64_t dev;
  void* st;
  if (!current(dev, st)) return none();
  for (int i = 0; i < 4; ++i) {
    t[i] = plain(a[i]);
    if (!t[i] || t[i]->get_device() != dev || t[i]->dim() != (i < 2 ? 4 : 2) ||
        t[i]->scalar_type() != t[0]->scalar_type())
      return none();
  }
  const at::Tensor &q = *t[0], &k = *t[1], &sn = *t[2], &cs = *t[3];
  const int64_t B = q.size(0), S = q.size(1), D = q.size(3), tw = sn.size(1);
  if (code16_32(q) < 0 || k.size(0) != B || k.size(1) != S || k.size(3) != D || D % 2 != 0 || sn.size(0) < S ||
      cs.size(0) < S || (tw != D && tw != D / 2) || cs.size(1) != tw || sn.stride(1) != 1 || cs.stride(1) != 1 ||
      sn.stride(0) != cs.stride(0))
    return none();
  const int interleaved = a[4] == Py_True ? 1 : 0;
  at::Tensor qo, ko;
  int rc;
  {
    NoGil free;
    qo = at::empty_like(q);
    ko = at::empty_like(k);
    rc = f_rope_qk(code16_32(q), B, S, q.size(2), k.size(2), D, q.data_ptr(), q.strides().data(), k.data_ptr(),
                   k.strides().data(), sn.data_ptr(), cs.data_ptr(), sn.stride(0), tw, interleaved, qo.data_ptr(),
                   qo.strides().data(), ko.data_ptr(), ko.strides().data(), st);
  }
  return rc == NTOPS_OK ? wrap2(qo, ko) : none();
  NTOPS_END
}

// mm(a, b) / addmm(c, a, b, beta, alpha): a K-major, b N- or K-major, both in
// 16-byte rows (what the matrix-core kernels read in place)
PyObject* gemm(const at::Tensor* c, PyObject* pa, PyObject* pb, double beta, double alpha) {
  const at::Tensor *x = plain(pa), *w = plain(pb);
  int64_t dev;
  void* st;
  if (!x || !w || code16_32(*x) < 0 || x->dim() != 2 || w->dim() != 2 || w->scalar_type() != x->scalar_type() ||
      x->size(1) != w->size(0) || !aligned16(*x) || !aligned16(*w) || !current(dev, st) || x->get_device() != dev ||
      w->get_device() != dev)
    return none();
  const int64_t M = x->size(0), K = x->size(1), N = w->size(1);
  const int64_t unit = x->scalar_type() == at::kFloat ? 4 : 8;
  if (M <= 0 || N <= unit || K <= 0 || K % unit != 0 || x->stride(1) != 1 || x->stride(0) % unit != 0) return none();
  const bool n_major = w->stride(1) == 1 && w->stride(0) % unit == 0 && N % unit == 0;
  const bool k_major = w->stride(0) == 1 && w->stride(1) != 1 && w->stride(1) % unit == 0;
  if (!n_major && !k_major) return none();
  int64_t cst[3] = {0, 0, 0};
  if (c) {
    if (c->scalar_type() != x->scalar_type() || c->get_device() != dev || c->dim() < 1 || c->dim() > 2) return none();
    const int64_t cn = c->size(c->dim() - 1), cm = c->dim() == 2 ? c->size(0) : 1;
    if ((cn != N && cn != 1) || (cm != M && cm != 1)) return none();
    cst[2] = cn == 1 && N != 1 ? 0 : c->stride(c->dim() - 1);
    cst[1] = cm == 1 && M != 1 ? 0 : c->dim() == 2 ? c->stride(0) : 0;
  }
  const int code = code16_32(*x);
  const int64_t ast[3] = {0, x->stride(0), 1}, bst[3] = {0, w->stride(0), w->stride(1)}, dst[3] = {0, N, 1};
  at::Tensor out;
  int rc;
  {
    NoGil free;
    out = new_like(*x, {M, N});
    const int64_t bytes = f_gemm_workspace(code, 1, M, N, K);
    at::Tensor ws;
    if (bytes > 0) ws = workspace(*x, bytes);
    rc = f_gemm_ws(code, 1, M, N, K, x->data_ptr(), ast, w->data_ptr(), bst, c ? c->data_ptr() : nullptr,
                   c ? cst : nullptr, alpha, beta, out.data_ptr(), dst, bytes > 0 ? ws.data_ptr() : nullptr, bytes, st);
  }
  return rc == NTOPS_OK ? wrap(out) : none();
}
PyObject* mm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  if (n != 2 || !usable()) return none();
  return gemm(nullptr, a[0], a[1], 0.0, 1.0);
  NTOPS_END
}
PyObject* addmm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  double beta, alpha;
  if (n != 5 || !usable() || !number(a[3], beta) || !number(a[4], alpha) || beta == 0.0) return none();
  const at::Tensor* c = plain(a[0]);
  return c ? gemm(c, a[1], a[2], beta, alpha) : none();
  NTOPS_END
}

// sdpa(q, k, v, mask, causal mode, scale (None: 1 / sqrt(D)), gqa, present_key,
// present_value, present_key_slot, present_value_slot)
PyObject* sdpa(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NTOPS_TRY
  if (n != 11 || !usable() || !PyLong_CheckExact(a[4]) || !PyBool_Check(a[6])) return none();
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  int64_t dev;
  void* st;
  if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || code16_32(*q) < 0 ||
      k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || !current(dev, st) ||
      q->get_device() != dev || k->get_device() != dev || v->get_device() != dev)
    return none();
  const int64_t B = q->size(0), Hq = q->size(1), Sq = q->size(2), D = q->size(3), Hk = k->size(1), Sk = k->size(2);
  if (k->size(0) != B || v->size(0) != B || v->size(1) != Hk || v->size(2) != Sk || k->size(3) != D ||
      v->size(3) != D || D <= 0 || Hk <= 0 || (a[6] == Py_True ? Hq % Hk != 0 : Hq != Hk))
    return none();
  double scale;
  if (a[5] == Py_None)
    scale = 1.0 / std::sqrt(static_cast<double>(D));
  else if (!number(a[5], scale))
    return none();
  const at::Tensor* m = nullptr;
  int64_t mst[4] = {0, 0, 0, 0};
  int mcode = 0;
  if (a[3] != Py_None) {
    m = plain(a[3]);
    if (!m || m->get_device() != dev || m->dim() < 1 || m->dim() > 4) return none();
    mcode = m->scalar_type() == at::kBool ? NTOPS_BOOL : code16_32(*m);
    if (mcode < 0) return none();
    const int64_t full[4] = {B, Hq, Sq, Sk};
    for (int64_t i = 0; i < m->dim(); ++i) {
      const int64_t d = 4 - m->dim() + i;
      if (m->size(i) != full[d] && m->size(i) != 1) return none();
      mst[d] = m->size(i) == 1 && full[d] != 1 ? 0 : m->stride(i);
    }
  }
  const int causal = static_cast<int>(PyLong_AsLong(a[4]));
  const at::Tensor* p[4] = {};
  if (a[7] != Py_None) {
    for (int i = 0; i < 4; ++i) {  // key, value, key slot, value slot
      p[i] = plain(a[7 + i]);
      if (!p[i] || p[i]->get_device() != dev || p[i]->scalar_type() != p[0]->scalar_type() || p[i]->dim() > 16 ||
          code16_32(*p[i]) < 0 || p[i]->sizes() != p[0]->sizes())
        return none();
    }
  }
  const int code = code16_32(*q);
  at::Tensor out;
  int rc = NTOPS_OK;
  {
    NoGil free;
    if (p[0])
      rc = f_copy2(code16_32(*p[0]), static_cast<int>(p[0]->dim()), p[0]->sizes().data(), p[0]->data_ptr(),
                   p[0]->strides().data(), p[2]->data_ptr(), p[2]->strides().data(), p[1]->data_ptr(),
                   p[1]->strides().data(), p[3]->data_ptr(), p[3]->strides().data(), st);
    if (rc == NTOPS_OK) {
      out = new_like(*q, q->sizes());
      int64_t bytes = 0;
      at::Tensor ws;
      if (!m && Sq <= 16) bytes = f_sdpa_workspace(code, B, Hq, Hk, Sq, Sk, D, 0);
      if (bytes > 0) ws = workspace(*q, bytes);
      rc = f_sdpa_ws(code, B, Hq, Hk, Sq, Sk, D, q->data_ptr(), q->strides().data(), k->data_ptr(), k->strides().data(),
                     v->data_ptr(), v->strides().data(), m ? m->data_ptr() : nullptr, mcode, m ? mst : nullptr, causal,
                     scale, out.data_ptr(), out.strides().data(), bytes > 0 ? ws.data_ptr() : nullptr, bytes, st);
    }
  }
  return rc == NTOPS_OK ? wrap(out) : none();
  NTOPS_END
}

// init({name: address}, get_device, get_stream)
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyDict_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "init(addresses, get_device, get_stream)");
    return nullptr;
  }
  ready = false;
  const auto set = [&](const char* name, auto& fn) {
    PyObject* v = PyDict_GetItemString(a[0], name);
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(p);
    return p != nullptr;
  };
  const bool all = set("ntops_unary", f_unary) & set("ntops_softmax", f_softmax) & set("ntops_rms_norm", f_rms_norm) &
                   set("ntops_layer_norm", f_layer_norm) & set("ntops_add_rms_norm", f_add_rms_norm) &
                   set("ntops_rope_qk", f_rope_qk) & set("ntops_gemm_ws", f_gemm_ws) &
                   set("ntops_gemm_workspace", f_gemm_workspace) & set("ntops_sdpa_ws", f_sdpa_ws) &
                   set("ntops_sdpa_workspace", f_sdpa_workspace) & set("ntops_copy2", f_copy2);
  if (PyErr_Occurred()) return nullptr;
  Py_INCREF(a[1]);
  Py_INCREF(a[2]);
  Py_XDECREF(get_device);
  Py_XDECREF(get_stream);
  get_device = a[1];
  get_stream = a[2];
  ready = all;
  return PyBool_FromLong(all);
}

#define NTOPS_M(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {NTOPS_M(init),         NTOPS_M(unary),   NTOPS_M(softmax), NTOPS_M(rms_norm), NTOPS_M(layer_norm),
                         NTOPS_M(add_rms_norm), NTOPS_M(rope_qk), NTOPS_M(mm),      NTOPS_M(addmm),    NTOPS_M(sdpa),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", "native host path of the torch wrappers", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }
