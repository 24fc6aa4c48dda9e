// Host half of the torch mirror (tattletale_amd/qlinear.py) in native code: from torch tensors to one call of the
// C ABI.  A decode step is dozens of these calls of 3 to 5 us of GPU time each, and the interpreter's share of a
// call -- tensor properties one by one, the argument struct, the output tensor, the stream, the foreign-function
// conversion -- was 7 of the 10 us a call took on the host; here it is below 2 us, and what is left is the launch.
//
// Nothing is kept between calls: every call reads its tensors anew.  Each function returns the output tensor(s), a
// negative ttq_status the library answered with, or 1 where the tensors do not meet the preconditions below: the
// caller then takes its own path, which raises the error that names what is wrong.  (That path makes the same call of
// the library, and serves all of them where this extension is not built.)
#include <torch/extension.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "../../include/ttq.h"

namespace {

// Entry points of libttq_hip.so, handed over by address (bind): this extension does not open the library itself.
decltype(&ttq_linear_forward) p_linear_forward = nullptr;
decltype(&ttq_linear_forward_ws) p_linear_forward_ws = nullptr;
decltype(&ttq_rmsnorm) p_rmsnorm = nullptr;
decltype(&ttq_silu_and_mul) p_silu_and_mul = nullptr;
decltype(&ttq_gemv_q4_k_silu_mul) p_gemv_q4_k_silu_mul = nullptr;
decltype(&ttq_gemm_q4_k_silu_mul) p_gemm_q4_k_silu_mul = nullptr;

PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
    return nullptr;
  }
  void* p[6];
  for (int i = 0; i < 6; i++) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  p_linear_forward = reinterpret_cast<decltype(p_linear_forward)>(p[0]);
  p_linear_forward_ws = reinterpret_cast<decltype(p_linear_forward_ws)>(p[1]);
  p_rmsnorm = reinterpret_cast<decltype(p_rmsnorm)>(p[2]);
  p_silu_and_mul = reinterpret_cast<decltype(p_silu_and_mul)>(p[3]);
  p_gemv_q4_k_silu_mul = reinterpret_cast<decltype(p_gemv_q4_k_silu_mul)>(p[4]);
  p_gemm_q4_k_silu_mul = reinterpret_cast<decltype(p_gemm_q4_k_silu_mul)>(p[5]);
  Py_RETURN_NONE;
}

PyObject* answer(long status) { return PyLong_FromLong(status); }

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return TTQ_F32;
    case at::kHalf: return TTQ_F16;
    case at::kBFloat16: return TTQ_BF16;
    default: return -1;
  }
}

// A contiguous tensor on a GPU; null for anything else.
const at::Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous() ? &t : nullptr;
}

// Binds the tensors' device and its current stream for one call.
struct OnDevice {
  explicit OnDevice(c10::Device d) : guard(d), stream(c10::hip::getCurrentHIPStream(d.index()).stream()) {}
  c10::DeviceGuard guard;
  hipStream_t stream;
};

// The part of a call that other Python threads need not wait for: the output tensors, whose allocation may go to the
// device or wait for another stream's block, and the library's call.  Back under the lock on an exception too.
template <class Call>
int released(Call call) {
  struct Lock {
    PyThreadState* state = PyEval_SaveThread();
    ~Lock() { PyEval_RestoreThread(state); }
  } lock;
  return call();
}

bool as_int64(PyObject* o, int64_t& v) {
  v = PyLong_AsLongLong(o);
  return !(v == -1 && PyErr_Occurred());
}

// An output with x's leading dimensions and device: described while x is read, made where the lock is released.
struct Output {
  Output(const at::Tensor& x, int64_t last, at::ScalarType type)
      : sizes(x.sizes().begin(), x.sizes().end()), options(x.options().dtype(type).requires_grad(false)) {
    sizes.back() = last;
  }
  at::Tensor make() const { return at::empty(sizes, options); }
  c10::SmallVector<int64_t, 6> sizes;
  at::TensorOptions options;
};

// (qweight, suh, svh, bias, format, n_in, n_out, bits, codebook, precision, x, out_dtype or None, workspace or None)
PyObject* linear_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 13 || !p_linear_forward) return answer(1);
  const at::Tensor *q = gpu_tensor(a[0]), *x = gpu_tensor(a[10]), *ws = nullptr;
  if (!q || !x || q->device() != x->device() || x->dim() == 0) return answer(1);
  if (a[12] != Py_None && (!(ws = gpu_tensor(a[12])) || ws->device() != x->device())) return answer(1);
  int64_t v[6];
  for (int i = 0; i < 6; i++)
    if (!as_int64(a[4 + i], v[i])) return nullptr;
  ttq_qlinear layer{};
  layer.format = (int32_t)v[0];
  layer.n_in = v[1];
  layer.n_out = v[2];
  layer.bits = (int32_t)v[3];
  layer.codebook = (int32_t)v[4];
  layer.precision = (int32_t)v[5];
  layer.qweight = q->data_ptr();
  if (layer.n_in <= 0 || layer.n_out < 0 || x->size(-1) != layer.n_in) return answer(1);
  const void** vectors[3] = {&layer.suh, &layer.svh, &layer.bias};
  for (int i = 0; i < 3; i++) {
    if (a[1 + i] == Py_None) continue;
    if (!THPVariable_Check(a[1 + i])) return answer(1);
    const at::Tensor& t = THPVariable_Unpack(a[1 + i]);
    *vectors[i] = t.data_ptr();
    if (i == 2 && (layer.bias_dtype = dtype_code(t.scalar_type())) < 0) return answer(1);
  }
  at::ScalarType yt = x->scalar_type();
  if (a[11] != Py_None) {
    if (!THPDtype_Check(a[11])) return answer(1);
    yt = reinterpret_cast<THPDtype*>(a[11])->scalar_type;
  }
  const int xd = dtype_code(x->scalar_type()), yd = dtype_code(yt);
  if (xd < 0 || yd < 0) return answer(1);
  const int64_t m = x->numel() / layer.n_in;
  const void* xp = x->data_ptr();
  void* wp = ws ? ws->data_ptr() : nullptr;
  const int64_t bytes = ws ? (int64_t)ws->nbytes() : 0;
  const c10::Device device = x->device();
  const Output out(*x, layer.n_out, yt);
  at::Tensor y;
  const int rc = released([&] {
    const OnDevice on(device);
    y = out.make();
    return ws ? p_linear_forward_ws(&layer, xp, xd, m, y.data_ptr(), yd, wp, bytes, on.stream)
              : p_linear_forward(&layer, xp, xd, m, y.data_ptr(), yd, on.stream);
  });
  return rc == TTQ_OK ? THPVariable_Wrap(std::move(y)) : answer(rc);
}

// (x, gamma, eps, residual or None) -> (normed, new_residual or None)
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 4 || !p_rmsnorm) return answer(1);
  const at::Tensor *x = gpu_tensor(a[0]), *g = gpu_tensor(a[1]), *r = nullptr;
  if (!x || !g || x->dim() == 0 || g->device() != x->device() || g->scalar_type() != x->scalar_type()) return answer(1);
  if (a[3] != Py_None && (!(r = gpu_tensor(a[3])) || r->device() != x->device() || r->sizes() != x->sizes() ||
                          r->scalar_type() != x->scalar_type()))
    return answer(1);
  const double eps = PyFloat_AsDouble(a[2]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const int64_t width = x->size(-1);
  const int xd = dtype_code(x->scalar_type());
  if (xd < 0 || width <= 0 || g->numel() != width) return answer(1);
  const void *xp = x->data_ptr(), *rp = r ? r->data_ptr() : nullptr, *gp = g->data_ptr();
  const int64_t m = x->numel() / width;
  const c10::Device device = x->device();
  const Output out(*x, width, x->scalar_type());
  at::Tensor normed, sum;
  const int rc = released([&] {
    const OnDevice on(device);
    normed = out.make();
    if (r) sum = out.make();                     // also for no rows, where rp is null
    return p_rmsnorm(xp, rp, gp, (float)eps, xd, r ? sum.data_ptr() : nullptr, normed.data_ptr(), m, width, on.stream);
  });
  if (rc != TTQ_OK) return answer(rc);
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(normed)));
  if (r) {
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(sum)));
  } else {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(pair, 1, Py_None);
  }
  return pair;
}

// (x) -> silu(x[..., :h]) * x[..., h:]
PyObject* silu_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1 || !p_silu_and_mul) return answer(1);
  const at::Tensor* x = gpu_tensor(a[0]);
  if (!x || x->dim() == 0 || x->size(-1) <= 0 || x->size(-1) % 2) return answer(1);
  const int xd = dtype_code(x->scalar_type());
  if (xd < 0) return answer(1);
  const int64_t h = x->size(-1) / 2;
  const void* xp = x->data_ptr();
  const int64_t m = x->numel() / (2 * h);
  const c10::Device device = x->device();
  const Output out(*x, h, x->scalar_type());
  at::Tensor y;
  const int rc = released([&] {
    const OnDevice on(device);
    y = out.make();
    return p_silu_and_mul(xp, y.data_ptr(), xd, m, h, on.stream);
  });
  return rc == TTQ_OK ? THPVariable_Wrap(std::move(y)) : answer(rc);
}

// (qweight, x, n_ff, n_in, gemm): silu(x Wg^T) * (x Wu^T) of a packed Q4_K [Wg; Wu] in the type and leading
// dimensions of x, by the decode kernel or the GEMM
PyObject* q4_k_silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5 || !p_gemv_q4_k_silu_mul) return answer(1);
  const at::Tensor *q = gpu_tensor(a[0]), *x = gpu_tensor(a[1]);
  int64_t n_ff, n_in;
  if (!as_int64(a[2], n_ff) || !as_int64(a[3], n_in)) return nullptr;
  if (!q || !x || q->device() != x->device() || x->dim() == 0 || n_in <= 0 || n_in % 256 || n_ff <= 0 ||
      x->size(-1) != n_in || n_ff > ((int64_t)1 << 40) / n_in || (int64_t)q->nbytes() != 2 * n_ff * (n_in / 256) * 144)
    return answer(1);
  const bool gemm = a[4] == Py_True;
  const int xd = dtype_code(x->scalar_type());
  if (xd < 0 || (gemm && xd != TTQ_BF16)) return answer(1);
  const void *wp = q->data_ptr(), *xp = x->data_ptr();
  const int64_t m = x->numel() / n_in;
  const c10::Device device = x->device();
  const Output out(*x, n_ff, x->scalar_type());
  at::Tensor y;
  const int rc = released([&] {
    const OnDevice on(device);
    y = out.make();
    void* yp = y.data_ptr();
    return gemm ? p_gemm_q4_k_silu_mul(wp, static_cast<const uint16_t*>(xp), static_cast<uint16_t*>(yp), m, n_ff, n_in,
                                       on.stream)
                : p_gemv_q4_k_silu_mul(wp, xp, xd, yp, xd, m, n_ff, n_in, on.stream);
  });
  return rc == TTQ_OK ? THPVariable_Wrap(std::move(y)) : answer(rc);
}

// A C++ exception (an allocation that failed) becomes a Python one.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(self, a, n);
  END_HANDLE_TH_ERRORS
}

#define TTQ_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&guarded<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TTQ_METHOD(bind),         TTQ_METHOD(linear_forward), TTQ_METHOD(rmsnorm),
                         TTQ_METHOD(silu_and_mul), TTQ_METHOD(q4_k_silu_mul),  {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ttq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ttq_torch() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TTQ_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
