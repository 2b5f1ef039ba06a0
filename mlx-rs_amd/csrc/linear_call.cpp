// The call around a quantized linear layer (mlx-rs/src/nn/quantized.rs:363-386) on torch tensors without the interpreter: the same
// checks, result, workspace and stream as ops.quantized_linear's own lines, which stay the general path.  One token's layer is 5 us of
// kernel; its call took 10 us in Python (checks 3, two allocations 2, the foreign call's conversions 3) and takes the kernel's time with this.
//
// quantized_linear(x, w, scales, biases, linear_bias, transpose, group_size, bits) returns the result, None for whatever is not a
// plain device tensor of the expected type, shape, layout and alignment (the caller then goes the general way, which takes it or words
// the refusal), or the library's status where that is not zero.  Nothing is kept between calls.  The interpreter is let go around the
// allocations and the launch, any of which may wait (for memory, for room in a queue, for a kernel to load).
#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/api/include/torch/version.h>

#include "../../include/mi_moe.h"

namespace {

decltype(&mi_moe_quantized_linear_typed) g_linear;
decltype(&mi_moe_quantized_matmul_typed) g_matmul;
decltype(&mi_moe_quantized_matmul_workspace_size) g_workspace;

// a tensor itself (no subclass), dense, on a GPU, contiguous, seen through no transform (vmap, functionalisation, a Python key)
const at::Tensor *plain(PyObject *o, at::ScalarType type) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || t.scalar_type() != type || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || !t.is_contiguous()) return nullptr;
  constexpr c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched,
                                       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return t.key_set().has_any(other) ? nullptr : &t;
}

PyObject *quantized_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "quantized_linear: eight arguments");
    return nullptr;
  }
  try {
    if (!THPVariable_CheckExact(args[0]) || !PyLong_Check(args[6]) || !PyLong_Check(args[7])) Py_RETURN_NONE;
    const at::ScalarType type = THPVariable_Unpack(args[0]).scalar_type();
    const int dt = type == at::kBFloat16 ? MI_MOE_DTYPE_BF16 : type == at::kHalf ? MI_MOE_DTYPE_F16 : type == at::kFloat ? MI_MOE_DTYPE_F32 : -1;
    const int transpose = PyObject_IsTrue(args[5]);
    const long group = PyLong_AsLong(args[6]), bits = PyLong_AsLong(args[7]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (dt < 0 || transpose < 0 || (group != 32 && group != 64 && group != 128) || (bits != 2 && bits != 4 && bits != 8)) Py_RETURN_NONE;
    const at::Tensor *const x = plain(args[0], type), *const w = plain(args[1], at::kInt), *const s = plain(args[2], type), *const b = plain(args[3], type);
    if (!x || !w || !s || !b || x->dim() < 1 || w->dim() != 2 || s->dim() != 2 || b->dim() != 2) Py_RETURN_NONE;
    const int64_t K = x->size(-1), per = 32 / bits;
    const int64_t N = transpose ? w->size(0) : w->size(1) * per, kw = transpose ? w->size(1) * per : w->size(0);
    const int64_t rows = transpose ? N : K, q_axis = transpose ? K : N;
    if (kw != K || x->numel() == 0 || N == 0 || q_axis % group || K > INT32_MAX || N > INT32_MAX) Py_RETURN_NONE;
    for (const at::Tensor *t : {s, b})
      if (t->size(0) != rows || t->size(1) != q_axis / group) Py_RETURN_NONE;
    const at::Tensor *lb = nullptr;
    if (args[4] != Py_None) {
      lb = plain(args[4], type);
      if (!lb || !transpose || lb->numel() != N) Py_RETURN_NONE;
    }
    for (const at::Tensor *t : {x, w, s, b})
      if (reinterpret_cast<uintptr_t>(t->const_data_ptr()) & 15u) Py_RETURN_NONE;
    const int64_t M = x->numel() / K;
    if (M > (int64_t)1 << 30) Py_RETURN_NONE;
    size_t need = 0;
    if (g_workspace(M, (int32_t)K, (int32_t)bits, &need)) Py_RETURN_NONE;
    at::DimVector shape(x->sizes().begin(), x->sizes().end());
    shape.back() = N;
    // (the operands' own references: another thread may drop the caller's while the interpreter is let go)
    const at::Tensor xk = *x, wk = *w, sk = *s, bk = *b, lk = lb ? *lb : at::Tensor();
    at::Tensor y;
    int status = 0;
    {
      pybind11::gil_scoped_release let_go;
      const at::TensorOptions on = at::TensorOptions().device(xk.device());
      y = at::empty(shape, on.dtype(type));
      at::Tensor ws = at::empty({(int64_t)need + 256}, on.dtype(at::kByte));
      void *const st = c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream();
      status = lk.defined()
                   ? g_linear(xk.const_data_ptr(), static_cast<const uint32_t *>(wk.const_data_ptr()), sk.const_data_ptr(), bk.const_data_ptr(), lk.const_data_ptr(),
                              M, (int32_t)N, (int32_t)K, (int32_t)group, (int32_t)bits, dt, y.data_ptr(), ws.data_ptr(), need + 256, st)
                   : g_matmul(xk.const_data_ptr(), static_cast<const uint32_t *>(wk.const_data_ptr()), sk.const_data_ptr(), bk.const_data_ptr(), M, (int32_t)N,
                              (int32_t)K, transpose, (int32_t)group, (int32_t)bits, dt, y.data_ptr(), ws.data_ptr(), need + 256, st);
    }
    if (status) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(y));
  } catch (python_error &e) {  // what a mode written in Python raised from an allocation: the caller's
    e.restore();
  } catch (pybind11::error_already_set &e) {
    e.restore();
  } catch (const std::exception &) {  // (out of memory: the general path meets it again and words it)
  }
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// bind(addresses of the library's quantized_linear_typed, quantized_matmul_typed and quantized_matmul_workspace_size)
PyObject *bind(PyObject *, PyObject *args) {
  unsigned long long l = 0, m = 0, ws = 0;
  if (!PyArg_ParseTuple(args, "KKK", &l, &m, &ws)) return nullptr;
  g_linear = reinterpret_cast<decltype(g_linear)>(l);
  g_matmul = reinterpret_cast<decltype(g_matmul)>(m);
  g_workspace = reinterpret_cast<decltype(g_workspace)>(ws);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"quantized_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(quantized_linear)), METH_FASTCALL, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_linear_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__linear_call() {
  PyObject *const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_with", TORCH_VERSION)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
