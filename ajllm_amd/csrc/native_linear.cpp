// A quantized layer's forward for the tensors it is nearly always called with, without the interpreter: one call of libajq.so.
//
// linear(inputs, wq, meta, int4, in_features, out_features, out_dtype or None) -> outputs, or None where anything is out of the
// ordinary (another dtype or layout, a subclass, a mode or a transform that wants to see the operators, another device, an error
// status): the caller then goes through its general path, which converts, refuses or reports.  What bounds a decode step's call is
// the host: 8.8 us through ctypes, where the kernel takes 3.6.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/ajq.h"

namespace {

constexpr int kMaxGemvRows = 16;

// entry points of the library that the package has loaded
decltype(&ajq_w4a16_gemv) w4_gemv;
decltype(&ajq_w8a16_gemv) w8_gemv;
decltype(&ajq_w4a16_matmul) w4_matmul;
decltype(&ajq_w8a16_matmul) w8_matmul;
decltype(&ajq_matmul_scratch_bytes) scratch_bytes;

// a tensor (or parameter) of the plain kind on the current device, or null
const at::Tensor* plain(PyObject* object) {
  if (!THPVariable_CheckExact(object)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(object);
  const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                     c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                     c10::DispatchKey::ZeroTensor, c10::DispatchKey::Named});
  return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(special) ? &t : nullptr;
}

// other threads run while the allocator and the runtime do (a full queue makes a launch wait)
struct WithoutInterpreter {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 7 || !scratch_bytes) {
    PyErr_SetString(PyExc_TypeError, count != 7 ? "linear takes seven arguments" : "linear is not bound to the library");
    return nullptr;
  }
  const at::Tensor *x = plain(args[0]), *wq = x ? plain(args[1]) : nullptr, *meta = wq ? plain(args[2]) : nullptr;
  if (!meta || c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const bool w4 = args[3] == Py_True;
  const int64_t k = PyLong_AsLongLong(args[4]), columns = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) return nullptr;
  at::ScalarType dtype = x->scalar_type();
  if (args[6] != Py_None) {
    if (!THPDtype_Check(args[6])) Py_RETURN_NONE;
    dtype = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
  }
  if (x->scalar_type() != at::kBFloat16 || (dtype != at::kBFloat16 && dtype != at::kFloat) || x->dim() < 1 || wq->dim() < 2 || k < 1 ||
      x->size(-1) != k || !x->is_contiguous() || x->numel() == 0)
    Py_RETURN_NONE;
  const int64_t tiles = wq->size(0), rows = x->numel() / k;
  const auto device = x->device().index();
  if (wq->size(1) * (w4 ? 128 : 64) != k || columns < 1 || columns > tiles * 16 || (!w4 && meta->numel() != tiles * 16) ||
      rows > INT32_MAX || k > INT32_MAX || tiles > INT32_MAX / 16 || device != c10::hip::current_device())
    Py_RETURN_NONE;
  const at::Tensor input = *x, packed = *wq, scales = *meta;  // held while the interpreter runs other threads
  at::Tensor y;
  int status;
  {
    const WithoutInterpreter released;
    at::DimVector sizes(input.sizes().begin(), input.sizes().end());
    sizes.back() = tiles * 16;
    y = at::empty(sizes, input.options().dtype(dtype));
    void* stream = c10::hip::getCurrentHIPStream(device).stream();
    const int m = (int)rows, n = (int)tiles * 16, depth = (int)k, out = dtype == at::kFloat ? AJQ_OUT_F32 : AJQ_OUT_BF16;
    const auto* in = static_cast<const uint16_t*>(input.const_data_ptr());
    const auto* weights = static_cast<const uint32_t*>(packed.const_data_ptr());
    const auto* groups = static_cast<const uint32_t*>(scales.const_data_ptr());
    const auto* channels = static_cast<const uint16_t*>(scales.const_data_ptr());
    void* to = y.mutable_data_ptr();
    if (m <= kMaxGemvRows) {
      status = w4 ? w4_gemv(in, m, depth, weights, groups, n, to, out, stream) : w8_gemv(in, m, depth, weights, channels, n, to, out, stream);
    } else {
      const size_t bytes = scratch_bytes(m, n, depth, w4);
      at::Tensor room;
      if (bytes) room = at::empty({(int64_t)bytes}, input.options().dtype(at::kByte));
      void* scratch = bytes ? room.mutable_data_ptr() : nullptr;
      status = w4 ? w4_matmul(in, m, depth, weights, groups, n, to, out, scratch, bytes, stream)
                  : w8_matmul(in, m, depth, weights, channels, n, to, out, scratch, bytes, stream);
    }
  }
  if (status != AJQ_OK) Py_RETURN_NONE;
  if (columns != tiles * 16) y = y.narrow(-1, 0, columns);  // a ragged number of rows: the padded columns stay behind a view
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// bind(w4_gemv, w8_gemv, w4_matmul, w8_matmul, scratch_bytes): their addresses in the loaded library
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 5) {
    PyErr_SetString(PyExc_TypeError, "bind takes five addresses");
    return nullptr;
  }
  void* at[5];
  for (int i = 0; i < 5; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (!at[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  w4_gemv = reinterpret_cast<decltype(w4_gemv)>(at[0]);
  w8_gemv = reinterpret_cast<decltype(w8_gemv)>(at[1]);
  w4_matmul = reinterpret_cast<decltype(w4_matmul)>(at[2]);
  w8_matmul = reinterpret_cast<decltype(w8_matmul)>(at[3]);
  scratch_bytes = reinterpret_cast<decltype(scratch_bytes)>(at[4]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&linear)), METH_FASTCALL, nullptr},
                         {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&bind)), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
