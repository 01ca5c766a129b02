// The two co-location kernels' calls from Python without Python in between.
//
// kernels.triad and kernels.gemm_bf16_nt hand their arguments here first.  For ordinary
// tensors, with nothing about that has to see every operation, the checks, the output's
// allocation, the current stream and the call of the C entry point take less than 1 us here;
// attribute by attribute and through ctypes 2.5 to 3.5, as long as the smaller kernels run
// (us a call: triad of 1,000,003 elements 5.3 so, 3.6 here; gemm 256 x 512 x 256 with its
// output allocated 7.2, 4.5).  Every other call, and every refusal, returns None and is
// made, or raised, by the Python code, so nothing is decided in two places but what is taken
// here.  Only the runtime's error is raised here: it is found behind the launch, which must
// not be made again.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "orion_kernels.h"

namespace {

decltype(&orion_triad_f32) triad_entry = nullptr;
decltype(&orion_gemm_bf16_nt) gemm_entry = nullptr;

// Modes, transforms and tracers that see operations: for the Python code.
bool plain() {
  using c10::impl::tls_is_dispatch_key_included;
  return !at::impl::torch_function_mode_enabled() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}

// A tensor or a parameter (no subclass) on a GPU, contiguous, without names.
const at::Tensor* tensor_of(PyObject* o) {
  if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || !t.is_contiguous() ||
      t.has_names())
    return nullptr;
  return &t;
}

// The stream that was named, or the current device's current one.
bool stream_of(PyObject* o, void** stream) {
  if (o == Py_None) {
    *stream = c10::hip::getCurrentHIPStream().stream();
    return true;
  }
  PyObject* handle = PyObject_GetAttrString(o, "cuda_stream");
  if (handle == nullptr) return false;
  const bool is_int = PyLong_CheckExact(handle);
  if (is_int) *stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return is_int && !PyErr_Occurred();
}

PyObject* none() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// What an entry point answered that has not taken the call: argument, shape and alignment are
// checked before anything is launched, and the Python code is refused in the same way.
PyObject* refused(const char* entry, int code) {
  if (code < ORION_ERR_LAUNCH) return none();
  PyObject* kernels = PyImport_ImportModule("orion_amd.kernels");
  PyObject* error = kernels ? PyObject_GetAttrString(kernels, "KernelError") : nullptr;
  PyObject* raised = error ? PyObject_CallFunction(error, "si", entry, code) : nullptr;
  if (raised) PyErr_SetObject(error, raised);
  Py_XDECREF(raised);
  Py_XDECREF(error);
  Py_XDECREF(kernels);
  return nullptr;
}

// entries(triad, gemm): addresses of the C entry points, 0 for none.
PyObject* entries(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 2) {
    PyErr_SetString(PyExc_TypeError, "entries(triad, gemm)");
    return nullptr;
  }
  void* triad = PyLong_AsVoidPtr(args[0]);
  void* gemm = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  triad_entry = reinterpret_cast<decltype(triad_entry)>(triad);
  gemm_entry = reinterpret_cast<decltype(gemm_entry)>(gemm);
  Py_RETURN_NONE;
}

// triad(a, b, c, s, grid_blocks, stream): a, or None
PyObject* triad(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 6 || triad_entry == nullptr) Py_RETURN_NONE;
  try {
    const at::Tensor *a = tensor_of(args[0]), *b = tensor_of(args[1]), *c = tensor_of(args[2]);
    if (!a || !b || !c || a->scalar_type() != at::kFloat || b->scalar_type() != at::kFloat ||
        c->scalar_type() != at::kFloat || a->numel() != b->numel() || a->numel() != c->numel() ||
        !plain())
      return none();
    if (!(PyFloat_CheckExact(args[3]) || PyLong_CheckExact(args[3])) ||
        !PyLong_CheckExact(args[4]))
      return none();
    const double s = PyFloat_AsDouble(args[3]);
    const long grid_blocks = PyLong_AsLong(args[4]);
    void* stream;
    if (PyErr_Occurred() || grid_blocks != (int)grid_blocks || !stream_of(args[5], &stream))
      return none();
    float* pa = static_cast<float*>(a->data_ptr());
    const float* pb = static_cast<const float*>(b->data_ptr());
    const float* pc = static_cast<const float*>(c->data_ptr());
    const size_t n = (size_t)a->numel();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = triad_entry(pa, pb, pc, (float)s, n, (int)grid_blocks, stream);
    Py_END_ALLOW_THREADS
    if (rc != ORION_OK) return refused("orion_triad_f32", rc);
  } catch (...) {
    return none();
  }
  Py_INCREF(args[0]);
  return args[0];
}

// gemm(a, b, out, out_dtype, stream): the output, or None
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 5 || gemm_entry == nullptr) Py_RETURN_NONE;
  try {
    const at::Tensor *a = tensor_of(args[0]), *b = tensor_of(args[1]);
    if (!a || !b || a->scalar_type() != at::kBFloat16 || b->scalar_type() != at::kBFloat16 ||
        a->dim() != 2 || b->dim() != 2 || a->size(1) != b->size(1) || !plain())
      return none();
    const int64_t m = a->size(0), n = b->size(0), k = a->size(1);
    void* stream;
    if (m != (int)m || n != (int)n || k != (int)k || !stream_of(args[4], &stream)) return none();
    at::Tensor made;
    const at::Tensor* out = &made;
    if (args[2] == Py_None) {
      if (!THPDtype_Check(args[3])) return none();
      const at::ScalarType dtype = reinterpret_cast<THPDtype*>(args[3])->scalar_type;
      if (dtype != at::kBFloat16 && dtype != at::kFloat) return none();
      made = at::empty({m, n}, at::TensorOptions().dtype(dtype).device(a->device()));
    } else {
      out = tensor_of(args[2]);
      if (!out || out->dim() != 2 || out->size(0) != m || out->size(1) != n ||
          (out->scalar_type() != at::kBFloat16 && out->scalar_type() != at::kFloat))
        return none();
    }
    const void *pa = a->data_ptr(), *pb = b->data_ptr();
    void* po = out->data_ptr();
    const int wide = out->scalar_type() == at::kFloat;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = gemm_entry(pa, pb, po, (int)m, (int)n, (int)k, wide, stream);
    Py_END_ALLOW_THREADS
    if (rc != ORION_OK) return refused("orion_gemm_bf16_nt", rc);
    if (made.defined()) return THPVariable_Wrap(std::move(made));
  } catch (...) {
    return none();
  }
  Py_INCREF(args[2]);
  return args[2];
}

PyMethodDef methods[] = {
    {"entries", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(entries)), METH_FASTCALL,
     nullptr},
    {"triad", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(triad)), METH_FASTCALL,
     nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gemm)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kernel_calls", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_kernel_calls() { return PyModule_Create(&module); }
