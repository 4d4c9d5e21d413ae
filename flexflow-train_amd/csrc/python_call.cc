// The way from Python to the entry points of ffk.h: one METH_FASTCALL function per entry point,
// generated from its C prototype.  Tensors are passed as they are (their device pointer is taken
// here), descriptors as the ctypes structures they are, and the stream, which every entry point
// takes first, is the current one and not passed at all.  A non-zero status raises FFKError.
//
// Why not ctypes: a call of ten arguments is 0.65 us there, a tensor's pointer with its two checks
// 0.2 us and torch.cuda.current_stream() 2.9 us, next to 2.6 us for the kernel launch itself: 8.0 us
// for a Linear forward, of which this leaves 3.8.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>
#include "../../include/ffk.h"

namespace {

PyObject *g_error = nullptr;       // FFKError
PyObject *g_get_device = nullptr;  // torch._C._cuda_getDevice
PyObject *g_get_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

// One argument: load() takes it or sets a Python error.  What it holds on to (a buffer) goes with it.
template <typename T, bool HOST_INTS, typename = void>
struct Arg;

// an int (or what serves as an index), its low bits, as ctypes takes them
template <typename T, bool HOST_INTS>
struct Arg<T, HOST_INTS, std::enable_if_t<std::is_integral_v<T>>> {
  T i;
  bool load(PyObject *o) {
    PyObject *const index = PyNumber_Index(o);
    if (index == nullptr) return false;
    i = (T)PyLong_AsUnsignedLongLongMask(index);
    Py_DECREF(index);
    return true;
  }
  T value() const { return i; }
};
template <bool HOST_INTS>
struct Arg<float, HOST_INTS> {
  float f;
  bool load(PyObject *o) {
    f = (float)PyFloat_AsDouble(o);
    return !PyErr_Occurred();
  }
  float value() const { return f; }
};
// Pointers to memory of the device (data of any type): None or a tensor, nothing else.  An address or
// the buffer of an array would reach a kernel as it is, which faults on the host's memory.
struct DevicePointer {
  void *address = nullptr;
  bool load(PyObject *o) {
    if (o == Py_None) return true;
    if (!THPVariable_Check(o)) {
      PyErr_Format(PyExc_TypeError, "tensor or None expected, %.200s given", Py_TYPE(o)->tp_name);
      return false;
    }
    // what torch has to say against the tensor (one under torch.vmap has no address) comes as a C++
    // exception, which must not reach the interpreter's frames
    try {
      at::Tensor const &t = THPVariable_Unpack(o);
      if (!t.is_cuda() || !t.is_contiguous()) {
        PyErr_SetString(PyExc_AssertionError, "device-resident contiguous tensor required");
        return false;
      }
      address = t.data_ptr();
      return true;
    } catch (std::exception const &) {
      torch::translate_exception_to_python(std::current_exception());
      return false;
    }
  }
};
// Pointers to memory of the host (descriptors; arrays of sizes and of pointers): a ctypes structure or
// array.  A structure has to be as long as the descriptor, an array's elements as its elements.
struct HostPointer {
  Py_buffer buffer = {};
  bool load(PyObject *o, size_t size, bool array, bool writable) {
    if (PyObject_GetBuffer(o, &buffer, writable ? PyBUF_WRITABLE : PyBUF_SIMPLE) != 0) return false;
    if ((size_t)(array ? buffer.itemsize : buffer.len) == size) return true;
    PyErr_Format(PyExc_TypeError, "%.200s is not what this argument points to (%zu bytes%s)", Py_TYPE(o)->tp_name, size,
                 array ? " an element" : "");
    return false;
  }
  ~HostPointer() {
    if (buffer.obj != nullptr) PyBuffer_Release(&buffer);
  }
};
// What lies on the host: structures, 64-bit sizes, pointers, the flop count of a probe, and an int
// array only where the entry point says so (ints are a permutation in Transpose, labels on the device
// elsewhere).
template <typename T, bool HOST_INTS>
constexpr bool kOnHost = std::is_pointer_v<T> || std::is_class_v<T> || std::is_same_v<std::remove_cv_t<T>, int64_t> ||
                         std::is_same_v<T, double> || (HOST_INTS && std::is_same_v<std::remove_cv_t<T>, int>);
template <typename T, bool HOST_INTS>
struct Arg<T *, HOST_INTS, std::enable_if_t<!kOnHost<T, HOST_INTS>>> {
  DevicePointer p;
  bool load(PyObject *o) { return p.load(o); }
  T *value() const { return (T *)p.address; }
};
template <typename T, bool HOST_INTS>
struct Arg<T *, HOST_INTS, std::enable_if_t<kOnHost<T, HOST_INTS>>> {
  HostPointer p;
  bool load(PyObject *o) { return p.load(o, sizeof(T), !std::is_class_v<T>, !std::is_const_v<T>); }
  T *value() const { return (T *)p.buffer.buf; }
};

bool current_stream(ffk_stream_t &stream) {
  PyObject *dev = PyObject_CallNoArgs(g_get_device);
  if (dev == nullptr) return false;
  PyObject *s = PyObject_CallOneArg(g_get_stream, dev);
  Py_DECREF(dev);
  if (s == nullptr) return false;
  stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  return !PyErr_Occurred();
}

template <auto FN, bool HOST_INTS = false>
struct Call;
// an entry point that launches: (stream, ...) -> status
template <typename... A, int (*FN)(ffk_stream_t, A...), bool HOST_INTS>
struct Call<FN, HOST_INTS> {
  template <size_t... I>
  static PyObject *run(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<Arg<A, HOST_INTS>...> a;
    ffk_stream_t stream = nullptr;
    if (!((std::get<I>(a).load(args[I]) && ...) && current_stream(stream))) return nullptr;
    int rc;
    // a launch can block when the queue is full
    Py_BEGIN_ALLOW_THREADS
    rc = FN(stream, std::get<I>(a).value()...);
    Py_END_ALLOW_THREADS
    if (rc != FFK_OK) {
      PyErr_Format(g_error, "ffk error %d: %s", rc, ffk_last_error());
      return nullptr;
    }
    Py_RETURN_NONE;
  }
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", (int)sizeof...(A), n);
    return run(args, std::index_sequence_for<A...>{});
  }
};
// a size query: (...) -> bytes
template <typename... A, size_t (*FN)(A...), bool HOST_INTS>
struct Call<FN, HOST_INTS> {
  template <size_t... I>
  static PyObject *run(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<Arg<A, HOST_INTS>...> a;
    if (!(std::get<I>(a).load(args[I]) && ...)) return nullptr;
    return PyLong_FromSize_t(FN(std::get<I>(a).value()...));
  }
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", (int)sizeof...(A), n);
    return run(args, std::index_sequence_for<A...>{});
  }
};

PyObject *set_error(PyObject *, PyObject *cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_error, cls);
  Py_RETURN_NONE;
}

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))Call<name>::call, METH_FASTCALL, nullptr}
#define ENTRY_HOST_INTS(name) {#name, (PyCFunction)(void (*)(void))Call<name, true>::call, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"set_error", set_error, METH_O, "The exception class a non-zero status raises."},
    ENTRY(ffk_linear_forward), ENTRY(ffk_linear_backward), ENTRY(ffk_linear_backward_workspace_bytes),
    ENTRY(ffk_linear_l2_regularizer_grad), ENTRY(ffk_probe_mfma_bf16), ENTRY(ffk_gemm), ENTRY(ffk_element_unary_forward),
    ENTRY(ffk_element_unary_backward), ENTRY(ffk_element_binary_forward), ENTRY(ffk_element_binary_backward),
    ENTRY(ffk_element_binary_backward_broadcast), ENTRY(ffk_layer_norm_forward), ENTRY(ffk_layer_norm_backward),
    ENTRY(ffk_layer_norm_backward_workspace_bytes), ENTRY(ffk_layer_norm_backward_static),
    ENTRY(ffk_layer_norm_backward_residual), ENTRY(ffk_dropout_add_layer_norm_forward), ENTRY(ffk_softmax_forward),
    ENTRY(ffk_softmax_backward), ENTRY(ffk_softmax_backward_copy), ENTRY(ffk_dropout_forward),
    ENTRY(ffk_dropout_backward), ENTRY(ffk_dropout_mask), ENTRY(ffk_dropout_add_forward), ENTRY(ffk_gelu_dropout_forward),
    ENTRY(ffk_dropout_gelu_backward), ENTRY(ffk_dropout_backward_bias_grad),
    ENTRY(ffk_dropout_backward_bias_grad_workspace_bytes), ENTRY(ffk_linear_gelu_dropout_forward),
    ENTRY(ffk_linear_dropout_add_forward), ENTRY(ffk_linear_backward_dropout_gelu),
    ENTRY(ffk_linear_backward_dropout_gelu_bias_grad), ENTRY(ffk_embedding_forward), ENTRY(ffk_embedding_backward),
    ENTRY(ffk_embedding_backward_workspace_bytes), ENTRY(ffk_embedding_backward_typed), ENTRY(ffk_attention_forward),
    ENTRY(ffk_attention_backward), ENTRY(ffk_mha_reserve_bytes), ENTRY(ffk_mha_forward), ENTRY(ffk_mha_backward),
    ENTRY(ffk_mha_backward_workspace_bytes), ENTRY(ffk_mha_backward_with_workspace),
    ENTRY(ffk_encoder_layer_workspace_bytes), ENTRY(ffk_encoder_layer_forward), ENTRY(ffk_encoder_layer_backward),
    ENTRY(ffk_sgd_update), ENTRY(ffk_adam_update), ENTRY(ffk_sparse_categorical_crossentropy_loss_backward),
    ENTRY(ffk_categorical_crossentropy_loss_backward), ENTRY(ffk_mean_squared_error_avg_loss_backward),
    ENTRY(ffk_identity_loss_backward), ENTRY(ffk_cast_forward), ENTRY(ffk_cast_backward), ENTRY(ffk_concat_forward),
    ENTRY(ffk_concat_backward), ENTRY(ffk_split_forward), ENTRY(ffk_split_backward), ENTRY_HOST_INTS(ffk_transpose_forward),
    ENTRY_HOST_INTS(ffk_transpose_backward), ENTRY(ffk_gather_forward), ENTRY(ffk_gather_backward),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ffk_call", "The entry points of ffk.h.", -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ffk_call() {
  PyObject *torch_c = PyImport_ImportModule("torch._C");
  if (torch_c == nullptr) return nullptr;
  g_get_device = PyObject_GetAttrString(torch_c, "_cuda_getDevice");
  g_get_stream = g_get_device != nullptr ? PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream") : nullptr;
  Py_DECREF(torch_c);
  if (g_get_stream == nullptr) return nullptr;
  g_error = PyExc_RuntimeError;
  Py_INCREF(g_error);
  return PyModule_Create(&module_def);
}
