// Python calls of the C ABI with torch tensors as arguments (the module arraydiff_cuda_amd._binding).
//
// Every function declared in adh_capi.h that launches work on tensors is callable under its own name with its own
// arguments but the last: the stream is torch's current one.  A device pointer is a tensor (contiguous, on the GPU) or None, a
// table of device pointers a sequence of tensors, and a table of lengths the sequence of tensors whose lengths they are.  The
// conversions are chosen by the parameters' C types.
// A small launch costs what its caller spends on the host: with ctypes, an exchange of the halos of four 14x56 tiles and
// its backward took 18.0 us, of which the two kernels are 6; here the pair takes 6.7 us, and the fused softmax loss over
// 256x1000 11.5 us instead of 23.8.
#include <Python.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <exception>
#include <memory>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "adh_capi.h"

namespace {

// the calls' temporaries: host tables of pointers and lengths
struct Tables {
  std::array<std::vector<uint64_t>, 12> table;
  size_t used = 0;
  std::vector<uint64_t> &next() {
    auto &t = table.at(used++);
    t.clear();
    return t;
  }
};

// (the tensor's methods throw, for instance where it has no storage: call() turns that into a Python error)
const at::Tensor *gpu_tensor(PyObject *o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
    return nullptr;
  }
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.is_cuda() || !t.is_contiguous()) {
    PyErr_SetString(PyExc_ValueError, "tensors must be contiguous GPU tensors");
    return nullptr;
  }
  return &t;
}

bool address_of(PyObject *o, uint64_t *p) {
  const at::Tensor *t = gpu_tensor(o);
  if (!t) return false;
  *p = reinterpret_cast<uint64_t>(t->data_ptr());
  return true;
}

struct Release {
  void operator()(PyObject *o) const { Py_DECREF(o); }
};
using Reference = std::unique_ptr<PyObject, Release>;

template <typename T>
bool convert(PyObject *o, T *v, Tables &tables) {
  if constexpr (std::is_floating_point_v<T>) {
    *v = static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_integral_v<T>) {
    *v = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  } else {
    using P = std::remove_pointer_t<T>;
    constexpr bool lengths = std::is_same_v<std::remove_const_t<P>, uint64_t>;
    if constexpr (!std::is_pointer_v<P> && !lengths) {
      uint64_t p = 0;
      if (o != Py_None && !address_of(o, &p)) return false;
      *v = reinterpret_cast<T>(p);
    } else {
      if (o == Py_None) {
        *v = nullptr;
        return true;
      }
      const Reference seq(PySequence_Fast(o, "expected a sequence of tensors"));
      if (!seq) return false;
      std::vector<uint64_t> &table = tables.next();
      const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq.get());
      bool ok = true;
      for (Py_ssize_t i = 0; ok && i < n; ++i) {
        PyObject *item = PySequence_Fast_GET_ITEM(seq.get(), i);
        uint64_t p = 0;
        if (lengths) {
          const at::Tensor *t = gpu_tensor(item);
          ok = t != nullptr;
          if (ok) p = static_cast<uint64_t>(t->numel());
        } else {
          ok = address_of(item, &p);
        }
        table.push_back(p);
      }
      if (!ok) return false;
      *v = reinterpret_cast<T>(table.data());
    }
  }
  return !PyErr_Occurred();
}

PyObject *current_device = nullptr, *current_stream = nullptr;  // torch's, given to load()

// the raw handle of torch's current stream on the current device
bool stream_of_torch(void **stream) {
  PyObject *device = PyObject_CallNoArgs(current_device);
  if (!device) return false;
  PyObject *handle = PyObject_CallOneArg(current_stream, device);
  Py_DECREF(device);
  if (!handle) return false;
  *stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return !PyErr_Occurred();
}

template <typename... A, size_t... I>
PyObject *call(int (*fn)(A...), PyObject *const *args, std::index_sequence<I...>) {
  static thread_local Tables tables;
  tables.used = 0;
  std::tuple<A...> values;
  try {
    if (!(convert(args[I], &std::get<I>(values), tables) && ...)) return nullptr;
  } catch (const c10::Error &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  if (!stream_of_torch(&std::get<sizeof...(I)>(values))) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = std::apply(fn, values);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// The functions are those of the library that load() opened, not of one linked to this module.
template <typename F>
struct Entry;
template <typename... A>
struct Entry<int (*)(A...)> {
  template <int N>
  static inline int (*address)(A...) = nullptr;
  template <int N>
  static PyObject *method(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (!address<N>) {
      PyErr_SetString(PyExc_RuntimeError, "the library is not loaded");
      return nullptr;
    }
    constexpr size_t wanted = sizeof...(A) - 1;
    if (nargs != static_cast<Py_ssize_t>(wanted)) {
      PyErr_Format(PyExc_TypeError, "%zd arguments given, %zd wanted", nargs, static_cast<Py_ssize_t>(wanted));
      return nullptr;
    }
    return call(address<N>, args, std::make_index_sequence<wanted>{});
  }
};

#define ADH_ENTRIES(X)                                                                                                        \
  X(adh_fill_f32) X(adh_add_f32) X(adh_halo_exchange_nchw) X(adh_halo_reduce_nchw) X(adh_halo_exchange_nchw_rank)             \
  X(adh_halo_reduce_nchw_rank) X(adh_halo_pad_nchw) X(adh_halo_pad_add_nchw) X(adh_halo_unpad_nchw) X(adh_halo_unpad_add_nchw) \
  X(adh_halo_repad_nchw) X(adh_slice_copy_nchw) X(adh_slice_add_nchw) X(adh_tiles_pack_nchw) X(adh_tiles_unpack_nchw)          \
  X(adh_conv3x3_slab_fwd_tiles) X(adh_conv3x3_slab_fwd_tiles_unexchanged) X(adh_conv3x3_slab_bwd_data_tiles)                   \
  X(adh_conv3x3_slab_bwd_data_tiles_reduced) X(adh_conv3x3_slab_bwd_filter_tiles)                                              \
  X(adh_conv3x3_slab_bwd_filter_tiles_unexchanged) X(adh_conv3x3_unpadded_fwd_tiles)                                           \
  X(adh_conv3x3_unpadded_fwd_residual_tiles) X(adh_conv3x3_unpadded_bwd_data_tiles) X(adh_conv3x3_unpadded_bwd_filter_tiles)   \
  X(adh_conv_bias_add_tiles) X(adh_conv_bwd_bias_tiles) X(adh_conv2d_slab_fwd_tiles) X(adh_conv2d_slab_fwd_bias_tiles)         \
  X(adh_conv2d_slab_bwd_data_tiles) X(adh_conv2d_slab_bwd_filter_tiles) X(adh_conv2d_unpadded_fwd_tiles)                       \
  X(adh_conv2d_unpadded_bwd_data_tiles) X(adh_conv2d_unpadded_bwd_filter_tiles) X(adh_batchnorm2d_fwd_tiles)                   \
  X(adh_batchnorm2d_bwd_tiles) X(adh_relu_fwd) X(adh_relu_bwd) X(adh_sum_fwd) X(adh_pool2d_slab_fwd_tiles)                     \
  X(adh_pool2d_slab_bwd_tiles) X(adh_pool2d_unpadded_fwd_tiles) X(adh_pool2d_unpadded_bwd_tiles) X(adh_softmax_fwd)            \
  X(adh_softmax_nll_loss_fwd) X(adh_softmax_nll_loss_bwd) X(adh_softmax_xent_fwd) X(adh_softmax_nll_loss_bwd_scaled)           \
  X(adh_softmax_xent_fwd_bwd) X(adh_scale_add_f32) X(adh_add_online_f32) X(adh_stat_step_f32) X(adh_flat_store_f32)            \
  X(adh_flat_load_f32) X(adh_sgd_step_f32)

enum EntryNumber {
#define ADH_NUMBER(name) k_##name,
  ADH_ENTRIES(ADH_NUMBER)
#undef ADH_NUMBER
};

PyObject *load(PyObject *, PyObject *args) {
  const char *path = nullptr;
  PyObject *device = nullptr, *stream = nullptr;
  if (!PyArg_ParseTuple(args, "sOO", &path, &device, &stream)) return nullptr;
  void *lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
#define ADH_LOAD(name)                                                                                        \
  if (!(Entry<decltype(&name)>::address<k_##name> = reinterpret_cast<decltype(&name)>(dlsym(lib, #name)))) { \
    PyErr_SetString(PyExc_RuntimeError, #name " is not exported");                                            \
    return nullptr;                                                                                           \
  }
  ADH_ENTRIES(ADH_LOAD)
#undef ADH_LOAD
  Py_INCREF(device);
  Py_INCREF(stream);
  current_device = device;
  current_stream = stream;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"load", load, METH_VARARGS, "load(path, device, stream): take the functions from the library at `path`; device() and\n"
                                  "stream(device) are torch's current device and the raw handle of its current stream"},
#define ADH_METHOD(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<decltype(&name)>::method<k_##name>)), METH_FASTCALL, nullptr},
    ADH_ENTRIES(ADH_METHOD)
#undef ADH_METHOD
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
