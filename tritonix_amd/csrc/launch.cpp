// Repeated calls of the Python entry points, from a kept argument struct to the launch, without the interpreter.
//
// A call of a size met before has nothing to decide: allocate the result, fill three pointers into a tnx_gemm_args, launch.  In
// Python that took 5.5 us around a launch of 3.5 (the tuple of sizes, strides and types that finds the struct, torch.empty,
// ctypes), which is what a small product waits for: its kernel takes 4 to 5.  Here it takes 1.2: 1024 x 768 x 512 through
// tritonix.matmul 8.97 -> 5.84 us, a small gated product 7.7 -> 4.9, conv2d 8.6 -> 5.5 and, in two launches, 12.4 -> 9.0.
//
// The entry points are looked up in the library that tritonix_amd/_C.py has loaded (their addresses are handed to bind()), the
// structs are the header's.  Every function answers None where the ordinary path has to take the call: a size not kept, a hook,
// a replaced config, a tensor on another than the current device, a subclass of torch.Tensor (but Parameter), an allocation that
// failed, a conv2d status other than TNX_OK.  That path then raises what is to be raised.  A product's status is raised here: its
// launch may have left counters set in the workspace, which is not to be launched over again.  All state is guarded by the
// interpreter lock, which no entry of the tables is read without.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/headeronly/version.h>

#include <cstring>
#include <unordered_map>

#include "../../include/tritonix_hip.h"

namespace {

int (*fn_gemm)(const tnx_gemm_args*) = nullptr;
int (*fn_gemm_f32)(const tnx_gemm_args*, void*, size_t) = nullptr;
int (*fn_conv)(const tnx_conv2d_args*) = nullptr;
PyObject* fn_workspace = nullptr;       // (device index, stream, bytes, atomic) -> tensor
PyObject* fn_failed = nullptr;          // (device index, stream, status, argument struct): raises

// What a launch depends on but its pointers.  Compared and hashed as bytes: zero-filled before it is written.
struct Key {
  int64_t tag;
  int64_t sizes[8], strides[8];
  int64_t options[6];
  int32_t type_a, type_b, type_c, device, aligned, count_c;
  bool operator==(const Key& o) const { return std::memcmp(this, &o, sizeof(Key)) == 0; }
};
struct Hash {
  size_t operator()(const Key& k) const {
    const unsigned char* p = (const unsigned char*)&k;
    uint64_t h = 0x9e3779b97f4a7c15ull;
    for (size_t i = 0; i < sizeof(Key); i += 8) {
      uint64_t w;
      std::memcpy(&w, p + i, 8);
      h = (h ^ w) * 0xff51afd7ed558ccdull;
      h ^= h >> 32;
    }
    return (size_t)h;
  }
};
static_assert(sizeof(Key) % 8 == 0, "hashed word by word");

struct Object {                          // a Python reference that goes with its plan
  PyObject* p = nullptr;
  Object() = default;
  explicit Object(PyObject* o) : p(o) { Py_XINCREF(p); }
  Object(Object&& o) noexcept : p(o.p) { o.p = nullptr; }
  Object& operator=(Object&& o) noexcept { std::swap(p, o.p); return *this; }
  ~Object() { Py_XDECREF(p); }
};

Object taken(PyObject* o) {              // a new reference
  Object t;
  t.p = o;
  return t;
}

struct Product {
  tnx_gemm_args args;
  int64_t rows, cols;
  at::ScalarType type;
  int64_t scratch, slices;
  bool atomic;
  Object memo_key, config;
};
struct Conv {
  tnx_conv2d_args args;
  int64_t shape[4], scratch;
};
// never destroyed: what they hold belongs to the interpreter, which is gone by the time destructors of statics run
std::unordered_map<Key, Product, Hash>& products = *new std::unordered_map<Key, Product, Hash>;
std::unordered_map<Key, Conv, Hash>& convs = *new std::unordered_map<Key, Conv, Hash>;

// an ordinary dense tensor on the GPU: nothing that intercepts the calls the Python path would make of it
bool plain(const at::Tensor& t, int64_t dim) {
  if (!t.defined() || !t.is_cuda() || t.dim() != dim || t.layout() != at::kStrided) return false;
  const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
  if (impl->is_python_dispatch()) return false;
  static const c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                          c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Batched});
  return !impl->key_set().has_any(other);
}

bool operand_key(int64_t tag, const at::Tensor& a, const at::Tensor& b, Key* k) {
  std::memset(k, 0, sizeof *k);
  k->tag = tag;
  for (int i = 0; i < 2; ++i) {
    k->sizes[i] = a.size(i); k->sizes[2 + i] = b.size(i);
    k->strides[i] = a.stride(i); k->strides[2 + i] = b.stride(i);
  }
  k->type_a = (int32_t)a.scalar_type(); k->type_b = (int32_t)b.scalar_type();
  k->device = a.get_device();
  k->aligned = (((uintptr_t)a.data_ptr() | (uintptr_t)b.data_ptr()) & 15) == 0;
  return b.get_device() == k->device;
}

at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type, c10::DeviceIndex device) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(c10::Device(c10::DeviceType::CUDA, device)));
}

bool tensor_arg(PyObject* o) { return THPVariable_Check(o); }
// a torch.Tensor or Parameter itself: a subclass may answer the Python path's calls in its own way, and gives its type to a result
// that comes from one of its methods (new_empty)
bool own_tensor(PyObject* o) { return THPVariable_CheckExact(o); }

// The interpreter lock is given back while memory is allocated and the launch is queued: both may wait for the GPU (an allocation
// that frees cached blocks, a full queue), and what the GPU waits for may be a host function or a thread that needs the lock.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// None, whatever Exception is set (the ordinary path meets its cause again); an interrupt or an exit goes on its way
PyObject* none() {
  if (PyErr_Occurred() && !PyErr_ExceptionMatches(PyExc_Exception)) return nullptr;
  PyErr_Clear();
  Py_RETURN_NONE;
}

// bind(tnx_gemm, tnx_gemm_f32, tnx_conv2d_forward, workspace, failed): addresses of the entry points
PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long g, f, c;
  PyObject *w, *e;
  if (!PyArg_ParseTuple(args, "KKKOO", &g, &f, &c, &w, &e)) return nullptr;
  fn_gemm = (decltype(fn_gemm))(uintptr_t)g;
  fn_gemm_f32 = (decltype(fn_gemm_f32))(uintptr_t)f;
  fn_conv = (decltype(fn_conv))(uintptr_t)c;
  Object workspace(w), failed(e);
  std::swap(fn_workspace, workspace.p);
  std::swap(fn_failed, failed.p);
  Py_RETURN_NONE;
}

// keep(tag, a, b, c, args, scratch, slices, atomic, memo key, config): the launch that gave c, from its argument struct's bytes
PyObject* keep(PyObject*, PyObject* args) {
  long long tag, scratch, slices;
  PyObject *a, *b, *c, *memo_key, *config;
  const char* bytes;
  Py_ssize_t len;
  int atomic;
  if (!PyArg_ParseTuple(args, "LOOOy#LLpOO", &tag, &a, &b, &c, &bytes, &len, &scratch, &slices, &atomic, &memo_key, &config)) return nullptr;
  if (len != (Py_ssize_t)sizeof(tnx_gemm_args) || !tensor_arg(a) || !tensor_arg(b) || !tensor_arg(c)) {
    PyErr_SetString(PyExc_ValueError, "keep: not an argument struct and its tensors");
    return nullptr;
  }
  try {
    const at::Tensor &ta = THPVariable_Unpack(a), &tb = THPVariable_Unpack(b), &tc = THPVariable_Unpack(c);
    Key k;
    if (!own_tensor(a) || !own_tensor(b) || !plain(ta, 2) || !plain(tb, 2) || !operand_key(tag, ta, tb, &k)) Py_RETURN_NONE;
    Product p;
    std::memcpy(&p.args, bytes, sizeof p.args);
    p.rows = tc.size(0); p.cols = tc.size(1);
    p.type = tc.scalar_type();
    p.scratch = scratch; p.slices = slices; p.atomic = atomic != 0;
    p.memo_key = Object(memo_key);
    p.config = Object(config);
    products[k] = std::move(p);
  } catch (...) {
    return none();
  }
  Py_RETURN_NONE;
}

// product(tag, a, b, memo, hooks) -> c, or None
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5 || !own_tensor(args[1]) || !own_tensor(args[2]) || !PyDict_Check(args[3]) || !PyList_Check(args[4]) ||
      PyList_GET_SIZE(args[4]) != 0)
    Py_RETURN_NONE;
  const long long tag = PyLong_AsLongLong(args[0]);
  if (PyErr_Occurred()) return nullptr;
  try {
    const at::Tensor &a = THPVariable_Unpack(args[1]), &b = THPVariable_Unpack(args[2]);
    Key k;
    if (products.empty() || !plain(a, 2) || !plain(b, 2) || !operand_key(tag, a, b, &k)) Py_RETURN_NONE;
    const auto hit = products.find(k);
    if (hit == products.end()) Py_RETURN_NONE;
    // by value: the comparison and the workspace call below run Python, and the lock is given back, behind which the entry may be
    // forgotten
    const Product& kept = hit->second;
    const struct { int64_t rows, cols; at::ScalarType type; int64_t scratch, slices; bool atomic; } p = {
        kept.rows, kept.cols, kept.type, kept.scratch, kept.slices, kept.atomic};
    tnx_gemm_args g = kept.args;
    const Object memo_key(kept.memo_key.p), config(kept.config.p);
    PyObject* now = PyDict_GetItemWithError(args[3], memo_key.p);        // the config memo may hold another tile by now
    if (!now) return none();
    const Object held(now);
    if (PyObject_RichCompareBool(now, config.p, Py_EQ) != 1) return none();
    const c10::DeviceIndex device = (c10::DeviceIndex)k.device;
    if (c10::hip::current_device() != device) Py_RETURN_NONE;
    g.a = a.data_ptr(); g.b = b.data_ptr();
    g.stream = c10::hip::getCurrentHIPStream(device).stream();
    // held until the launch is queued: while the lock is given back another thread may have the buffer replaced by a larger one
    // or evicted, and a block that goes back to the stream's pool before then is handed out again -- to the result below, even
    Object workspace;
    if (p.slices > 0) {
      workspace = taken(PyObject_CallFunction(fn_workspace, "iKLi", (int)device, (unsigned long long)(uintptr_t)g.stream, (long long)p.slices, (int)p.atomic));
      if (!workspace.p || !tensor_arg(workspace.p)) return none();
      const at::Tensor& ws = THPVariable_Unpack(workspace.p);
      g.workspace = ws.data_ptr();
      g.workspace_bytes = (size_t)ws.nbytes();
    }
    at::Tensor c;
    int status;
    {
      const Unlocked unlocked;
      c = fresh({p.rows, p.cols}, p.type, device);
      g.c = c.data_ptr();
      if (g.in_dtype == TNX_F32) {
        at::Tensor scratch;
        if (p.scratch > 0) scratch = fresh({p.scratch}, at::kByte, device);
        status = fn_gemm_f32(&g, p.scratch > 0 ? scratch.data_ptr() : nullptr, (size_t)p.scratch);
      } else {
        status = fn_gemm(&g);
      }
    }
    if (status != TNX_OK) {
      taken(PyObject_CallFunction(fn_failed, "iKiy#", (int)device, (unsigned long long)(uintptr_t)g.stream, status, (const char*)&g, (Py_ssize_t)sizeof g));
      return PyErr_Occurred() ? nullptr : none();
    }
    return THPVariable_Wrap(c);
  } catch (...) {
    return none();
  }
}

bool pair_of(PyObject* t, int64_t* out) {
  if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 2) return false;
  for (int i = 0; i < 2; ++i) {
    PyObject* v = PyTuple_GET_ITEM(t, i);
    if (!PyLong_CheckExact(v)) return false;
    out[i] = PyLong_AsLongLong(v);
  }
  return !PyErr_Occurred();
}

// (input, weight, bias or None, stride, padding, dilation) -> key; false: the ordinary path
bool conv_key(PyObject* const* args, Key* k) {
  if (!own_tensor(args[0]) || !own_tensor(args[1]) || !(args[2] == Py_None || own_tensor(args[2]))) return false;
  const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]);
  if (!plain(x, 4) || !plain(w, 4) || !x.is_contiguous() || !w.is_contiguous()) return false;
  std::memset(k, 0, sizeof *k);
  for (int i = 0; i < 4; ++i) { k->sizes[i] = x.size(i); k->sizes[4 + i] = w.size(i); }
  for (int i = 0; i < 3; ++i)
    if (!pair_of(args[3 + i], k->options + 2 * i)) { PyErr_Clear(); return false; }
  k->type_a = (int32_t)x.scalar_type(); k->type_b = (int32_t)w.scalar_type();
  k->device = x.get_device();
  k->type_c = -1;
  if (w.get_device() != k->device) return false;
  if (args[2] != Py_None) {
    const at::Tensor& bias = THPVariable_Unpack(args[2]);
    if (!plain(bias, 1) || !bias.is_contiguous() || bias.get_device() != k->device) return false;
    k->type_c = (int32_t)bias.scalar_type();
    k->count_c = (int32_t)bias.numel();
  }
  return true;
}

// keep_conv(input, weight, bias, stride, padding, dilation, args, shape, scratch)
PyObject* keep_conv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 9 || !PyBytes_Check(args[6]) || PyBytes_GET_SIZE(args[6]) != (Py_ssize_t)sizeof(tnx_conv2d_args) || !PyTuple_Check(args[7]) ||
      PyTuple_GET_SIZE(args[7]) != 4) {
    PyErr_SetString(PyExc_ValueError, "keep_conv: not an argument struct, a shape and a size");
    return nullptr;
  }
  try {
    Key k;
    if (!conv_key(args, &k)) Py_RETURN_NONE;
    Conv p;
    std::memcpy(&p.args, PyBytes_AS_STRING(args[6]), sizeof p.args);
    for (int i = 0; i < 4; ++i) p.shape[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[7], i));
    p.scratch = PyLong_AsLongLong(args[8]);
    if (PyErr_Occurred()) return nullptr;
    convs[k] = p;
  } catch (...) {
    return none();
  }
  Py_RETURN_NONE;
}

// conv(input, weight, bias, stride, padding, dilation) -> output, or None
PyObject* conv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6 || convs.empty()) Py_RETURN_NONE;
  try {
    Key k;
    if (!conv_key(args, &k)) Py_RETURN_NONE;
    const auto hit = convs.find(k);
    if (hit == convs.end()) Py_RETURN_NONE;
    const Conv p = hit->second;
    const c10::DeviceIndex device = (c10::DeviceIndex)k.device;
    if (c10::hip::current_device() != device) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]);
    tnx_conv2d_args a = p.args;
    a.input = x.data_ptr(); a.weight = w.data_ptr();
    a.bias = args[2] == Py_None ? nullptr : THPVariable_Unpack(args[2]).data_ptr();
    a.stream = c10::hip::getCurrentHIPStream(device).stream();
    at::Tensor y;
    int status;
    {
      const Unlocked unlocked;
      y = fresh({p.shape[0], p.shape[1], p.shape[2], p.shape[3]}, (at::ScalarType)k.type_a, device);
      at::Tensor scratch;
      if (p.scratch > 0) {
        scratch = fresh({p.scratch}, at::kByte, device);
        a.workspace = scratch.data_ptr();
        a.workspace_bytes = (size_t)p.scratch;
      }
      a.output = y.data_ptr();
      status = fn_conv(&a);
    }
    if (status != TNX_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(y);
  } catch (...) {
    return none();
  }
}

PyObject* forget(PyObject*, PyObject*) {
  products.clear();
  Py_RETURN_NONE;
}
PyObject* forget_convs(PyObject*, PyObject*) {
  convs.clear();
  Py_RETURN_NONE;
}

// the stream a launch on the device would go to, for tests
PyObject* stream_of(PyObject*, PyObject* arg) {
  const long index = PyLong_AsLong(arg);
  if (PyErr_Occurred()) return nullptr;
  return PyLong_FromUnsignedLongLong((unsigned long long)(uintptr_t)c10::hip::getCurrentHIPStream((c10::DeviceIndex)index).stream());
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"keep", keep, METH_VARARGS, nullptr},
    {"product", (PyCFunction)(void (*)(void))product, METH_FASTCALL, nullptr},
    {"keep_conv", (PyCFunction)(void (*)(void))keep_conv, METH_FASTCALL, nullptr},
    {"conv", (PyCFunction)(void (*)(void))conv, METH_FASTCALL, nullptr},
    {"forget", forget, METH_NOARGS, nullptr},
    {"forget_convs", forget_convs, METH_NOARGS, nullptr},
    {"stream_of", stream_of, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {      // whose classes it was compiled against
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
