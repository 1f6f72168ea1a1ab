// Native half of the op adapter (ops.py): a CPython extension with one callable per diopi* function that does what DIPU's
// generated C++ wrappers do per call (dipu/scripts/autogen_diopi_wrapper/diopi_wrapper_template.py:100-141): tensors become
// descriptors on the stack, Python numbers diopiScalar_t, a context is opened on the current stream unless the caller
// brings one, the entry point runs inside a named range with the interpreter lock released, and a return code other than
// success raises. Output shapes and dtypes are inferred here too (like, rows_of, broadcast_of).
//
// Why native: with the marshalling in Python (ctypes structures filled field by field) a call cost 25 us of host time, of
// which the launch itself is three, and every layer of small kernels was bound by it (16 calls of the fp32 block of
// 2 x 128 tokens: 357 us for 175 us of kernels).
//
// The diopi* and runtime symbols are looked up in the process when the module is imported (both libraries are loaded with
// global symbols before it), so this module links against neither.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/ExpandUtils.h>
#include <ATen/native/TypeProperties.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>

#include <new>
#include <type_traits>
#include <vector>

#include <diopi/functions.h>
#include <diopi/functions_ext.h>
#include <dipu_amd/runtime.h>

namespace {

PyObject* g_error = nullptr;       // the exception class of marshalling errors
PyObject* g_onFailure = nullptr;   // called with (name, return code): raises with the library's own text

// ------------------------------------------------------------------ runtime symbols
decltype(&dipuAmdContextCreate) g_contextCreate;
decltype(&dipuAmdContextDestroy) g_contextDestroy;
decltype(&diopiRecordStart) g_recordStart;
decltype(&diopiRecordEnd) g_recordEnd;

template <class F>
bool resolve(F* f, const char* name) {
  *f = reinterpret_cast<F>(dlsym(RTLD_DEFAULT, name));
  if (!*f) PyErr_Format(PyExc_ImportError, "%s is not loaded in this process", name);
  return *f != nullptr;
}

// ------------------------------------------------------------------ arguments
int dtypeOf(at::ScalarType t) {
  switch (t) {
    case at::kChar: return diopi_dtype_int8;
    case at::kByte: return diopi_dtype_uint8;
    case at::kShort: return diopi_dtype_int16;
    case at::kInt: return diopi_dtype_int32;
    case at::kLong: return diopi_dtype_int64;
    case at::kHalf: return diopi_dtype_float16;
    case at::kFloat: return diopi_dtype_float32;
    case at::kDouble: return diopi_dtype_float64;
    case at::kBool: return diopi_dtype_bool;
    case at::kBFloat16: return diopi_dtype_bfloat16;
    default: return diopi_dtype_unsupported;
  }
}

// The address in the `ptr` of an object of the ctypes view (a Handle, a Context): a c_void_p, or None for a closed one.
bool addressOf(PyObject* o, void** p) {
  PyObject* ptr = PyObject_GetAttrString(o, "ptr");
  PyObject* value = ptr && ptr != Py_None ? PyObject_GetAttrString(ptr, "value") : ptr;
  if (value != ptr) Py_XDECREF(ptr);
  if (!value) return false;
  *p = value == Py_None ? nullptr : PyLong_AsVoidPtr(value);
  Py_DECREF(value);
  return !PyErr_Occurred();
}

// A tensor's descriptor lives here for the length of the call; None is the null handle, and an object with a `ptr` (a
// Handle made by the ctypes view) passes that.
struct TensorArg {
  dipuAmdTensor d;
  void* p = nullptr;
  bool load(PyObject* o) {
    if (o == Py_None) return true;
    if (!THPVariable_Check(o)) {
      if (addressOf(o, &p)) return true;
      PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
      return false;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    const int64_t nd = t.dim();
    if (nd > DIPU_AMD_MAX_DIMS) {
      PyErr_Format(g_error, "tensors of rank %lld are not supported (max %d)", (long long)nd, DIPU_AMD_MAX_DIMS);
      return false;
    }
    const int dt = dtypeOf(t.scalar_type());
    if (dt == diopi_dtype_unsupported) {
      PyObject* name = PyObject_GetAttrString(o, "dtype");
      PyErr_Format(g_error, "dtype %S has no DIOPI equivalent on this backend", name ? name : Py_None);
      Py_XDECREF(name);
      return false;
    }
    d.data = t.data_ptr();
    d.ndim = nd;
    const auto shape = t.sizes(), stride = t.strides();
    for (int64_t i = 0; i < nd; ++i) d.shape[i] = shape[i], d.stride[i] = stride[i];
    d.dtype = dt;
    d.device = t.device().is_cpu() ? diopi_host : diopi_device;
    d.device_index = t.device().has_index() ? t.device().index() : -1;
    d.reserved = 0;
    d.storage_offset = t.storage_offset();
    d.storage_nbytes = t.storage().nbytes();
    d.storage_ptr = d.storage_nbytes ? const_cast<void*>(t.storage().data()) : nullptr;
    p = &d;
    return true;
  }
};

// Python integers are reduced modulo 2^64, as the fields of the ctypes view reduce them: a mask like 2^64 - 1 is -1.
int64_t integerOf(PyObject* o) { return static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(o)); }

template <class T>
struct Arg;
template <>
struct Arg<diopiTensorHandle_t> : TensorArg {
  diopiTensorHandle_t get() { return static_cast<diopiTensorHandle_t>(p); }
};
template <>
struct Arg<diopiConstTensorHandle_t> : TensorArg {
  diopiConstTensorHandle_t get() { return static_cast<diopiConstTensorHandle_t>(p); }
};
struct TensorListArg {
  PyObject* items = nullptr;  // a tuple of the tensors for the length of the call: a sequence may make them as it is read, a list may change
  std::vector<TensorArg> held;
  std::vector<diopiConstTensorHandle_t> handles;
  TensorListArg() = default;
  TensorListArg(const TensorListArg&) = delete;
  ~TensorListArg() { Py_XDECREF(items); }
  bool load(PyObject* o) {
    items = PySequence_Tuple(o);
    if (!items) return false;
    const Py_ssize_t n = PyTuple_GET_SIZE(items);
    held.resize(n), handles.resize(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
      if (!held[i].load(PyTuple_GET_ITEM(items, i))) return false;
      handles[i] = static_cast<diopiConstTensorHandle_t>(held[i].p);
    }
    return true;
  }
};
template <>
struct Arg<const diopiConstTensorHandle_t*> : TensorListArg {
  const diopiConstTensorHandle_t* get() { return handles.data(); }
};
template <>
struct Arg<diopiConstTensorHandle_t*> : TensorListArg {
  diopiConstTensorHandle_t* get() { return handles.data(); }
};
template <>
struct Arg<const diopiScalar_t*> {  // dipu/torch_dipu/csrc_dipu/diopirt/diopi_helper.cpp:74-97
  diopiScalar_t s;
  bool load(PyObject* o) {
    if (PyLong_Check(o)) {  // (a bool is one too)
      s.stype = diopi_dtype_int64;
      s.ival = integerOf(o);
      return !PyErr_Occurred();
    }
    if (PyFloat_Check(o)) {
      s.stype = diopi_dtype_float64;
      s.fval = PyFloat_AS_DOUBLE(o);
      return true;
    }
    PyErr_Format(PyExc_TypeError, "invalid scalar type %R", (PyObject*)Py_TYPE(o));
    return false;
  }
  const diopiScalar_t* get() { return &s; }
};
template <>
struct Arg<diopiSize_t> {
  std::vector<int64_t> v;
  bool load(PyObject* o) {
    PyObject* seq = PySequence_Fast(o, "expected a list of integers");
    if (!seq) return false;
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); ++i) v.push_back(integerOf(PySequence_Fast_GET_ITEM(seq, i)));
    Py_DECREF(seq);
    return !PyErr_Occurred();
  }
  diopiSize_t get() { return diopiSize_t{v.data(), (int64_t)v.size()}; }
};
template <class I>
struct IntegerArg {
  I v;
  bool load(PyObject* o) {
    v = static_cast<I>(integerOf(o));
    return !PyErr_Occurred();
  }
  I get() { return v; }
};
template <>
struct Arg<int64_t> : IntegerArg<int64_t> {};
template <>
struct Arg<int> : IntegerArg<int> {};
template <>
struct Arg<diopiRoundMode_t> : IntegerArg<diopiRoundMode_t> {};
template <>
struct Arg<bool> {
  bool v;
  bool load(PyObject* o) {
    const int r = PyObject_IsTrue(o);
    v = r == 1;
    return r >= 0;
  }
  bool get() { return v; }
};
template <>
struct Arg<double> {
  double v;
  bool load(PyObject* o) {
    v = PyFloat_AsDouble(o);
    return !PyErr_Occurred();
  }
  double get() { return v; }
};

// ------------------------------------------------------------------ calls
// C++ exceptions of the tensor library become the Python exceptions torch itself raises for them.
template <class F>
PyObject* translated(F&& f) {
  HANDLE_TH_ERRORS
  return f();
  END_HANDLE_TH_ERRORS
}

// The interpreter lock is released for the life of this object, and taken again also where an exception passes.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// args[0]: 0 to open a context on the current stream for this call, a Context to run in that (its address is read on every
// call: one that has been closed since is a null context, which the entry point refuses), or an address.
template <class... A, size_t... I>
PyObject* invoke(diopiError_t (*fn)(diopiContextHandle_t, A...), const char* name, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != (Py_ssize_t)sizeof...(A) + 1) return PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %d", name, (int)sizeof...(A) + 1, (int)n);
  return translated([&]() -> PyObject* {
    void* ctx = nullptr;
    const bool number = PyLong_Check(args[0]);
    if (number) ctx = PyLong_AsVoidPtr(args[0]);
    else if (!addressOf(args[0], &ctx)) return nullptr;
    if (number && !ctx && PyErr_Occurred()) return nullptr;
    std::tuple<Arg<A>...> held;
    if (!(std::get<I>(held).load(args[I + 1]) && ...)) return nullptr;
    void* own = nullptr;
    if (number && !ctx) {
      if (g_contextCreate(c10::hip::getCurrentHIPStream().stream(), &own) != 0) return PyObject_CallFunction(g_onFailure, "si", "dipuAmdContextCreate", 1);
      ctx = own;
    }
    diopiError_t rc;
    {
      Unlocked unlocked;
      void* record = nullptr;
      g_recordStart(name, &record);
      rc = fn(static_cast<diopiContextHandle_t>(ctx), std::get<I>(held).get()...);
      g_recordEnd(&record);
      if (own && rc == diopiSuccess) g_contextDestroy(own);
    }
    if (rc != diopiSuccess) {
      PyObject* r = PyObject_CallFunction(g_onFailure, "si", name, (int)rc);  // (reads the error text before the context goes)
      if (own) g_contextDestroy(own);
      return r;
    }
    Py_RETURN_NONE;
  });
}

template <class Tag>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return [&]<class... A>(diopiError_t (*fn)(diopiContextHandle_t, A...)) {
    return invoke(fn, Tag::name(), args, n, std::index_sequence_for<A...>{});
  }(Tag::fn);
}

#define DIOPI_FUNCTIONS(X)                                                                                                    \
  X(diopiAdd) X(diopiAddInp) X(diopiAddScalar) X(diopiAddInpScalar) X(diopiSub) X(diopiSubScalar) X(diopiMul) X(diopiMulInp)  \
  X(diopiMulScalar) X(diopiMulInpScalar) X(diopiDiv) X(diopiDivScalar) X(diopiSilu) X(diopiSiluInp) X(diopiSigmoid)           \
  X(diopiRsqrt) X(diopiNeg) X(diopiSin) X(diopiCos) X(diopiExp) X(diopiPow) X(diopiFill) X(diopiSoftmax) X(diopiMean)         \
  X(diopiCopyInp) X(diopiCat) X(diopiIndexPutInp) X(diopiWhere) X(diopiMaskedFill) X(diopiMaskedFillInp)                      \
  X(diopiMaskedFillScalar) X(diopiMaskedFillInpScalar) X(diopiTril) X(diopiTriu) X(diopiTriuInp) X(diopiArange)               \
  X(diopiIndexSelect) X(diopiGather) X(diopiEq) X(diopiEqScalar) X(diopiNe) X(diopiNeScalar) X(diopiLt) X(diopiLtScalar)      \
  X(diopiLe) X(diopiLeScalar) X(diopiGt) X(diopiGtScalar) X(diopiGe) X(diopiGeScalar) X(diopiMm) X(diopiBmm) X(diopiMatmul)   \
  X(diopiAddmm) X(diopiBaddbmm) X(diopiLinear) X(diopiRMSNorm) X(diopiRotaryEmbedding) X(diopiDestIndexCopyKV)                \
  X(diopiDestIndexCopyKVPair) X(diopiTokenAttentionInference) X(diopiTokenSoftmaxReduceVInference)                            \
  X(diopiContextAttentionInference) X(diopiTokenDecodeAttentionInference) X(diopiTokenDecodeAttentionInferenceNoAlloc)        \
  X(diopiWeightOnlyInt8Linear) X(diopiSiluMul) X(diopiLinearSiluMul) X(diopiLinearRotary)

#define X(f)                                        \
  struct Tag_##f {                                  \
    static decltype(&::f) fn;                       \
    static const char* name() { return #f; }        \
  };                                                \
  decltype(&::f) Tag_##f::fn = nullptr;
DIOPI_FUNCTIONS(X)
#undef X

// ------------------------------------------------------------------ outputs
const at::Tensor* tensorOf(PyObject* o) {
  if (THPVariable_Check(o)) return &THPVariable_Unpack(o);
  PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
  return nullptr;
}

// like(t): an empty dense tensor of t's shape and dtype.
PyObject* like(PyObject*, PyObject* o) {
  return translated([&]() -> PyObject* {
    const at::Tensor* t = tensorOf(o);
    return t ? THPVariable_Wrap(at::empty(t->sizes(), t->options())) : nullptr;
  });
}

// rows_of(t, n): an empty dense tensor of t's shape with the last extent n.
PyObject* rowsOf(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2) return PyErr_Format(PyExc_TypeError, "rows_of takes 2 arguments");
  return translated([&]() -> PyObject* {
    const at::Tensor* t = tensorOf(args[0]);
    const int64_t cols = PyLong_AsLongLong(args[1]);
    if (!t || PyErr_Occurred()) return nullptr;
    auto shape = t->sizes().vec();
    if (shape.empty()) return PyErr_Format(PyExc_IndexError, "a tensor without dims has no rows");
    shape.back() = cols;
    return THPVariable_Wrap(at::empty(shape, t->options()));
  });
}

// broadcast_of(a, b, bool): an empty dense tensor on a's device of the shape a and b (a tensor or a number) broadcast to
// and of their promoted dtype, or bool.
PyObject* broadcastOf(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 3) return PyErr_Format(PyExc_TypeError, "broadcast_of takes 3 arguments");
  return translated([&]() -> PyObject* {
    const at::Tensor* a = tensorOf(args[0]);
    const bool toBool = args[2] == Py_True;
    if (!a) return nullptr;
    PyObject* o = args[1];
    if (THPVariable_Check(o)) {
      const at::Tensor& b = THPVariable_Unpack(o);
      const at::ScalarType dt = toBool ? at::kBool : a->scalar_type() == b.scalar_type() ? a->scalar_type() : at::result_type(*a, b);
      if (a->sizes() == b.sizes()) return THPVariable_Wrap(at::empty(a->sizes(), a->options().dtype(dt)));
      return THPVariable_Wrap(at::empty(at::infer_size_dimvector(a->sizes(), b.sizes()), a->options().dtype(dt)));
    }
    at::ScalarType dt = at::kBool;
    if (!toBool) {
      if (PyBool_Check(o)) dt = at::result_type(*a, at::Scalar(o == Py_True));
      else if (PyLong_Check(o)) {
        int beyond = 0;
        (void)PyLong_AsLongLongAndOverflow(o, &beyond);
        if (beyond) (void)PyLong_AsUnsignedLongLong(o);  // (torch promotes with whatever 64 bits hold, and refuses the rest)
        if (PyErr_Occurred()) return nullptr;
        dt = at::result_type(*a, at::Scalar((int64_t)0));  // the kind of the number counts, not its value
      }
      else if (PyFloat_Check(o)) dt = at::result_type(*a, at::Scalar(0.0));
      else return PyErr_Format(PyExc_TypeError, "invalid scalar type %R", (PyObject*)Py_TYPE(o));
    }
    return THPVariable_Wrap(at::empty(a->sizes(), a->options().dtype(dt)));
  });
}

// setup(error class, failure callback): resolves every entry point.
PyObject* setup(PyObject*, PyObject* args) {
  PyObject *error, *onFailure;
  if (!PyArg_ParseTuple(args, "OO", &error, &onFailure)) return nullptr;
  if (!resolve(&g_contextCreate, "dipuAmdContextCreate") || !resolve(&g_contextDestroy, "dipuAmdContextDestroy") ||
      !resolve(&g_recordStart, "diopiRecordStart") || !resolve(&g_recordEnd, "diopiRecordEnd"))
    return nullptr;
#define X(f) \
  if (!resolve(&Tag_##f::fn, #f)) return nullptr;
  DIOPI_FUNCTIONS(X)
#undef X
  Py_INCREF(error), Py_INCREF(onFailure);
  g_error = error, g_onFailure = onFailure;
  Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
#define X(f) {#f, (PyCFunction)(void (*)(void))&entry<Tag_##f>, METH_FASTCALL, nullptr},
    DIOPI_FUNCTIONS(X)
#undef X
    {"like", like, METH_O, nullptr},
    {"rows_of", (PyCFunction)(void (*)(void))rowsOf, METH_FASTCALL, nullptr},
    {"broadcast_of", (PyCFunction)(void (*)(void))broadcastOf, METH_FASTCALL, nullptr},
    {"setup", setup, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "dipu_amd_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_dipu_amd_host() { return PyModule_Create(&g_module); }
