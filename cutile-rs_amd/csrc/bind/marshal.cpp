// CPython extension behind the launcher functions of the Python binding: reads torch tensors into the ABI's records and
// calls the entry launcher, in one call from Python.
//
// A launch from Python was bound by this marshalling: filling ctypes records field by field took 1.5 us a tensor and 2.4 us a
// partition, and asking torch for its current stream 2.9 us, of 11.4 us for a saxpy launch whose C part takes 3.4 us.  Nothing
// here computes or decides anything; the addresses of the launchers come from the library that the binding loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/core/ScalarType.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <string>
#include <tuple>
#include <utility>

#include "../../../include/cutile_hip.h"

namespace {

PyObject *s_tensor, *s_shape, *s_prefix, *s_dtype, *s_arg;   // attribute names of the binding's Partition

// What the binding does in Python for the objects that are not read here: anything that offers a tensor's or a partition's methods.
struct Binding {
  PyObject* tensor_arg;        // tensor_arg(object, element type or None) -> the ABI's record as a ctypes structure
  PyObject* partition_type;    // the class Partition; objects of any other class are asked for their record: o.arg()
  PyObject* stream_source;     // () -> (ordinal of the current device, (ordinal) -> handle of its current stream), or None without a GPU
  PyObject* check;             // check(status) raises
};
// That pair, once it is known: a GPU that torch has found stays.
PyObject *s_device_of = nullptr, *s_stream_of = nullptr;

// Copies a ctypes structure; takes the reference.
template <typename T>
bool take_record(PyObject* record, T* out) {
  if (!record) return false;
  Py_buffer view;
  bool ok = PyObject_GetBuffer(record, &view, PyBUF_SIMPLE) == 0;
  if (ok) {
    ok = view.len == (Py_ssize_t)sizeof(T);
    if (ok)
      memcpy(out, view.buf, sizeof(T));
    else
      PyErr_Format(PyExc_TypeError, "expected a record of %zd bytes, got one of %zd (%s)", (Py_ssize_t)sizeof(T), view.len, Py_TYPE(record)->tp_name);
    PyBuffer_Release(&view);
  }
  Py_DECREF(record);
  return ok;
}

int dtype_of(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return CUTILE_DTYPE_F32;
    case at::kDouble: return CUTILE_DTYPE_F64;
    case at::kHalf: return CUTILE_DTYPE_F16;
    case at::kBFloat16: return CUTILE_DTYPE_BF16;
    case at::kChar: return CUTILE_DTYPE_I8;
    case at::kShort: return CUTILE_DTYPE_I16;
    case at::kInt: return CUTILE_DTYPE_I32;
    case at::kLong: return CUTILE_DTYPE_I64;
    case at::kByte: return CUTILE_DTYPE_U8;
    case at::kUInt16: return CUTILE_DTYPE_U16;
    case at::kUInt32: return CUTILE_DTYPE_U32;
    case at::kUInt64: return CUTILE_DTYPE_U64;
    case at::kBool: return CUTILE_DTYPE_BOOL;
    case at::kFloat8_e4m3fn: return CUTILE_DTYPE_F8E4M3FN;
    case at::kFloat8_e5m2: return CUTILE_DTYPE_F8E5M2;
    case at::kFloat8_e8m0fnu: return CUTILE_DTYPE_F8E8M0FNU;
    default: return -1;
  }
}

bool fill_tensor(PyObject* o, int dtype, const Binding& b, cutile_tensor_arg_t* a) try {
  if (!THPVariable_Check(o))
    return take_record(dtype < 0 ? PyObject_CallFunctionObjArgs(b.tensor_arg, o, nullptr) : PyObject_CallFunction(b.tensor_arg, "Oi", o, dtype), a);
  const at::Tensor& t = THPVariable_Unpack(o);
  const int64_t rank = t.dim();
  if (rank > CUTILE_MAX_RANK) {
    PyErr_Format(PyExc_IndexError, "a tensor argument has at most %d axes, got %lld", CUTILE_MAX_RANK, (long long)rank);
    return false;
  }
  if (dtype < 0 && (dtype = dtype_of(t)) < 0) {
    PyErr_SetString(PyExc_KeyError, "torch dtype without an element type of the ABI");
    return false;
  }
  a->ptr = t.data_ptr();
  a->dtype = (cutile_dtype_t)dtype;
  a->rank = (int32_t)rank;
  const auto sizes = t.sizes(), strides = t.strides();
  for (int64_t i = 0; i < CUTILE_MAX_RANK; ++i) {
    a->shape[i] = i < rank ? (int32_t)sizes[i] : 0;
    a->strides[i] = i < rank ? (int32_t)strides[i] : 0;
  }
  return true;
} catch (const std::exception& e) {   // a tensor without plain storage
  PyErr_SetString(PyExc_RuntimeError, e.what());
  return false;
}

bool to_int(PyObject* o, long long* v) {
  if (PyFloat_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "expected an integer, got a float");
    return false;
  }
  *v = PyLong_AsLongLong(o);
  return !(*v == -1 && PyErr_Occurred());
}

bool fill_partition(PyObject* o, const Binding& b, cutile_partition_arg_t* p) {
  if ((PyObject*)Py_TYPE(o) != b.partition_type) return take_record(PyObject_CallMethodNoArgs(o, s_arg), p);
  PyObject *tensor = PyObject_GetAttr(o, s_tensor), *shape = nullptr, *prefix = nullptr, *dtype = nullptr;
  bool ok = tensor && (shape = PyObject_GetAttr(o, s_shape)) && (prefix = PyObject_GetAttr(o, s_prefix)) && (dtype = PyObject_GetAttr(o, s_dtype));
  long long code = -1;
  if (ok && dtype != Py_None) ok = to_int(dtype, &code);
  ok = ok && fill_tensor(tensor, (int)code, b, &p->tensor);
  PyObject* seq = ok ? PySequence_Fast(shape, "a partition's shape is a sequence of integers") : nullptr;
  if ((ok = seq != nullptr)) {
    if (PySequence_Fast_GET_SIZE(seq) != p->tensor.rank) {
      Py_XDECREF(PyObject_CallMethodNoArgs(o, s_arg));   // raises the binding's error
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "partition rank does not match tensor rank");
      ok = false;
    }
    for (int i = 0; ok && i < CUTILE_MAX_RANK; ++i) {
      long long v = 0;
      if (i < p->tensor.rank) ok = to_int(PySequence_Fast_GET_ITEM(seq, i), &v);
      p->partition_shape[i] = (int32_t)v;
      p->partition_strides[i] = p->tensor.strides[i];   // cutile/src/tensor.rs:1423-1427
    }
    p->prefix_coverage = PyObject_IsTrue(prefix);
  }
  Py_XDECREF(seq);
  Py_XDECREF(tensor);
  Py_XDECREF(shape);
  Py_XDECREF(prefix);
  Py_XDECREF(dtype);
  return ok;
}

// The stream of a launch: the caller's, or the current one of torch.
bool read_stream(PyObject* o, const Binding& b, void** stream) {
  PyObject* handle;
  if (o != Py_None) {
    handle = PyNumber_Long(o);
  } else {
    if (!s_stream_of) {
      PyObject* pair = PyObject_CallNoArgs(b.stream_source);
      if (!pair) return false;
      if (pair == Py_None || !PyArg_ParseTuple(pair, "OO", &s_device_of, &s_stream_of)) {
        const bool none = pair == Py_None;
        Py_DECREF(pair);
        *stream = nullptr;
        return none;
      }
      Py_INCREF(s_device_of);
      Py_INCREF(s_stream_of);
      Py_DECREF(pair);
    }
    PyObject* device = PyObject_CallNoArgs(s_device_of);
    handle = device ? PyObject_CallOneArg(s_stream_of, device) : nullptr;
    Py_XDECREF(device);
  }
  if (!handle) return false;
  *stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return !PyErr_Occurred();
}

// ---- one Python argument -> one argument of the launcher ----
template <typename T>
struct From;
template <>
struct From<void*> {   // a stream or a device address
  void* v;
  bool read(PyObject* o, const Binding&) {
    v = o == Py_None ? nullptr : PyLong_AsVoidPtr(o);
    return !PyErr_Occurred();
  }
  void* get() { return v; }
};
template <>
struct From<const void*> : From<void*> {};
template <>
struct From<int32_t> {
  long long v;
  bool read(PyObject* o, const Binding&) { return to_int(o, &v); }
  int32_t get() { return (int32_t)v; }
};
template <>
struct From<int64_t> : From<int32_t> {
  int64_t get() { return v; }
};
template <>
struct From<double> {
  double v;
  bool read(PyObject* o, const Binding&) {
    v = PyFloat_AsDouble(o);
    return !(v == -1.0 && PyErr_Occurred());
  }
  double get() { return v; }
};
template <>
struct From<float> : From<double> {
  float get() { return (float)v; }
};
template <>
struct From<const int32_t*> {   // a sequence of at most 8 integers
  int32_t v[8];
  bool read(PyObject* o, const Binding&) {
    PyObject* seq = PySequence_Fast(o, "expected a sequence of integers");
    bool ok = seq != nullptr;
    if (ok && PySequence_Fast_GET_SIZE(seq) > 8) {
      PyErr_SetString(PyExc_IndexError, "at most 8 integers");
      ok = false;
    }
    for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(seq); ++i) {
      long long x = 0;
      ok = to_int(PySequence_Fast_GET_ITEM(seq, i), &x);
      v[i] = (int32_t)x;
    }
    Py_XDECREF(seq);
    return ok;
  }
  const int32_t* get() { return v; }
};
template <>
struct From<const cutile_tensor_arg_t*> {   // a tensor, (tensor, element type) or None
  cutile_tensor_arg_t a;
  bool present;
  bool read(PyObject* o, const Binding& b) {
    if (!(present = o != Py_None)) return true;
    if (!PyTuple_Check(o)) return fill_tensor(o, -1, b, &a);
    if (PyTuple_GET_SIZE(o) != 2) {
      PyErr_SetString(PyExc_TypeError, "expected a tensor, got a tuple");
      return false;
    }
    long long code;
    return to_int(PyTuple_GET_ITEM(o, 1), &code) && fill_tensor(PyTuple_GET_ITEM(o, 0), (int)code, b, &a);
  }
  const cutile_tensor_arg_t* get() { return present ? &a : nullptr; }
};
template <>
struct From<const cutile_partition_arg_t*> {
  cutile_partition_arg_t a;
  bool read(PyObject* o, const Binding& b) { return fill_partition(o, b, &a); }
  const cutile_partition_arg_t* get() { return &a; }
};
template <>
struct From<const cutile_launch_opts_t*> {   // (grid or None, generics or None, variant or None), or None
  static constexpr int kMost = 16;
  cutile_launch_opts_t o{};
  std::string text[kMost];
  const char* items[kMost];
  bool read(PyObject* t, const Binding&) {
    if (t == Py_None) return true;
    PyObject *grid = PyTuple_GET_ITEM(t, 0), *generics = PyTuple_GET_ITEM(t, 1), *variant = PyTuple_GET_ITEM(t, 2);
    if (grid != Py_None) {
      PyObject* seq = PySequence_Fast(grid, "a grid is a sequence of three integers");
      bool ok = seq != nullptr;
      if (ok && PySequence_Fast_GET_SIZE(seq) < 3) {
        PyErr_SetString(PyExc_IndexError, "a grid has three axes");
        ok = false;
      }
      for (int i = 0; ok && i < 3; ++i) {
        long long v = 0;
        ok = to_int(PySequence_Fast_GET_ITEM(seq, i), &v);
        o.grid[i] = (uint32_t)v;
      }
      Py_XDECREF(seq);
      if (!ok) return false;
    }
    if (generics != Py_None) {
      PyObject* seq = PySequence_Fast(generics, "generics are a sequence");
      if (!seq) return false;
      const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
      bool ok = n <= kMost;
      if (!ok) PyErr_Format(PyExc_ValueError, "at most %d generics", kMost);
      for (Py_ssize_t i = 0; ok && i < n; ++i) {
        PyObject* s = PyObject_Str(PySequence_Fast_GET_ITEM(seq, i));
        const char* c = s ? PyUnicode_AsUTF8(s) : nullptr;
        if ((ok = c != nullptr)) text[i] = c, items[i] = text[i].c_str();
        Py_XDECREF(s);
      }
      Py_DECREF(seq);
      if (!ok) return false;
      o.generics = items;
      o.n_generics = (int32_t)n;
    }
    if (variant != Py_None && !(o.variant = PyUnicode_AsUTF8(variant))) return false;
    return true;
  }
  const cutile_launch_opts_t* get() { return &o; }
};

template <typename... A, size_t... I>
PyObject* call_with(cutile_status_t (*fn)(cutile_stream_t, A...), const Binding& b, PyObject* const* args, std::index_sequence<I...>) {
  void* stream;
  std::tuple<From<A>...> from;
  if (!read_stream(args[0], b, &stream) || !(std::get<I>(from).read(args[1 + I], b) && ...)) return nullptr;
  cutile_status_t status;
  Py_BEGIN_ALLOW_THREADS   // a launch may wait for room in a full queue
  status = fn((cutile_stream_t)stream, std::get<I>(from).get()...);
  Py_END_ALLOW_THREADS
  if (status == CUTILE_SUCCESS) Py_RETURN_NONE;
  return PyObject_CallFunction(b.check, "i", (int)status);
}
template <typename... A>
PyObject* call(cutile_status_t (*fn)(cutile_stream_t, A...), const Binding& b, PyObject* const* args, Py_ssize_t n) {
  if (n != 1 + (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "the launcher takes %zd arguments, got %zd", 1 + (Py_ssize_t)sizeof...(A), n);
  return call_with(fn, b, args, std::make_index_sequence<sizeof...(A)>());
}

// A launcher of one loaded library: name -> signature from the header, address from the binding.
#define LAUNCHERS(X)                                                                                                          \
  X(saxpy) X(axpy) X(add) X(relu) X(dropout) X(scale_ptr) X(matvec) X(batch_matmul) X(convert) X(rms_norm_f16) X(rms_norm_f32) \
  X(softmax) X(rms_norm_all_f16) X(softmax_all_f16) X(add_rms_norm_f16) X(qk_norm_f16) X(add_2d_f16) X(silu_mul_2d_f16)       \
  X(kv_cache_update_f16) X(fmha_decode_gqa_split) X(splitk_reduce_merge) X(fmha_decode_gqa_noalloc) X(rope_f16) X(gemm) X(fmha) \
  X(add_rms_norm_decode_raw_f16) X(qk_norm_rope_kv_prefill_raw_f16) X(qk_norm_rope_kv_decode_raw_f16) X(group_gemm_f16_nt_desc) \
  X(argmax_blocks_f16) X(lm_head_argmax_blocks_f16) X(argmax_reduce_blocks_to_u32) X(embedding_batch_f16) X(gather_row_f16)   \
  X(fmha_prefill_gqa_lpt_raw_f16) X(fmha_seq_f16) X(linear_tile_mxfp8) X(linear_tile_nvfp4) \
  X(attention_decode_kernel_grouped_f16)

struct Launcher {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  void* address;
  Binding binding;             // owned references
  PyObject* (*invoke)(const Launcher& l, PyObject* const* args, Py_ssize_t n);
};
PyObject* launcher_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  if (kwnames && PyTuple_GET_SIZE(kwnames)) return PyErr_Format(PyExc_TypeError, "a launcher takes positional arguments only");
  Launcher* l = (Launcher*)self;
  return l->invoke(*l, args, PyVectorcall_NARGS(nargsf));
}
void launcher_dealloc(PyObject* self) {
  Binding& b = ((Launcher*)self)->binding;
  Py_XDECREF(b.tensor_arg);
  Py_XDECREF(b.partition_type);
  Py_XDECREF(b.stream_source);
  Py_XDECREF(b.check);
  PyObject_Free(self);
}
PyTypeObject launcher_type = {PyVarObject_HEAD_INIT(nullptr, 0) "cutile_marshal.Launcher", sizeof(Launcher)};

#define INVOKE(NAME)                                                                      \
  PyObject* invoke_##NAME(const Launcher& l, PyObject* const* args, Py_ssize_t n) {       \
    return call(reinterpret_cast<decltype(&cutile_launch_##NAME)>(l.address), l.binding, args, n); \
  }
LAUNCHERS(INVOKE)

const struct { const char* name; PyObject* (*invoke)(const Launcher&, PyObject* const*, Py_ssize_t); } kLaunchers[] = {
#define ROW(NAME) {#NAME, invoke_##NAME},
    LAUNCHERS(ROW)};

PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  for (auto& k : kLaunchers) {
    PyObject* s = list ? PyUnicode_FromString(k.name) : nullptr;
    if (!s || PyList_Append(list, s) < 0) {
      Py_XDECREF(s);
      Py_XDECREF(list);
      return nullptr;
    }
    Py_DECREF(s);
  }
  return list;
}

PyObject* launcher(PyObject*, PyObject* args) {
  const char* name;
  unsigned long long address;
  PyObject *tensor_arg, *partition_type, *stream_source, *check;
  if (!PyArg_ParseTuple(args, "sKOOOO", &name, &address, &tensor_arg, &partition_type, &stream_source, &check)) return nullptr;
  for (auto& k : kLaunchers)
    if (strcmp(k.name, name) == 0) {
      Launcher* l = PyObject_New(Launcher, &launcher_type);
      if (!l) return nullptr;
      l->vectorcall = launcher_call;
      l->address = (void*)(uintptr_t)address;
      Py_INCREF(tensor_arg);
      Py_INCREF(partition_type);
      Py_INCREF(stream_source);
      Py_INCREF(check);
      l->binding = {tensor_arg, partition_type, stream_source, check};
      l->invoke = k.invoke;
      return (PyObject*)l;
    }
  return PyErr_Format(PyExc_KeyError, "no launcher %s", name);
}

PyMethodDef methods[] = {{"names", names, METH_NOARGS, "names of the launchers this module can call"},
                         {"launcher", launcher, METH_VARARGS, "launcher(name, address, tensor_arg, Partition, stream_source, check): the callable for cutile_launch_<name> at that address"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "cutile_marshal", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_cutile_marshal() {
  s_tensor = PyUnicode_InternFromString("tensor");
  s_shape = PyUnicode_InternFromString("shape");
  s_prefix = PyUnicode_InternFromString("prefix");
  s_dtype = PyUnicode_InternFromString("dtype");
  s_arg = PyUnicode_InternFromString("arg");
  launcher_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  launcher_type.tp_vectorcall_offset = offsetof(Launcher, vectorcall);
  launcher_type.tp_call = PyVectorcall_Call;
  launcher_type.tp_dealloc = launcher_dealloc;
  if (PyType_Ready(&launcher_type) < 0) return nullptr;
  return PyModule_Create(&module);
}
