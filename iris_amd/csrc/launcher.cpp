// Python module `_launch`: from an operator call in Python to the entry points of libiris_hip.so.
//
// A small launch runs 4-8 us on the GPU; checking an operator's arguments in Python and passing thirty of them
// through ctypes took the host 8-10 us, so that programs of small calls ran at the host's pace.  Two layers:
//
//   <entry>(...)   one entry point with its C arguments (pointers as integers or None, the rest as int / float), returns
//                  its int.  Types come from the declarations in iris_hip.h.
//   try_<op>(...)  a whole operator call on its tensors: reads what the Python wrapper reads, and when every argument
//                  is as it should be and the workspace can be used as it is, calls the entry point and returns its int.
//                  Anything else - an argument to report, a preamble to run - returns None with nothing done, and the
//                  Python wrapper takes the call from its start.  The wrapper is the authority on what is an error.
//                  An entry point that fails is not called again: its error may be an earlier call's, found behind
//                  a launch that went out.
//
//   load(path)     dlopen the library (once) and resolve the entry points; raises OSError
#include <c10/hip/HIPCachingAllocator.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <dlfcn.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "iris_hip.h"

namespace {

// ------------------------------------------------------------------------------------------------
// Entry points with C arguments
// ------------------------------------------------------------------------------------------------
template <class T>
T convert(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    return o == Py_None ? nullptr : (T)PyLong_AsUnsignedLongLong(o);
  } else if constexpr (std::is_floating_point_v<T>) {
    return (T)PyFloat_AsDouble(o);
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (v != (T)v && !PyErr_Occurred()) PyErr_Format(PyExc_OverflowError, "%lld does not fit a 32-bit argument", v);
    return (T)v;
  }
}

template <class... A, size_t... I>
PyObject* invoke(int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  const std::tuple<A...> v{convert<A>(args[I])...};
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

template <class... A>
PyObject* call(int (*fn)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
  if (!fn) return PyErr_Format(PyExc_RuntimeError, "%s: load() the library first", name);
  if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, (Py_ssize_t)sizeof...(A), n);
  return invoke(fn, args, std::index_sequence_for<A...>{});
}

#define ENTRY_POINTS(X)             \
  X(iris_hip_matmul_all_reduce)     \
  X(iris_hip_matmul_reduce_scatter) \
  X(iris_hip_all_gather_matmul)     \
  X(iris_hip_matmul_all_gather)     \
  X(iris_hip_all_reduce)            \
  X(iris_hip_reduce_scatter)

int (*fn_stream_capturing)(void*) = nullptr;

#define DEFINE(name)                     \
  decltype(&::name) fn_##name = nullptr; \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) { return call(fn_##name, #name, args, n); }
ENTRY_POINTS(DEFINE)

// Memory for the length of a launch comes from torch's caching allocator, which hands a block on to later work of the same
// stream only.
void* allocate_scratch(size_t bytes, void* stream) noexcept {
  try {
    return c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, (hipStream_t)stream);
  } catch (...) {
    return nullptr;
  }
}
void release_scratch(void* memory) noexcept {
  try {
    c10::hip::HIPCachingAllocator::raw_delete(memory);
  } catch (...) {
  }
}

PyObject* load(PyObject*, PyObject* path_object) {
  const char* path = PyUnicode_AsUTF8(path_object);
  if (!path) return nullptr;
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) return PyErr_Format(PyExc_OSError, "%s", dlerror());
#define RESOLVE(name)                                 \
  fn_##name = (decltype(fn_##name))dlsym(lib, #name); \
  if (!fn_##name) return PyErr_Format(PyExc_OSError, "%s has no %s", path, #name);
  ENTRY_POINTS(RESOLVE)
  fn_stream_capturing = (decltype(fn_stream_capturing))dlsym(lib, "iris_hip_stream_capturing");
  if (!fn_stream_capturing) return PyErr_Format(PyExc_OSError, "%s has no iris_hip_stream_capturing", path);
  const auto set_allocator = (decltype(&::iris_hip_set_scratch_allocator))dlsym(lib, "iris_hip_set_scratch_allocator");
  if (set_allocator) set_allocator(allocate_scratch, release_scratch);
  Py_RETURN_NONE;
}

// ------------------------------------------------------------------------------------------------
// Whole operator calls
// ------------------------------------------------------------------------------------------------
#define ATTRIBUTES(X)                                                                                                   \
  X(cur_rank) X(num_ranks) X(gpu_id) X(spin_limit) X(_device_context) X(_status) X(_own_begin) X(_own_end) X(heap_bases) \
  X(runs_alone) X(block_size_m) X(block_size_n) X(block_size_k) X(group_size_m) X(num_sms) X(num_xcds) X(chunk_size)     \
  X(all_reduce_variant) X(all_reduce_num_rings) X(all_reduce_distribution) X(reduce_scatter_variant) X(swizzle_size)     \
  X(comm_sms) X(use_gluon) X(operation) X(shape) X(dtype) X(world_size) X(variant) X(aux_buffer) X(locks) X(prepared)    \
  X(stream) X(captured)
#define ATTRIBUTE_NAME(name) PyObject* at_##name = nullptr;
ATTRIBUTES(ATTRIBUTE_NAME)

// Thrown (and caught at the boundary) when a call is one for the Python wrapper.
struct Decline {};
inline void require(bool ok) {
  if (!ok) throw Decline{};
}

struct Ref {
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) { require(p != nullptr); }
  ~Ref() { Py_DECREF(o); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

long long as_int(PyObject* o) {
  require(PyLong_Check(o));
  const long long v = PyLong_AsLongLong(o);
  require(v != -1 || !PyErr_Occurred());
  return v;
}
long long int_of(PyObject* o, PyObject* name) { return as_int(Ref(PyObject_GetAttr(o, name)).o); }
int positive(PyObject* o, PyObject* name) {
  const long long v = int_of(o, name);
  require(v > 0 && v < (1ll << 31));
  return (int)v;
}
bool is_text(PyObject* o, const char* text) { return PyUnicode_Check(o) && PyUnicode_CompareWithASCIIString(o, text) == 0; }

// A plain tensor (no subclass), borrowed from an object that outlives the call.
const at::Tensor& tensor(PyObject* o) {
  require(THPVariable_CheckExact(o));
  return THPVariable_Unpack(o);
}

int type_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return IRIS_HIP_BF16;
    case at::kHalf: return IRIS_HIP_FP16;
    case at::kFloat: return IRIS_HIP_FP32;
    case at::kFloat8_e4m3fn: return IRIS_HIP_FP8_E4M3;
    default: throw Decline{};
  }
}

struct Shmem {
  PyObject* o;
  int rank, world, device;
  explicit Shmem(PyObject* s) : o(s), rank((int)int_of(s, at_cur_rank)), world((int)int_of(s, at_num_ranks)), device((int)int_of(s, at_gpu_id)) {
    require(device >= 0);
  }
  void on_device(const at::Tensor& t) const { require(t.is_cuda() && t.get_device() == device); }
  bool symmetric(const at::Tensor& t) const {
    const long long p = (long long)t.const_data_ptr();
    return t.is_cuda() && int_of(o, at__own_begin) <= p && p < int_of(o, at__own_end);
  }
  const int64_t* words(PyObject* name) const { return (const int64_t*)tensor(Ref(PyObject_GetAttr(o, name)).o).const_data_ptr(); }
  int32_t* status() const { return (int32_t*)tensor(Ref(PyObject_GetAttr(o, at__status)).o).mutable_data_ptr(); }
  bool runs_alone() const { return Ref(PyObject_CallMethodNoArgs(o, at_runs_alone)).o == Py_True; }
};

struct Matrix {
  const at::Tensor& t;
  int64_t rows, cols, s0, s1;
  void* data;
  Matrix(PyObject* o, const Shmem& shmem) : t(tensor(o)) {
    require(t.dim() == 2);
    shmem.on_device(t);
    rows = t.size(0), cols = t.size(1), s0 = t.stride(0), s1 = t.stride(1);
    require(rows > 0 && cols > 0);
    data = t.mutable_data_ptr();  // (here, where it may throw: a tensor inside vmap has no memory to point at)
  }
  void* ptr() const { return data; }
};

struct Blocks {
  int m, n, k;
  explicit Blocks(PyObject* config)
      : m(positive(config, at_block_size_m)), n(positive(config, at_block_size_n)), k(positive(config, at_block_size_k)) {}
  void fit(int64_t rows, int64_t cols, int64_t depth) const { require(rows >= m && cols >= n && depth >= k); }
  // The rest of what FusedConfig.validate looks at.
  static void validate(PyObject* config) {
    positive(config, at_group_size_m), positive(config, at_num_xcds), positive(config, at_chunk_size), positive(config, at_all_reduce_num_rings);
    const Ref sms(PyObject_GetAttr(config, at_num_sms));
    require(sms.o == Py_None || as_int(sms.o) > 0);
  }
  int64_t tiles(int64_t rows, int64_t cols) const { return ((rows + m - 1) / m) * ((cols + n - 1) / n); }
};

struct Types {
  int in, out;
  float scale = 1.f;
  Types(const at::Tensor& a, const at::Tensor& b, const at::Tensor& c, PyObject* scale_a, PyObject* scale_b)
      : in(type_code(a.scalar_type())), out(type_code(c.scalar_type())) {
    require(a.scalar_type() == b.scalar_type());
    if (in == IRIS_HIP_FP8_E4M3) {
      require(out == IRIS_HIP_BF16 || out == IRIS_HIP_FP16);
      double s = 1.0;
      for (PyObject* x : {scale_a, scale_b}) {
        require(x == Py_None || PyFloat_Check(x));
        if (x != Py_None) s *= PyFloat_AS_DOUBLE(x);
      }
      scale = (float)s;
    } else {
      require(in == out && scale_a == Py_None && scale_b == Py_None);
    }
  }
};

int path_code(PyObject* path) {
  if (is_text(path, "auto")) return IRIS_HIP_PATH_AUTO;
  require(is_text(path, "mfma") || is_text(path, "generic"));
  return is_text(path, "mfma") ? IRIS_HIP_PATH_MFMA : IRIS_HIP_PATH_GENERIC;
}
int acc_code(PyObject* rule) {
  require(is_text(rule, "fp32") || is_text(rule, "reference"));
  return is_text(rule, "fp32") ? IRIS_HIP_ACC_FP32 : IRIS_HIP_ACC_REFERENCE;
}

// Whether launches on `stream` are being recorded into a graph.  The null stream, on which most programs run, cannot be
// captured and is not asked about.
bool is_capturing(PyObject* stream) {
  void* const raw = PyLong_AsVoidPtr(stream);
  return raw && fn_stream_capturing(raw) != 0;
}

// Whether a workspace that has been used may be used again by a call on `stream` as it is: the last launch was on the same
// stream, and neither that nor an earlier one, nor this one, is part of a graph.
// (`capturing`: what is_capturing() says of the stream, asked once per call: 0.1 us.)
void require_same_stream(PyObject* ws, const Shmem& shmem, PyObject* stream, bool capturing) {
  const Ref last(PyObject_GetAttr(ws, at_stream));
  require(last.o != Py_None && PyLong_AsUnsignedLongLong(last.o) == PyLong_AsUnsignedLongLong(stream) && !PyErr_Occurred());
  require(Ref(PyObject_GetAttr(ws, at_captured)).o == Py_False && !capturing);
  require(shmem.runs_alone() && *shmem.status() == 0);  // (a status to report is the wrapper's business)
}

// The buffers of a workspace that this very call used before (or, when `prepared` counts, has been prepared for).
struct Workspace {
  void* aux = nullptr;
  int32_t* locks = nullptr;
  bool clear = false;  // reused without a preamble (rearmed() of the Python side states the conditions)
  Workspace(PyObject* ws, const Shmem& shmem, const char* operation, const char* variant, bool prepared_counts, const Matrix& A,
            const Matrix& C, int64_t tiles, PyObject* stream, bool capturing) {
    require(ws != Py_None);
    require(is_text(Ref(PyObject_GetAttr(ws, at_operation)).o, operation) && is_text(Ref(PyObject_GetAttr(ws, at_variant)).o, variant));
    require(int_of(ws, at_world_size) == shmem.world);
    const Ref shape(PyObject_GetAttr(ws, at_shape)), dtype(PyObject_GetAttr(ws, at_dtype));
    require(PyTuple_CheckExact(shape.o) && PyTuple_GET_SIZE(shape.o) == 3 && as_int(PyTuple_GET_ITEM(shape.o, 0)) == C.rows &&
            as_int(PyTuple_GET_ITEM(shape.o, 1)) == C.cols && as_int(PyTuple_GET_ITEM(shape.o, 2)) == A.cols);
    require(THPDtype_Check(dtype.o) && ((THPDtype*)dtype.o)->scalar_type == A.t.scalar_type());
    clear = !(prepared_counts && Ref(PyObject_GetAttr(ws, at_prepared)).o == Py_True);
    if (clear) require_same_stream(ws, shmem, stream, capturing);
    if (strcmp(variant, "atomic") == 0) {
      require(shmem.symmetric(C.t));
      return;
    }
    const Ref a(PyObject_GetAttr(ws, at_aux_buffer)), l(PyObject_GetAttr(ws, at_locks));
    const at::Tensor &ta = tensor(a.o), &tl = tensor(l.o);
    require(ta.scalar_type() == C.t.scalar_type() && tl.scalar_type() == at::kInt && ta.dim() == 2 && ta.size(0) == C.rows && ta.size(1) == C.cols);
    require(clear ? tl.numel() == tiles : tl.numel() >= tiles);
    require((C.rows - 1) * C.s0 + (C.cols - 1) * C.s1 < ta.numel());
    aux = ta.mutable_data_ptr();
    locks = (int32_t*)tl.mutable_data_ptr();
  }
};

// Calls `f`, which must not throw: the interpreter's lock is not held.
template <class F>
PyObject* launch(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// Runs `body`; whatever it declines, or trips over in front of the launch, is the wrapper's.
template <class F>
PyObject* attempt(Py_ssize_t n, Py_ssize_t expected, F&& body) {
  if (n != expected) return PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", expected, n);
  try {
    return body();
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// Notes in the workspace that a launch (whose result is `rc`) has used it; returns rc, or NULL with a Python error set.
PyObject* used(PyObject* rc, PyObject* ws, PyObject* stream, bool capturing, bool unprepare) {
  if (!rc || PyLong_AsLong(rc) != 0) return rc;
  if ((unprepare && PyObject_SetAttr(ws, at_prepared, Py_False) != 0) || PyObject_SetAttr(ws, at_stream, stream) != 0 ||
      (capturing && PyObject_SetAttr(ws, at_captured, Py_True) != 0))
    Py_CLEAR(rc);
  return rc;
}

// try_matmul_all_reduce(shmem, C, A, B, config, workspace, scale_a, scale_b, slot_sum, kernel_path, stream)
PyObject* try_matmul_all_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 11, [&]() -> PyObject* {
    const Shmem shmem(a[0]);
    const Matrix C(a[1], shmem), A(a[2], shmem), B(a[3], shmem);
    require(A.cols == B.rows && C.rows == A.rows && C.cols == B.cols);
    const Types types(A.t, B.t, C.t, a[6], a[7]);
    const Blocks blocks(a[4]);
    blocks.fit(A.rows, B.cols, A.cols);
    Blocks::validate(a[4]);
    const Ref variant(PyObject_GetAttr(a[4], at_all_reduce_variant));
    const char* const name = is_text(variant.o, "one_shot") ? "one_shot" : is_text(variant.o, "two_shot") ? "two_shot" : "atomic";
    require(is_text(variant.o, name));
    const int code = name[0] == 'o' ? IRIS_HIP_VARIANT_ONE_SHOT : name[0] == 't' ? IRIS_HIP_VARIANT_TWO_SHOT : IRIS_HIP_VARIANT_ATOMIC;
    const bool capturing = is_capturing(a[10]);
    const Workspace ws(a[5], shmem, "matmul_all_reduce", name, true, A, C, blocks.tiles(C.rows, C.cols), a[10], capturing);
    const int acc = acc_code(a[8]) | (ws.clear ? IRIS_HIP_CLEAR_C : 0), path = path_code(a[9]);
    const int64_t* const context = shmem.words(at__device_context);
    const long long spin = int_of(a[0], at_spin_limit);
    int32_t* const status = shmem.status();
    void* const stream = PyLong_AsVoidPtr(a[10]);
    PyObject* const rc = launch([&] {
      return fn_iris_hip_matmul_all_reduce(A.ptr(), B.ptr(), C.ptr(), ws.aux, ws.locks, C.rows, C.cols, A.cols, A.s0, A.s1, B.s0, B.s1, C.s0, C.s1,
                                           context, shmem.rank, shmem.world, blocks.m, blocks.n, blocks.k, code, types.in, types.out,
                                           types.scale, acc, spin, status, path, stream);
    });
    return used(rc, a[5], a[10], capturing, true);
  });
}

// try_matmul_reduce_scatter(shmem, C, A, B, config, workspace, all_owners, sum_peers, scale_a, scale_b, slot_sum, kernel_path, stream)
PyObject* try_matmul_reduce_scatter(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 13, [&]() -> PyObject* {
    const Shmem shmem(a[0]);
    const Matrix C(a[1], shmem), A(a[2], shmem), B(a[3], shmem);
    require(A.cols == B.rows && C.rows == A.rows && C.cols == B.cols);
    const Types types(A.t, B.t, C.t, a[8], a[9]);
    const Blocks blocks(a[4]);
    Blocks::validate(a[4]);
    const Ref variant(PyObject_GetAttr(a[4], at_all_reduce_variant));
    require(is_text(variant.o, "two_shot") || is_text(variant.o, "one_shot") || is_text(variant.o, "atomic"));
    const bool capturing = is_capturing(a[12]);
    const Workspace ws(a[5], shmem, "matmul_reduce_scatter", "two_shot", false, A, C, blocks.tiles(C.rows, C.cols), a[12], capturing);
    const int acc = acc_code(a[10]) | IRIS_HIP_CLEAR_C, path = path_code(a[11]);
    const int all_owners = PyObject_IsTrue(a[6]), sum_peers = PyObject_IsTrue(a[7]);
    require(all_owners >= 0 && sum_peers >= 0);
    const int64_t* const context = shmem.words(at__device_context);
    const long long spin = int_of(a[0], at_spin_limit);
    int32_t* const status = shmem.status();
    void* const stream = PyLong_AsVoidPtr(a[12]);
    PyObject* const rc = launch([&] {
      return fn_iris_hip_matmul_reduce_scatter(A.ptr(), B.ptr(), C.ptr(), ws.aux, ws.locks, C.rows, C.cols, A.cols, A.s0, A.s1, B.s0, B.s1, C.s0,
                                               C.s1, context, shmem.rank, shmem.world, blocks.m, blocks.n, blocks.k, all_owners, sum_peers,
                                               types.in, types.out, types.scale, acc, spin, status, path, stream);
    });
    return used(rc, a[5], a[12], capturing, false);
  });
}

struct Bias {
  const void* ptr = nullptr;
  int64_t stride = 1;
  int type = IRIS_HIP_FP32;
  Bias(PyObject* o, const Shmem& shmem, int64_t rows) {
    if (o == Py_None) return;
    const at::Tensor& t = tensor(o);
    shmem.on_device(t);
    require(t.dim() == 1 && t.size(0) == rows);
    ptr = t.const_data_ptr(), stride = t.stride(0), type = type_code(t.scalar_type());
  }
};

// try_all_gather_matmul(shmem, out, A_sharded, B, bias, config, gather_dim, scale_a, scale_b, kernel_path, stream)
PyObject* try_all_gather_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 11, [&]() -> PyObject* {
    const Shmem shmem(a[0]);
    const Matrix C(a[1], shmem), A(a[2], shmem), B(a[3], shmem);
    const long long dim = as_int(a[6]);
    require(dim == 0 || dim == 1);
    const int64_t M = dim == 1 ? A.rows : A.rows * shmem.world;
    require(B.rows == (dim == 1 ? A.cols * shmem.world : A.cols) && C.rows == M && C.cols == B.cols && shmem.symmetric(A.t));
    const Types types(A.t, B.t, C.t, a[7], a[8]);
    const Blocks blocks(a[5]);
    blocks.fit(A.rows, B.cols, A.cols);
    const Bias bias(a[4], shmem, M);
    const int path = path_code(a[9]);
    const int64_t* const context = shmem.words(at__device_context);
    void* const stream = PyLong_AsVoidPtr(a[10]);
    return launch([&] {
      return fn_iris_hip_all_gather_matmul(A.ptr(), B.ptr(), C.ptr(), bias.ptr, M, C.cols, B.rows, A.cols, A.s0, A.s1, B.s0, B.s1, C.s0, C.s1,
                                           bias.stride, context, shmem.rank, shmem.world, blocks.m, blocks.n, blocks.k,
                                           dim == 1 ? IRIS_HIP_GATHER_K : IRIS_HIP_GATHER_M, types.in, types.out, bias.type, types.scale,
                                           path, stream);
    });
  });
}

// try_matmul_all_gather(shmem, out, A, B, bias, config, scale_a, scale_b, kernel_path, stream)
PyObject* try_matmul_all_gather(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 10, [&]() -> PyObject* {
    const Shmem shmem(a[0]);
    const Matrix C(a[1], shmem), A(a[2], shmem), B(a[3], shmem);
    require(A.cols == B.rows && C.rows == A.rows * shmem.world && C.cols == B.cols && shmem.symmetric(C.t));
    const Types types(A.t, B.t, C.t, a[6], a[7]);
    const Blocks blocks(a[5]);
    blocks.fit(A.rows, B.cols, A.cols);
    const Bias bias(a[4], shmem, A.rows);
    const int path = path_code(a[8]);
    const int64_t* const context = shmem.words(at__device_context);
    void* const stream = PyLong_AsVoidPtr(a[9]);
    return launch([&] {
      return fn_iris_hip_matmul_all_gather(A.ptr(), B.ptr(), C.ptr(), bias.ptr, A.rows, C.rows, C.cols, A.cols, A.s0, A.s1, B.s0, B.s1, C.s0, C.s1,
                                           bias.stride, context, shmem.rank, shmem.world, blocks.m, blocks.n, blocks.k, types.in, types.out,
                                           bias.type, types.scale, path, stream);
    });
  });
}

// The collectives of all ranks of the context (group None), op SUM.
struct Collective {
  const Shmem shmem;
  const Matrix out, in;
  const int type, bm, bn, swizzle, sms, xcds, chunk, distribution;
  Collective(PyObject* ctx, PyObject* o, PyObject* i, PyObject* config)
      : shmem(ctx), out(o, shmem), in(i, shmem), type(type_code(in.t.scalar_type())), bm(positive(config, at_block_size_m)),
        bn(positive(config, at_block_size_n)), swizzle(positive(config, at_swizzle_size)), sms(positive(config, at_comm_sms)),
        xcds(positive(config, at_num_xcds)), chunk((int)int_of(config, at_chunk_size)), distribution((int)int_of(config, at_all_reduce_distribution)) {
    require(out.t.scalar_type() == in.t.scalar_type() && out.rows == in.rows && out.cols == in.cols && shmem.symmetric(in.t) &&
            type != IRIS_HIP_FP8_E4M3);
    require(Ref(PyObject_GetAttr(config, at_use_gluon)).o == Py_False);
  }
};

// try_ccl_all_reduce(ctx, output, input, config, workspace, stream)
PyObject* try_ccl_all_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 6, [&]() -> PyObject* {
    const Collective c(a[0], a[1], a[2], a[3]);
    const Ref variant(PyObject_GetAttr(a[3], at_all_reduce_variant));
    const bool one_shot = is_text(variant.o, "one_shot");
    require(one_shot || (is_text(variant.o, "two_shot") && c.shmem.symmetric(c.out.t)));
    PyObject* const ws = a[4];
    require(ws != Py_None && is_text(Ref(PyObject_GetAttr(ws, at_variant)).o, one_shot ? "one_shot" : "two_shot"));
    const Ref shape(PyObject_GetAttr(ws, at_shape)), dtype(PyObject_GetAttr(ws, at_dtype));
    require(PyTuple_CheckExact(shape.o) && PyTuple_GET_SIZE(shape.o) == 2 && as_int(PyTuple_GET_ITEM(shape.o, 0)) == c.in.rows &&
            as_int(PyTuple_GET_ITEM(shape.o, 1)) == c.in.cols);
    require(THPDtype_Check(dtype.o) && ((THPDtype*)dtype.o)->scalar_type == c.in.t.scalar_type());
    const bool capturing = is_capturing(a[5]);
    if (Ref(PyObject_GetAttr(ws, at_prepared)).o != Py_True) require_same_stream(ws, c.shmem, a[5], capturing);
    const int64_t* const bases = c.shmem.words(at_heap_bases);
    void* const stream = PyLong_AsVoidPtr(a[5]);
    PyObject* const rc = launch([&] {
      return fn_iris_hip_all_reduce(c.in.ptr(), c.out.ptr(), c.in.rows, c.in.cols, c.in.s0, c.in.s1, c.out.s0, c.out.s1, bases, c.shmem.rank,
                                    c.shmem.rank, c.shmem.world, 0, 1, c.bm, c.bn, c.swizzle, c.sms, c.xcds, c.chunk,
                                    one_shot ? IRIS_HIP_VARIANT_ONE_SHOT : IRIS_HIP_VARIANT_TWO_SHOT, c.distribution, c.type, stream);
    });
    return used(rc, ws, a[5], capturing, true);
  });
}

// try_ccl_reduce_scatter(ctx, output, input, config, stream)
PyObject* try_ccl_reduce_scatter(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return attempt(n, 5, [&]() -> PyObject* {
    const Collective c(a[0], a[1], a[2], a[3]);
    require(is_text(Ref(PyObject_GetAttr(a[3], at_reduce_scatter_variant)).o, "two_shot"));
    const int64_t* const bases = c.shmem.words(at_heap_bases);
    void* const stream = PyLong_AsVoidPtr(a[4]);
    return launch([&] {
      return fn_iris_hip_reduce_scatter(c.in.ptr(), c.out.ptr(), c.in.rows, c.in.cols, c.in.s0, c.in.s1, c.out.s0, c.out.s1, bases, c.shmem.rank,
                                        c.shmem.rank, c.shmem.world, 0, 1, c.bm, c.bn, c.swizzle, c.sms, c.xcds, c.chunk, c.distribution,
                                        c.type, stream);
    });
  });
}

#define METHOD(name, function) {name, (PyCFunction)(void (*)(void))function, METH_FASTCALL, nullptr},
#define ENTRY_METHOD(name) METHOD(#name, py_##name)
#define TRY_METHOD(name) METHOD(#name, name)
PyMethodDef methods[] = {
    {"load", load, METH_O, "load(path): open libiris_hip.so and resolve its entry points"},
    ENTRY_POINTS(ENTRY_METHOD)
    TRY_METHOD(try_matmul_all_reduce) TRY_METHOD(try_matmul_reduce_scatter) TRY_METHOD(try_all_gather_matmul)
    TRY_METHOD(try_matmul_all_gather) TRY_METHOD(try_ccl_all_reduce) TRY_METHOD(try_ccl_reduce_scatter)
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_definition = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch() {
#define INTERN(name) \
  if (!(at_##name = PyUnicode_InternFromString(#name))) return nullptr;
  ATTRIBUTES(INTERN)
  PyObject* const module = PyModule_Create(&module_definition);
  if (module && PyModule_AddStringConstant(module, "BUILT_FOR", IRIS_LAUNCHER_TAG) != 0) return nullptr;
  return module;
}
