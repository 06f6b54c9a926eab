// Python module `_native`: the host side of the calls a step makes in every layer.
//
// A decode step of a small batch is bound by the host: its kernels take 15-50 us together, and building one call's
// arguments in Python -- a few dozen attribute reads of tensors, the current stream, the workspace, then a ctypes call
// of 20-50 converted arguments -- took 12-20 us per call on the same machine.  Here the checks, the result tensor, the
// workspace look-up and the C-ABI call are one function of the CPython vector-call interface (positional arguments
// only; the Python wrappers in ops.py keep the keyword signatures).
//
// Two groups:
//   * `abi_<entry point>`: the entry point as declared in mi355_decode.h, one Python argument per C argument; a pointer
//     takes a tensor (its data), an integer, None (null) or an object with the buffer protocol (host structs).
//   * the operations (`kv_append`, `decode_step_attention`, ...): tensors in, checks, result tensor out.  A failed check
//     is a ValueError, a tensor that is not on a GPU a RuntimeError, a code of the library a KernelError.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/CachingHostAllocator.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>

#include <chrono>
#include <cmath>
#include <string>
#include <tuple>
#include <type_traits>
#include <unordered_map>
#include <utility>

#include "mi355_decode.h"

namespace {

using at::Tensor;

// Objects of the Python side, set once by setup() and held for the life of the process.
PyObject* g_kernel_error = nullptr;   // exception class of a rejected call
PyObject* g_raw_stream = nullptr;     // device index -> current stream handle
PyObject* g_grow = nullptr;           // (device index, stream, bytes) -> workspace tensor, already stored by set_workspace

struct PyFailure {};  // a Python exception is set

[[noreturn]] void fail_value(const char* msg) {
  PyErr_SetString(PyExc_ValueError, msg);
  throw PyFailure{};
}
#define REQUIRE(cond, msg) \
  do {                     \
    if (!(cond)) fail_value(msg); \
  } while (0)

// ------------------------------------------------------------------------------------------ arguments
const Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s must be a tensor, got %s", name, Py_TYPE(o)->tp_name);
    throw PyFailure{};
  }
  return THPVariable_Unpack(o);
}
const Tensor* opt_tensor(PyObject* o, const char* name) { return o == Py_None ? nullptr : &tensor(o, name); }

int64_t as_int(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailure{};
  return v;
}
double as_float(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFailure{};
  return v;
}
bool as_bool(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyFailure{};
  return v != 0;
}
// Address of a host struct handed over as a buffer (a ctypes structure), null for None.
const void* host_struct(PyObject* o) {
  if (o == Py_None) return nullptr;
  Py_buffer view;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) throw PyFailure{};
  const void* p = view.buf;
  PyBuffer_Release(&view);  // the caller's reference keeps the object alive through the call
  return p;
}

template <typename T>
T convert(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) return nullptr;
    if (THPVariable_Check(o)) return reinterpret_cast<T>(THPVariable_Unpack(o).data_ptr());
    if (PyLong_Check(o)) return reinterpret_cast<T>(PyLong_AsVoidPtr(o));
    return reinterpret_cast<T>(const_cast<void*>(host_struct(o)));
  } else if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(as_float(o));
  } else {
    return static_cast<T>(as_int(o));
  }
}

template <typename F, F fn>
struct Abi;
template <typename R, typename... A, R (*fn)(A...)>
struct Abi<R (*)(A...), fn> {
  template <size_t... I>
  static R call(PyObject* const* a, std::index_sequence<I...>) {
    return fn(convert<A>(a[I])...);
  }
  static PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "this entry point takes %zd arguments, got %zd", (Py_ssize_t)sizeof...(A), n);
      return nullptr;
    }
    try {
      const R r = call(a, std::index_sequence_for<A...>{});
      if (PyErr_Occurred()) return nullptr;
      return PyLong_FromLongLong((long long)r);
    } catch (const PyFailure&) {
      return nullptr;
    } catch (const std::exception& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what());
      return nullptr;
    }
  }
};

void check(int code, const char* what) {
  if (code == 0) return;
  PyErr_Format(g_kernel_error, "%s failed with code %d: %s", what, code, mi_last_error());
  throw PyFailure{};
}

// ------------------------------------------------------------------------------------------ devices, workspaces
void* stream_of(const Tensor& t) {
  if (!t.is_cuda()) {
    PyErr_Format(PyExc_RuntimeError, "the HIP kernels need device tensors, got a tensor on %s; there is no CPU path",
                 t.device().str().c_str());
    throw PyFailure{};
  }
  PyObject* index = PyLong_FromLong(t.device().index());
  PyObject* args[1] = {index};
  PyObject* r = PyObject_Vectorcall(g_raw_stream, args, 1, nullptr);
  Py_DECREF(index);
  if (!r) throw PyFailure{};
  void* s = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  if (PyErr_Occurred()) throw PyFailure{};
  return s;
}

// Scratch per (device, stream): calls on one stream are ordered and share it, another stream has its own.  The
// tensors are allocated and retired by the Python side (`grow`); this map only finds them.  Guarded by the
// interpreter lock, never destroyed (the device runtime may be gone when static destructors run).
struct Key {
  int device;
  void* stream;
  bool operator==(const Key& o) const { return device == o.device && stream == o.stream; }
};
struct KeyHash {
  size_t operator()(const Key& k) const { return std::hash<void*>()(k.stream) * 31 + (size_t)k.device; }
};
auto& pool() {
  static auto* p = new std::unordered_map<Key, Tensor, KeyHash>();
  return *p;
}

struct Scratch {
  void* ptr = nullptr;
  int64_t bytes = 0;
};
// The scratch of a call that needs `need` bytes: the caller's tensor (`given`; the library checks its size), else the
// innermost use_workspace buffer of the thread (`over`), else the pool's.
Scratch scratch(const Tensor& ref, void* stream, int64_t need, PyObject* given, PyObject* over) {
  if (given != Py_None) {
    const Tensor& w = tensor(given, "workspace");
    return {w.data_ptr(), (int64_t)(w.numel() * w.element_size())};
  }
  if (need <= 0) return {};
  if (over != Py_None) {
    const Tensor& w = tensor(over, "workspace");
    REQUIRE(w.device() == ref.device() && w.numel() >= need, "the workspace given to use_workspace is too small");
    return {w.data_ptr(), (int64_t)w.numel()};
  }
  const Key key{ref.device().index(), stream};
  auto it = pool().find(key);
  if (it == pool().end() || it->second.numel() < need) {
    PyObject* r = PyObject_CallFunction(g_grow, "iNL", (int)key.device, PyLong_FromVoidPtr(stream), (long long)need);
    if (!r) throw PyFailure{};
    Py_DECREF(r);
    it = pool().find(key);
    REQUIRE(it != pool().end() && it->second.numel() >= need, "the workspace was not grown");
  }
  return {it->second.data_ptr(), (int64_t)it->second.numel()};
}

// Whether a use_workspace buffer serves a call that can do without it.
bool usable(const Tensor& w, const Tensor& ref, int64_t need, uintptr_t align) {
  return w.device() == ref.device() && w.numel() >= need && (reinterpret_cast<uintptr_t>(w.data_ptr()) & (align - 1)) == 0;
}

// ------------------------------------------------------------------------------------------ shared checks
bool is_16bit(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int dtype_code(const Tensor& t) { return t.scalar_type() == at::kHalf ? MI_DTYPE_FP16 : MI_DTYPE_BF16; }
int dtype_code(const Tensor& t, const char* name) {
  if (!is_16bit(t)) {
    PyErr_Format(PyExc_ValueError, "%s must be bf16 or fp16, got %s", name, c10::toString(t.scalar_type()));
    throw PyFailure{};
  }
  return dtype_code(t);
}
int logits_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return 0;
    case at::kBFloat16: return 1;
    case at::kHalf: return 2;
    default: fail_value("logits must be fp32, bf16 or fp16");
  }
}

// `[T, (1,) H, d]` without touching the tensor: sizes and strides of the three dimensions.
struct Rows3 {
  const Tensor* t = nullptr;
  int64_t n = 0, h = 0, d = 0, sn = 0, sh = 0;
  void* ptr() const { return t ? t->data_ptr() : nullptr; }
};
[[noreturn]] void fail_named(const char* name, const char* what) {
  PyErr_Format(PyExc_ValueError, "%s %s", name, what);
  throw PyFailure{};
}
Rows3 rows3(const Tensor& t, const char* name) {
  Rows3 r;
  r.t = &t;
  const auto size = t.sizes(), stride = t.strides();
  if (size.size() == 4) {
    if (size[1] != 1) fail_named(name, "must be [T, 1, Hq, d] or [T, Hq, d]");
    r.n = size[0]; r.h = size[2]; r.d = size[3]; r.sn = stride[0]; r.sh = stride[2];
    if (stride[3] != 1) fail_named(name, "must be [T, Hq, d] with contiguous d");
  } else {
    if (size.size() != 3 || stride[2] != 1) fail_named(name, "must be [T, Hq, d] with contiguous d");
    r.n = size[0]; r.h = size[1]; r.d = size[2]; r.sn = stride[0]; r.sh = stride[1];
  }
  dtype_code(t, name);
  return r;
}

struct Cache {
  const Tensor* t;
  int64_t n, c, h, d, sc, st, sh;
};
Cache cache_of(const Tensor& t) {
  REQUIRE(t.dim() == 4 && t.stride(3) == 1, "KV cache must be [N, C, Hkv, d] with contiguous d");
  const auto size = t.sizes(), stride = t.strides();
  return {&t, size[0], size[1], size[2], size[3], stride[0], stride[1], stride[2]};
}
bool same_strides(const Cache& a, const Cache& b) { return a.sc == b.sc && a.st == b.st && a.sh == b.sh; }
bool same_shape(const Tensor& a, const Tensor& b) { return a.sizes() == b.sizes(); }

void check_table(const Tensor& table, const Tensor& lens, int64_t R) {
  REQUIRE(table.scalar_type() == at::kInt && table.dim() == 2 && table.stride(1) == 1, "bad block_table");
  REQUIRE(lens.scalar_type() == at::kInt && lens.is_contiguous(), "kv_lens must be contiguous int32");
  REQUIRE(table.size(0) >= R && lens.numel() >= R, "block_table / kv_lens shorter than the batch");
}
bool scales_ok(const Tensor* s, int64_t N, int64_t H) {
  return s && s->scalar_type() == at::kFloat && s->is_contiguous() && s->dim() == 2 && s->size(0) == N && s->size(1) == H;
}
void check_index_row(const Tensor* t, int64_t T, const char* msg) {
  REQUIRE(!t || (t->scalar_type() == at::kLong && t->is_contiguous() && t->numel() >= T), msg);
}
void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// The rotary table `[max_seq, 1, 1, rot]` or `[max_seq, rot]`: fp32 rows of angles.
struct Angles {
  const float* ptr = nullptr;
  int64_t stride = 0;
  int rot = 0;
};
Angles angles_of(const Tensor* e) {
  Angles a;
  if (!e) return a;
  REQUIRE(e->scalar_type() == at::kFloat, "rotary table must be fp32 angles");
  const int64_t dims = e->dim();
  for (int64_t i = 1; i + 1 < dims; ++i) REQUIRE(e->size(i) == 1, "rotary table must be [max_seq, (1, 1,) rot]");
  REQUIRE(dims >= 2 && e->stride(dims - 1) == 1, "rotary table rows must be contiguous");
  a.ptr = static_cast<const float*>(e->data_ptr());
  a.stride = e->stride(0);
  a.rot = (int)e->size(dims - 1);
  return a;
}
void check_norm_weight(const Tensor* w, const Tensor& ref, int64_t d) {
  REQUIRE(!w || (w->scalar_type() == ref.scalar_type() && w->numel() == d && w->is_contiguous()),
          "norm weights must be [d] of the tensors' 16-bit type");
}

float default_scale(int64_t d) { return (float)(1.0 / std::sqrt((double)d)); }

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* same(PyObject* o) {
  Py_INCREF(o);
  return o;
}

// ------------------------------------------------------------------------------------------ operations
// kv_append(key, value|None, k_cache, v_cache|None, token_to_chunk_idx, token_to_local_pos)
PyObject* kv_append(PyObject* const* a) {
  const Tensor& key = tensor(a[0], "key");
  void* stream = stream_of(key);
  const Tensor* value = opt_tensor(a[1], "value");
  const Tensor& kc = tensor(a[2], "k_cache");
  const Tensor* vc = opt_tensor(a[3], "v_cache");
  const Tensor &chunk = tensor(a[4], "token_to_chunk_idx"), &local = tensor(a[5], "token_to_local_pos");
  auto rows = [](const Tensor& x, const char* name) {
    Rows3 r;
    r.t = &x;
    const auto size = x.sizes(), stride = x.strides();
    if (size.size() == 4 && size[1] != 1) fail_named(name, ".size(1) must be 1");
    if (size.size() != 3 && size.size() != 4) fail_named(name, "must be [T, Hkv, d]");
    const size_t k = size.size() - 2;
    r.n = size[0]; r.h = size[k]; r.d = size[k + 1]; r.sn = stride[0]; r.sh = stride[k];
    if (r.h == 1) r.sh = r.d;   // (the stride of a dimension of one says nothing: slices and transposes leave any)
    if (stride[k + 1] != 1 || r.sh != r.d) fail_named(name, "rows must be contiguous");
    return r;
  };
  const Rows3 k3 = rows(key, "key");
  const int64_t row = k3.h * k3.d;
  REQUIRE((value == nullptr) == (vc == nullptr), "value and v_cache go together");
  const Cache kcache = cache_of(kc);
  REQUIRE(key.scalar_type() == kc.scalar_type(), "dtype mismatch between K/V and cache");
  if (value) {
    const Rows3 v3 = rows(*value, "value");
    REQUIRE(v3.h * v3.d == row && v3.n == k3.n && v3.sn == k3.sn, "key/value shapes differ");
    REQUIRE(vc->scalar_type() == key.scalar_type() && value->scalar_type() == key.scalar_type(),
            "dtype mismatch between K/V and cache");
    REQUIRE(same_strides(cache_of(*vc), kcache), "k_cache / v_cache strides differ");
  }
  REQUIRE(kcache.sh == kcache.d && row == kcache.h * kcache.d, "cache rows must be contiguous [Hkv, d]");
  REQUIRE(chunk.scalar_type() == at::kLong && local.scalar_type() == at::kLong, "slot index tensors must be int64");
  REQUIRE(chunk.numel() >= k3.n && local.numel() >= k3.n, "slot index tensors too short");
  REQUIRE(chunk.is_contiguous() && local.is_contiguous(), "slot index tensors must be contiguous");
  check(mi_kv_append(key.data_ptr(), ptr(value), k3.sn, kc.data_ptr(), ptr(vc), kcache.sc, kcache.st,
                     (const int64_t*)chunk.data_ptr(), (const int64_t*)local.data_ptr(), (int)k3.n, (int)row,
                     (int)key.element_size(), stream),
        "mi_kv_append");
  Py_RETURN_NONE;
}

// kv_append_fp8(key, value, k_cache, v_cache, k_scales, v_scales, token_to_chunk_idx, token_to_local_pos, headroom)
PyObject* kv_append_fp8(PyObject* const* a) {
  const Tensor& key = tensor(a[0], "key");
  void* stream = stream_of(key);
  const Tensor &value = tensor(a[1], "value"), &kc = tensor(a[2], "k_cache"), &vc = tensor(a[3], "v_cache");
  const Tensor &ks = tensor(a[4], "k_scales"), &vs = tensor(a[5], "v_scales");
  const Tensor &chunk = tensor(a[6], "token_to_chunk_idx"), &local = tensor(a[7], "token_to_local_pos");
  REQUIRE(is_16bit(key) && value.scalar_type() == key.scalar_type(),
          "K/V must share one 16-bit type and have equal shapes");
  const Rows3 k3 = rows3(key, "key"), v3 = rows3(value, "value");
  REQUIRE(k3.n == v3.n && k3.h == v3.h && k3.d == v3.d, "K/V must share one 16-bit type and have equal shapes");
  REQUIRE(kc.element_size() == 1 && vc.element_size() == 1, "fp8 caches hold one byte per element");
  const Cache kcache = cache_of(kc);
  REQUIRE(same_strides(cache_of(vc), kcache) && kcache.sh == kcache.d && k3.h * k3.d == kcache.h * kcache.sh, "cache layout");
  REQUIRE(ks.scalar_type() == at::kFloat && vs.scalar_type() == at::kFloat, "scales must be fp32");
  REQUIRE(ks.is_contiguous() && vs.is_contiguous(), "scales must be contiguous");
  check_index_row(&chunk, k3.n, "slot rows must be int64 [>=T]");
  check_index_row(&local, k3.n, "slot rows must be int64 [>=T]");
  // (rows are split into the cache's heads; a source whose rows are whole may name its heads differently)
  const bool whole = k3.sh == k3.d && v3.sh == v3.d;
  REQUIRE(whole || (k3.h == kcache.h && k3.d == kcache.d), "key / value rows must be contiguous or have the cache's heads");
  check(mi_kv_append_fp8_strided(key.data_ptr(), k3.sn, whole ? kcache.d : k3.sh, value.data_ptr(), v3.sn, whole ? kcache.d : v3.sh,
                                 kc.data_ptr(), vc.data_ptr(), kcache.sc, kcache.st, (float*)ks.data_ptr(),
                                 (float*)vs.data_ptr(), (const int64_t*)chunk.data_ptr(), (const int64_t*)local.data_ptr(),
                                 (int)k3.n, (int)kcache.c, (int)kcache.h, (int)kcache.d, (float)as_float(a[8]),
                                 dtype_code(key), stream),
        "mi_kv_append_fp8");
  Py_RETURN_NONE;
}

// paged_decode_attention(q, k_cache, v_cache, kv_lens, block_table, softmax_scale|None, max_kv_len|None, split_tokens,
//                        out|None, workspace|None, k_scales|None, v_scales|None, tuning|None, override|None)
PyObject* paged_decode_attention(PyObject* const* a) {
  const Tensor& q = tensor(a[0], "q");
  void* stream = stream_of(q);
  const Tensor &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache"), &lens = tensor(a[3], "kv_lens"), &table = tensor(a[4], "block_table");
  const Rows3 q3 = rows3(q, "q");
  const int64_t R = q3.n;
  REQUIRE(kc.dim() == 4 && kc.size(3) == q3.d && same_shape(kc, vc), "cache shape mismatch");
  const bool fp8 = kc.element_size() == 1;
  REQUIRE(fp8 || kc.scalar_type() == q.scalar_type(), "the KV cache must have the queries' 16-bit type, or be a one-byte fp8 type");
  REQUIRE(vc.scalar_type() == kc.scalar_type(), "k_cache / v_cache dtypes differ");
  const Cache c = cache_of(kc);
  REQUIRE(same_strides(cache_of(vc), c), "k_cache / v_cache strides differ");
  check_table(table, lens, R);
  const Tensor *ks = opt_tensor(a[10], "k_scales"), *vs = opt_tensor(a[11], "v_scales");
  if (fp8) {
    REQUIRE(ks && vs, "fp8 cache needs k_scales and v_scales");
    REQUIRE(scales_ok(ks, c.n, c.h) && scales_ok(vs, c.n, c.h), "scales must be contiguous fp32 [N, Hkv]");
  }
  const int64_t max_len = a[6] == Py_None ? table.size(1) * c.c : as_int(a[6]);
  const float scale = a[5] == Py_None ? default_scale(q3.d) : (float)as_float(a[5]);
  const int split = (int)as_int(a[7]);
  Tensor made;
  if (a[8] == Py_None) made = at::empty_like(q);
  const Tensor& out = a[8] == Py_None ? made : tensor(a[8], "out");
  const Rows3 o3 = rows3(out, "out");
  REQUIRE(o3.n == R && o3.h == q3.h && o3.d == q3.d && out.scalar_type() == q.scalar_type(), "out shape / dtype mismatch");
  const auto* tune = (const MiTuning*)host_struct(a[12]);
  const Scratch ws = scratch(q, stream, mi_decode_workspace_bytes((int)R, (int)q3.h, (int)c.h, (int)q3.d, (int)c.c, (int)max_len, split, tune), a[9], a[13]);
  check(mi_paged_decode_attention(q.data_ptr(), q3.sn, q3.sh, kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh,
                                  (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)lens.data_ptr(),
                                  out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes, (int)R, (int)q3.h, (int)c.h, (int)q3.d,
                                  (int)c.c, (int)max_len, split, scale, fp8 ? MI_KV_FP8_E4M3 : MI_KV_16BIT,
                                  (const float*)ptr(ks), (const float*)ptr(vs), dtype_code(q), tune, stream),
        "mi_paged_decode_attention");
  return a[8] == Py_None ? wrap(made) : same(a[8]);
}

// `shape` of q with the last dimension replaced (a result of another width)
Tensor with_width(const Tensor& q, int64_t width) {
  auto shape = q.sizes().vec();
  shape.back() = width;
  return at::empty(shape, q.options());
}

// paged_mla_decode_attention(q, kv_cache, kv_lens, block_table, softmax_scale, head_dim_v, max_kv_len|None, out|None,
//                            tuning|None, override|None)
PyObject* paged_mla_decode_attention(PyObject* const* a) {
  const Tensor& q = tensor(a[0], "q");
  void* stream = stream_of(q);
  const Tensor &kv = tensor(a[1], "kv_cache"), &lens = tensor(a[2], "kv_lens"), &table = tensor(a[3], "block_table");
  const Rows3 q3 = rows3(q, "q");
  const int64_t R = q3.n, dims = kv.dim();
  REQUIRE(dims != 4 || kv.size(2) == 1, "the latent cache has one row per token");
  REQUIRE((dims == 3 || dims == 4) && kv.stride(dims - 1) == 1 && kv.size(dims - 1) == q3.d && kv.scalar_type() == q.scalar_type(),
          "kv_cache must be [N, C, 576] of the queries' type with contiguous rows");
  REQUIRE(table.scalar_type() == at::kInt && table.dim() == 2 && table.stride(1) == 1, "bad block_table");
  REQUIRE(lens.scalar_type() == at::kInt && lens.is_contiguous() && lens.numel() >= R, "bad kv_lens");
  const int64_t C = kv.size(1), dv = as_int(a[5]);
  const int64_t max_len = a[6] == Py_None ? table.size(1) * C : as_int(a[6]);
  Tensor made;
  if (a[7] == Py_None) made = with_width(q, dv);
  const Tensor& out = a[7] == Py_None ? made : tensor(a[7], "out");
  const Rows3 o3 = rows3(out, "out");
  REQUIRE(o3.n == R && o3.h == q3.h && o3.d == dv, "out shape mismatch");
  const auto* tune = (const MiTuning*)host_struct(a[8]);
  const Scratch ws = scratch(q, stream, mi_mla_decode_workspace_bytes((int)R, (int)q3.h, (int)dv, tune), Py_None, a[9]);
  check(mi_paged_mla_decode_attention(q.data_ptr(), q3.sn, q3.sh, kv.data_ptr(), kv.stride(0), kv.stride(1),
                                      (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)lens.data_ptr(),
                                      out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes, (int)R, (int)q3.h, (int)q3.d, (int)dv,
                                      (int)C, (int)max_len, (float)as_float(a[4]), dtype_code(q), tune, stream),
        "mi_paged_mla_decode_attention");
  return a[7] == Py_None ? wrap(made) : same(a[7]);
}

// paged_prefill_attention(q, k_cache, v_cache, cu_seqlens_q, kv_lens, block_table, softmax_scale|None, max_kv_len|None,
//                         out|None, k_scales|None, v_scales|None, tuning|None, override|None, one_row_requests)
PyObject* paged_prefill_attention(PyObject* const* a) {
  const Tensor& q = tensor(a[0], "q");
  void* stream = stream_of(q);
  const Tensor &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache"), &cu = tensor(a[3], "cu_seqlens_q");
  const Tensor &lens = tensor(a[4], "kv_lens"), &table = tensor(a[5], "block_table");
  const Rows3 q3 = rows3(q, "q");
  REQUIRE(kc.dim() == 4 && kc.size(3) == q3.d && same_shape(kc, vc), "cache shape mismatch");
  const Tensor *ks = opt_tensor(a[9], "k_scales"), *vs = opt_tensor(a[10], "v_scales");
  const Cache c = cache_of(kc);
  if (ks) {
    REQUIRE(kc.element_size() == 1 && vc.element_size() == 1, "fp8 caches hold one byte per element");
    REQUIRE(scales_ok(ks, c.n, c.h) && scales_ok(vs, c.n, c.h), "scales must be contiguous fp32 [N, Hkv]");
  } else {
    REQUIRE(kc.scalar_type() == q.scalar_type() && vc.scalar_type() == q.scalar_type(),
            "the cache must have the queries' 16-bit type, or be bytes with scales");
  }
  REQUIRE(same_strides(cache_of(vc), c), "k_cache / v_cache strides differ");
  REQUIRE(cu.scalar_type() == at::kInt && cu.is_contiguous(), "cu_seqlens_q must be contiguous int32");
  const int64_t R = cu.numel() - 1, T = q3.n;
  check_table(table, lens, R);
  const int64_t max_len = a[7] == Py_None ? table.size(1) * c.c : as_int(a[7]);
  const float scale = a[6] == Py_None ? default_scale(q3.d) : (float)as_float(a[6]);
  Tensor made;
  if (a[8] == Py_None) made = at::empty_like(q);
  const Tensor& out = a[8] == Py_None ? made : tensor(a[8], "out");
  const Rows3 o3 = rows3(out, "out");
  REQUIRE(o3.n == T && o3.h == q3.h && o3.d == q3.d && out.scalar_type() == q.scalar_type(), "out shape / dtype mismatch");
  const auto* tune = (const MiTuning*)host_struct(a[11]);
  const Scratch ws = scratch(q, stream, mi_prefill_workspace_bytes((int)T, (int)R, (int)q3.h, (int)c.h, (int)q3.d, (int)max_len, 0, tune), Py_None, a[12]);
  if (!as_bool(a[13])) {
    check(mi_paged_prefill_attention_tiles(q.data_ptr(), q3.sn, q3.sh, kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh,
                                           ks ? MI_KV_FP8_E4M3 : MI_KV_16BIT, (const float*)ptr(ks), (const float*)ptr(vs),
                                           (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)cu.data_ptr(),
                                           (const int32_t*)lens.data_ptr(), out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes,
                                           (int)T, (int)R, (int)q3.h, (int)c.h, (int)q3.d, (int)c.c, (int)max_len, scale,
                                           dtype_code(q), tune, stream),
          "mi_paged_prefill_attention_tiles");
  } else if (ks) {
    check(mi_paged_prefill_attention_fp8(q.data_ptr(), q3.sn, q3.sh, kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh,
                                         (const float*)ks->data_ptr(), (const float*)vs->data_ptr(),
                                         (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)cu.data_ptr(),
                                         (const int32_t*)lens.data_ptr(), out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes,
                                         (int)T, (int)R, (int)q3.h, (int)c.h, (int)q3.d, (int)c.c, (int)max_len, 0, scale,
                                         dtype_code(q), tune, stream),
          "mi_paged_prefill_attention_fp8");
  } else {
    check(mi_paged_prefill_attention(q.data_ptr(), q3.sn, q3.sh, kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh,
                                     (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)cu.data_ptr(),
                                     (const int32_t*)lens.data_ptr(), out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes,
                                     (int)T, (int)R, (int)q3.h, (int)c.h, (int)q3.d, (int)c.c, (int)max_len, 0, scale,
                                     dtype_code(q), tune, stream),
          "mi_paged_prefill_attention");
  }
  return a[8] == Py_None ? wrap(made) : same(a[8]);
}

// paged_prefill_attention_mla(q, k_cache, v_cache, cu_seqlens_q, kv_lens, block_table, softmax_scale, max_kv_len|None,
//                             out|None, tuning|None, override|None)
PyObject* paged_prefill_attention_mla(PyObject* const* a) {
  const Tensor& q = tensor(a[0], "q");
  void* stream = stream_of(q);
  const Tensor &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache"), &cu = tensor(a[3], "cu_seqlens_q");
  const Tensor &lens = tensor(a[4], "kv_lens"), &table = tensor(a[5], "block_table");
  const Rows3 q3 = rows3(q, "q");
  REQUIRE(kc.dim() == 4 && vc.dim() == 4 && kc.size(0) == vc.size(0) && kc.size(1) == vc.size(1) && kc.size(2) == vc.size(2),
          "key / value caches must be [N, C, H, d] with equal leading dimensions");
  REQUIRE(kc.scalar_type() == q.scalar_type() && vc.scalar_type() == q.scalar_type(), "the caches must have the queries' 16-bit type");
  REQUIRE(kc.size(3) == q3.d, "query and key widths differ");
  const Cache k = cache_of(kc), v = cache_of(vc);
  REQUIRE(cu.scalar_type() == at::kInt && cu.is_contiguous(), "cu_seqlens_q must be contiguous int32");
  const int64_t R = cu.numel() - 1, T = q3.n;
  check_table(table, lens, R);
  Tensor made;
  if (a[8] == Py_None) made = with_width(q, v.d);
  const Tensor& out = a[8] == Py_None ? made : tensor(a[8], "out");
  const Rows3 o3 = rows3(out, "out");
  REQUIRE(o3.n == T && o3.h == q3.h && o3.d == v.d && out.scalar_type() == q.scalar_type(), "out shape / dtype mismatch");
  const int64_t max_len = a[7] == Py_None ? table.size(1) * k.c : as_int(a[7]);
  const auto* tune = (const MiTuning*)host_struct(a[9]);
  const int64_t need = mi_prefill_workspace_bytes((int)T, (int)R, (int)q3.h, (int)k.h, (int)v.d, (int)max_len, 0, tune);
  Scratch ws;  // the split of the keys is optional here: a caller-sized workspace that is too small turns it off
  if (a[10] == Py_None || tensor(a[10], "workspace").numel() >= need) ws = scratch(q, stream, need, Py_None, a[10]);
  check(mi_paged_prefill_attention_mla(q.data_ptr(), q3.sn, q3.sh, kc.data_ptr(), k.sc, k.st, k.sh, vc.data_ptr(), v.sc, v.st, v.sh,
                                       (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)cu.data_ptr(),
                                       (const int32_t*)lens.data_ptr(), out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes, (int)T, (int)R,
                                       (int)q3.h, (int)k.h, (int)q3.d, (int)v.d, (int)k.c, (int)max_len, (float)as_float(a[6]),
                                       dtype_code(q), tune, stream),
        "mi_paged_prefill_attention_mla");
  return a[8] == Py_None ? wrap(made) : same(a[8]);
}

// The slots of a norm / rotary call that writes the cache: strides, and the checks of what names the slot.
struct CacheSlots {
  int64_t sc = 0, st = 0;
  int chunk = 0;
};
CacheSlots slots_of(const Tensor* kc, const Tensor* vc, const Tensor* table, const Tensor* lens, const Tensor& ref, int64_t d,
                    const char* type_msg) {
  CacheSlots s;
  if (!kc) return s;
  REQUIRE(kc->scalar_type() == ref.scalar_type() && vc && vc->scalar_type() == ref.scalar_type(), type_msg);
  const Cache c = cache_of(*kc);
  REQUIRE(same_strides(cache_of(*vc), c) && c.sh == d, "cache layout");
  s.sc = c.sc; s.st = c.st; s.chunk = (int)c.c;
  if (table) {
    REQUIRE(table->scalar_type() == at::kInt && table->stride(1) == 1, "bad block_table");
    REQUIRE(lens && lens->scalar_type() == at::kInt && lens->is_contiguous(), "bad kv_lens");
  }
  return s;
}

// norm_rope_append(query|None, key|None, value|None, q_weight|None, k_weight|None, eps, norm_kind, rotary_emb|None,
//                  q_positions|None, k_positions|None, interleaved, mscale, query_out|None, key_out|None, k_cache|None,
//                  v_cache|None, token_to_chunk_idx|None, token_to_local_pos|None, block_table|None, kv_lens|None,
//                  faithful_rounding, tuning|None)
PyObject* norm_rope_append(PyObject* const* a) {
  const Tensor *query = opt_tensor(a[0], "query"), *key = opt_tensor(a[1], "key"), *value = opt_tensor(a[2], "value");
  REQUIRE(query || key, "need query and/or key");
  const Tensor& ref = query ? *query : *key;
  Rows3 q3, k3, qo, ko, v3;
  const int64_t D = ref.size(-1);
  int64_t T = 0;
  if (query) {
    q3 = rows3(*query, "query");
    REQUIRE(q3.sh == D, "query heads must be contiguous");
    T = q3.n;
  }
  if (key) {
    k3 = rows3(*key, "key");
    REQUIRE(k3.sh == D, "key heads must be contiguous");
    T = k3.n;
    REQUIRE(!query || q3.n == T, "query / key token counts differ");
  }
  qo = q3;
  if (const Tensor* t = opt_tensor(a[12], "query_out")) {
    qo = rows3(*t, "query_out");
    REQUIRE(query && qo.n == q3.n && qo.h == q3.h && qo.d == q3.d && qo.sh == D, "query_out shape");
  }
  if (const Tensor* t = opt_tensor(a[13], "key_out")) {
    ko = rows3(*t, "key_out");
    REQUIRE(key && ko.n == k3.n && ko.h == k3.h && ko.d == k3.d && ko.sh == D, "key_out shape");
  }
  if (value) {
    v3 = rows3(*value, "value");
    REQUIRE(key && v3.n == k3.n && v3.h == k3.h && v3.d == k3.d && v3.sh == D, "value shape");
  }
  const Angles ang = angles_of(opt_tensor(a[7], "rotary_emb"));
  const Tensor *qw = opt_tensor(a[3], "q_weight"), *kw = opt_tensor(a[4], "k_weight");
  check_norm_weight(qw, ref, D);
  check_norm_weight(kw, ref, D);
  const Tensor *qp = opt_tensor(a[8], "q_positions"), *kp = opt_tensor(a[9], "k_positions");
  const Tensor *ci = opt_tensor(a[16], "token_to_chunk_idx"), *lp = opt_tensor(a[17], "token_to_local_pos");
  for (const Tensor* t : {qp, kp, ci, lp}) check_index_row(t, T, "index rows must be int64 [>=T]");
  const Tensor *kc = opt_tensor(a[14], "k_cache"), *vc = opt_tensor(a[15], "v_cache");
  const Tensor *bt = opt_tensor(a[18], "block_table"), *lens = opt_tensor(a[19], "kv_lens");
  const CacheSlots s = slots_of(kc, vc, bt, lens, ref, D, "the caches must have the tensors' 16-bit type");
  for (const Rows3* r : {&q3, &k3, &qo, &ko, &v3})
    REQUIRE(!r->t || r->t->scalar_type() == ref.scalar_type(), "query / key / value / outputs must share one 16-bit type");
  const int code = dtype_code(ref, "query / key");
  const auto* tune = (const MiTuning*)host_struct(a[21]);
  check(mi_norm_rope_append(q3.ptr(), q3.sn, qo.ptr(), qo.sn, k3.ptr(), k3.sn, ko.ptr(), ko.sn, v3.ptr(), v3.sn, ptr(qw), ptr(kw),
                            (float)as_float(a[5]), (int)as_int(a[6]), ang.ptr, ang.stride, ang.rot, as_bool(a[10]),
                            (float)as_float(a[11]), (const int64_t*)ptr(qp), (const int64_t*)ptr(kp), ptr(kc), ptr(vc), s.sc, s.st,
                            (const int64_t*)ptr(ci), (const int64_t*)ptr(lp), (const int32_t*)ptr(bt), bt ? bt->stride(0) : 0,
                            (const int32_t*)ptr(lens), s.chunk, (int)T, (int)q3.h, (int)k3.h, (int)D, as_bool(a[20]), code, tune,
                            stream_of(ref)),
        "mi_norm_rope_append");
  Py_RETURN_NONE;
}

// The QKV projection's output `[T, (1,) (Hq + 2 Hkv) d]` and the head counts that read it.
struct Mixed {
  const Tensor* t;
  int64_t T, W, st, Hq, Hkv, D;
};
Mixed mixed_of(PyObject* o, PyObject* hq, PyObject* hkv, const char* shape3) {
  const Tensor& m = tensor(o, "mixed_qkv");
  REQUIRE(m.is_cuda() && is_16bit(m), "mixed_qkv must be a bf16 or fp16 device tensor");
  Mixed r;
  r.t = &m;
  const int64_t dims = m.dim();
  REQUIRE(dims != 3 || m.size(1) == 1, shape3);
  REQUIRE((dims == 2 || dims == 3) && m.stride(dims - 1) == 1, "mixed_qkv must be [T, W] with contiguous rows");
  r.T = m.size(0); r.W = m.size(dims - 1); r.st = m.stride(0);
  r.Hq = as_int(hq); r.Hkv = as_int(hkv);
  REQUIRE(r.Hq > 0 && r.Hkv > 0 && r.Hq % r.Hkv == 0 && r.W % (r.Hq + 2 * r.Hkv) == 0, "mixed_qkv width / head counts");
  r.D = r.W / (r.Hq + 2 * r.Hkv);
  return r;
}

// qkv_norm_rope_append(mixed_qkv, num_query_heads, num_kv_heads, query_out, key_out|None, q_weight|None, k_weight|None,
//                      eps, norm_kind, rotary_emb|None, q_positions|None, k_positions|None, interleaved, mscale,
//                      k_cache|None, v_cache|None, token_to_chunk_idx|None, token_to_local_pos|None, block_table|None,
//                      kv_lens|None, faithful_rounding, tuning|None)
PyObject* qkv_norm_rope_append(PyObject* const* a) {
  const Mixed m = mixed_of(a[0], a[1], a[2], "mixed_qkv must be [T, 1, W]");
  const Tensor& ref = *m.t;
  const Tensor& query_out = tensor(a[3], "query_out");
  const Rows3 qo = rows3(query_out, "query_out");
  REQUIRE(qo.n == m.T && qo.h == m.Hq && qo.d == m.D && qo.sh == m.D && query_out.scalar_type() == ref.scalar_type(),
          "query_out must be [T, Hq, d] of the projection's type");
  Rows3 ko;
  if (const Tensor* t = opt_tensor(a[4], "key_out")) {
    ko = rows3(*t, "key_out");
    REQUIRE(ko.n == m.T && ko.h == m.Hkv && ko.d == m.D && ko.sh == m.D, "key_out must be [T, Hkv, d]");
  }
  const Tensor *kc = opt_tensor(a[14], "k_cache"), *vc = opt_tensor(a[15], "v_cache");
  REQUIRE(ko.t || kc, "the key needs a destination: key_out and/or the cache");
  const Angles ang = angles_of(opt_tensor(a[9], "rotary_emb"));
  const Tensor *qw = opt_tensor(a[5], "q_weight"), *kw = opt_tensor(a[6], "k_weight");
  check_norm_weight(qw, ref, m.D);
  check_norm_weight(kw, ref, m.D);
  const Tensor *qp = opt_tensor(a[10], "q_positions"), *kp = opt_tensor(a[11], "k_positions");
  const Tensor *ci = opt_tensor(a[16], "token_to_chunk_idx"), *lp = opt_tensor(a[17], "token_to_local_pos");
  for (const Tensor* t : {qp, kp, ci, lp}) check_index_row(t, m.T, "index rows must be int64 [>=T]");
  const Tensor *bt = opt_tensor(a[18], "block_table"), *lens = opt_tensor(a[19], "kv_lens");
  const CacheSlots s = slots_of(kc, vc, bt, lens, ref, m.D, "the caches must have the projection's 16-bit type");
  const auto* tune = (const MiTuning*)host_struct(a[21]);
  check(mi_qkv_norm_rope_append(ref.data_ptr(), m.st, query_out.data_ptr(), qo.sn, ko.ptr(), ko.sn, ptr(qw), ptr(kw),
                                (float)as_float(a[7]), (int)as_int(a[8]), ang.ptr, ang.stride, ang.rot, as_bool(a[12]),
                                (float)as_float(a[13]), (const int64_t*)ptr(qp), (const int64_t*)ptr(kp), ptr(kc), ptr(vc), s.sc,
                                s.st, (const int64_t*)ptr(ci), (const int64_t*)ptr(lp), (const int32_t*)ptr(bt),
                                bt ? bt->stride(0) : 0, (const int32_t*)ptr(lens), s.chunk, (int)m.T, (int)m.Hq, (int)m.Hkv,
                                (int)m.D, as_bool(a[20]), dtype_code(ref), tune, stream_of(ref)),
        "mi_qkv_norm_rope_append");
  Py_RETURN_NONE;
}

// qkv_key_append(mixed_qkv, num_query_heads, num_kv_heads, key_out|None, k_weight|None, eps, norm_kind, rotary_emb|None,
//                q_positions, k_positions, interleaved, mscale, k_cache|None, v_cache|None, token_to_chunk_idx|None,
//                token_to_local_pos|None) -> cos | sin [T, 2, d] of the query positions (None without rotary_emb)
PyObject* qkv_key_append(PyObject* const* a) {
  const Mixed m = mixed_of(a[0], a[1], a[2], "mixed_qkv must be [T, 1, W]");
  const Tensor& ref = *m.t;
  Rows3 ko;
  if (const Tensor* t = opt_tensor(a[3], "key_out")) {
    ko = rows3(*t, "key_out");
    REQUIRE(ko.n == m.T && ko.h == m.Hkv && ko.d == m.D && ko.sh == m.D && t->scalar_type() == ref.scalar_type(), "key_out must be [T, Hkv, d]");
  }
  const Tensor *kc = opt_tensor(a[12], "k_cache"), *vc = opt_tensor(a[13], "v_cache");
  REQUIRE(ko.t || kc, "the key needs a destination: key_out and/or the cache");
  const Angles ang = angles_of(opt_tensor(a[7], "rotary_emb"));
  REQUIRE(!ang.ptr || ang.rot == m.D, "rotary_emb must be as wide as a head");
  const Tensor* kw = opt_tensor(a[4], "k_weight");
  check_norm_weight(kw, ref, m.D);
  const Tensor *qp = opt_tensor(a[8], "q_positions"), *kp = opt_tensor(a[9], "k_positions");
  const Tensor *ci = opt_tensor(a[14], "token_to_chunk_idx"), *lp = opt_tensor(a[15], "token_to_local_pos");
  for (const Tensor* t : {qp, kp, ci, lp}) check_index_row(t, m.T, "index rows must be int64 [>=T]");
  const CacheSlots s = slots_of(kc, vc, nullptr, nullptr, ref, m.D, "the caches must have the projection's 16-bit type");
  REQUIRE(!kc || kc->size(2) == m.Hkv, "cache shape mismatch");
  Tensor angles;
  if (ang.ptr) angles = at::empty({m.T, 2, m.D}, ref.options());
  check(mi_qkv_key_append(ref.data_ptr(), m.st, ko.ptr(), ko.sn, ptr(kw), (float)as_float(a[5]), (int)as_int(a[6]), ang.ptr,
                          ang.stride, as_bool(a[10]), (float)as_float(a[11]), (const int64_t*)ptr(qp), (const int64_t*)ptr(kp),
                          ptr(kc), ptr(vc), s.sc, s.st, (const int64_t*)ptr(ci), (const int64_t*)ptr(lp),
                          ang.ptr ? angles.data_ptr() : nullptr, (int)m.T, (int)m.Hq, (int)m.Hkv, (int)m.D, dtype_code(ref),
                          stream_of(ref)),
        "mi_qkv_key_append");
  return ang.ptr ? wrap(angles) : same(Py_None);
}

// qkv_prefill_attention(mixed_qkv, num_query_heads, num_kv_heads, q_weight|None, eps, norm_kind, cos_sin|None, interleaved,
//                       k_cache, v_cache, cu_seqlens_q, kv_lens, block_table, softmax_scale|None, max_kv_len, k_scales|None,
//                       v_scales|None, override|None) -> [T, 1, Hq, d]
PyObject* qkv_prefill_attention(PyObject* const* a) {
  const Mixed m = mixed_of(a[0], a[1], a[2], "mixed_qkv must be [T, 1, W]");
  const Tensor& ref = *m.t;
  void* stream = stream_of(ref);
  const Tensor &kc = tensor(a[8], "k_cache"), &vc = tensor(a[9], "v_cache"), &cu = tensor(a[10], "cu_seqlens_q");
  const Tensor &lens = tensor(a[11], "kv_lens"), &table = tensor(a[12], "block_table");
  const Tensor *qw = opt_tensor(a[3], "q_weight"), *angles = opt_tensor(a[6], "cos_sin");
  check_norm_weight(qw, ref, m.D);
  REQUIRE(kc.dim() == 4 && kc.size(3) == m.D && kc.size(2) == m.Hkv && same_shape(kc, vc), "cache shape mismatch");
  const Tensor *ks = opt_tensor(a[15], "k_scales"), *vs = opt_tensor(a[16], "v_scales");
  const Cache c = cache_of(kc);
  if (ks) {
    REQUIRE(kc.element_size() == 1 && vc.element_size() == 1, "fp8 caches hold one byte per element");
    REQUIRE(scales_ok(ks, c.n, c.h) && scales_ok(vs, c.n, c.h), "scales must be contiguous fp32 [N, Hkv]");
  } else {
    REQUIRE(kc.scalar_type() == ref.scalar_type() && vc.scalar_type() == ref.scalar_type(), "the cache must have the queries' 16-bit type, or be bytes with scales");
  }
  REQUIRE(same_strides(cache_of(vc), c), "k_cache / v_cache strides differ");
  REQUIRE(cu.scalar_type() == at::kInt && cu.is_contiguous(), "cu_seqlens_q must be contiguous int32");
  REQUIRE(!angles || (angles->scalar_type() == ref.scalar_type() && angles->is_contiguous() && angles->numel() >= m.T * 2 * m.D),
          "cos_sin must be [T, 2, d] of the projection's type");
  const int64_t R = cu.numel() - 1, max_len = as_int(a[14]);
  check_table(table, lens, R);
  Tensor out = at::empty({m.T, 1, m.Hq, m.D}, ref.options());
  const Scratch ws = scratch(ref, stream, mi_prefill_workspace_bytes((int)m.T, (int)R, (int)m.Hq, (int)m.Hkv, (int)m.D, (int)max_len, 0, nullptr), Py_None, a[17]);
  check(mi_qkv_prefill_attention(ref.data_ptr(), m.st, ptr(qw), (float)as_float(a[4]), (int)as_int(a[5]), angles ? angles->data_ptr() : nullptr,
                                 as_bool(a[7]), kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh, ks ? MI_KV_FP8_E4M3 : MI_KV_16BIT,
                                 (const float*)ptr(ks), (const float*)ptr(vs), (const int32_t*)table.data_ptr(), table.stride(0),
                                 (const int32_t*)cu.data_ptr(), (const int32_t*)lens.data_ptr(), out.data_ptr(), m.Hq * m.D, m.D,
                                 ws.ptr, ws.bytes, (int)m.T, (int)R, (int)m.Hq, (int)m.Hkv, (int)m.D, (int)c.c, (int)max_len,
                                 a[13] == Py_None ? default_scale(m.D) : (float)as_float(a[13]), dtype_code(ref), stream),
        "mi_qkv_prefill_attention");
  return wrap(out);
}

// decode_step_attention(query|None, key|None, value|None, mixed_qkv|None, num_query_heads, num_kv_heads, k_cache, v_cache,
//                       kv_lens, block_table, q_weight|None, k_weight|None, eps, norm_kind, rotary_emb|None,
//                       positions|None, interleaved, mscale, softmax_scale|None, max_kv_len|None, split_tokens, out|None,
//                       workspace|None, faithful_rounding, k_scales|None, v_scales|None, headroom, tuning|None, override|None)
//
// `next`: the matrix of the projection that follows at once (the layer's step), or null.
PyObject* decode_step(PyObject* const* a, const Tensor* next) {
  const Tensor &kc = tensor(a[6], "k_cache"), &vc = tensor(a[7], "v_cache"), &lens = tensor(a[8], "kv_lens"), &table = tensor(a[9], "block_table");
  int64_t R, Hq, Hkv, D;
  const uint8_t *qp, *kp, *vp;
  int64_t q_st, q_gst, k_st, k_hst, v_st, v_hst;
  const Tensor* ref;
  bool four_d = false;
  if (a[3] != Py_None) {
    REQUIRE(a[0] == Py_None && a[1] == Py_None && a[2] == Py_None, "give either query / key / value or mixed_qkv");
    const Mixed m = mixed_of(a[3], a[4], a[5], "mixed_qkv must be [R, 1, W]");
    ref = m.t;
    R = m.T; Hq = m.Hq; Hkv = m.Hkv; D = m.D;
    const int64_t G = Hq / Hkv, group = (G + 2) * D;
    qp = (const uint8_t*)ref->data_ptr();
    kp = qp + 2 * G * D;
    vp = qp + 2 * (G + 1) * D;
    q_st = k_st = v_st = m.st;
    q_gst = k_hst = v_hst = group;
    four_d = ref->dim() == 3;
  } else {
    const Tensor &query = tensor(a[0], "query"), &key = tensor(a[1], "key"), &value = tensor(a[2], "value");
    const Rows3 q3 = rows3(query, "query"), k3 = rows3(key, "key"), v3 = rows3(value, "value");
    R = q3.n; Hq = q3.h; D = q3.d; Hkv = k3.h;
    REQUIRE(k3.n == R && k3.d == D && v3.n == R && v3.h == Hkv && v3.d == D && Hkv > 0 && Hq % Hkv == 0,
            "query / key / value shapes");
    REQUIRE(q3.sh == D, "query heads must be contiguous");
    REQUIRE(key.scalar_type() == query.scalar_type() && value.scalar_type() == query.scalar_type(),
            "query / key / value must share one 16-bit type");
    ref = &query;
    qp = (const uint8_t*)query.data_ptr(); kp = (const uint8_t*)key.data_ptr(); vp = (const uint8_t*)value.data_ptr();
    q_st = q3.sn; q_gst = (Hq / Hkv) * D;
    k_st = k3.sn; k_hst = k3.sh; v_st = v3.sn; v_hst = v3.sh;
    four_d = query.dim() == 4;
  }
  void* stream = stream_of(*ref);
  REQUIRE(kc.dim() == 4 && kc.size(3) == D && kc.size(2) == Hkv && same_shape(kc, vc), "cache shape mismatch");
  const Cache c = cache_of(kc);
  const bool fp8 = kc.element_size() == 1;
  const Tensor *ks = opt_tensor(a[24], "k_scales"), *vs = opt_tensor(a[25], "v_scales");
  if (fp8) {
    REQUIRE(vc.element_size() == 1 && ks && vs, "byte caches hold e4m3 values and need k_scales / v_scales");
    REQUIRE(scales_ok(ks, c.n, Hkv) && scales_ok(vs, c.n, Hkv), "scales must be fp32 [n_chunks, Hkv]");
  } else {
    REQUIRE(kc.scalar_type() == ref->scalar_type() && vc.scalar_type() == ref->scalar_type(), "the caches must have the tensors' 16-bit type");
  }
  REQUIRE(same_strides(cache_of(vc), c), "k_cache / v_cache strides differ");
  check_table(table, lens, R);
  const Angles ang = angles_of(opt_tensor(a[14], "rotary_emb"));
  const Tensor* pos = opt_tensor(a[15], "positions");
  check_index_row(pos, R, "positions must be int64 [>= R] (None: kv_lens - 1)");
  const Tensor *qw = opt_tensor(a[10], "q_weight"), *kw = opt_tensor(a[11], "k_weight");
  check_norm_weight(qw, *ref, D);
  check_norm_weight(kw, *ref, D);
  const int64_t max_len = a[19] == Py_None ? table.size(1) * c.c : as_int(a[19]);
  const float scale = a[18] == Py_None ? default_scale(D) : (float)as_float(a[18]);
  const int split = (int)as_int(a[20]);
  Tensor made;
  if (a[21] == Py_None) made = four_d ? at::empty({R, 1, Hq, D}, ref->options()) : at::empty({R, Hq, D}, ref->options());
  const Tensor& out = a[21] == Py_None ? made : tensor(a[21], "out");
  const Rows3 o3 = rows3(out, "out");
  REQUIRE(o3.n == R && o3.h == Hq && o3.d == D && out.scalar_type() == ref->scalar_type(), "out shape / dtype mismatch");
  const auto* tune = (const MiTuning*)host_struct(a[27]);
  const Scratch ws = scratch(*ref, stream, mi_decode_workspace_bytes((int)R, (int)Hq, (int)Hkv, (int)D, (int)c.c, (int)max_len, split, tune), a[22], a[28]);
  const float eps = (float)as_float(a[12]), mscale = (float)as_float(a[17]);
  const int norm = (int)as_int(a[13]), inter = as_bool(a[16]), faithful = as_bool(a[23]);
  if (next) {
    check(mi_decode_step_attention_before_linear(
              qp, q_st, q_gst, kp, k_st, k_hst, vp, v_st, v_hst, ptr(qw), ptr(kw), eps, norm, ang.ptr, ang.stride, ang.rot, inter,
              mscale, (const int64_t*)ptr(pos), kc.data_ptr(), vc.data_ptr(), c.sc, c.st, c.sh, fp8 ? MI_KV_FP8_E4M3 : MI_KV_16BIT,
              fp8 ? (float*)ks->data_ptr() : nullptr, fp8 ? (float*)vs->data_ptr() : nullptr, fp8 ? (float)as_float(a[26]) : 1.f,
              (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)lens.data_ptr(), out.data_ptr(), o3.sn, o3.sh,
              ws.ptr, ws.bytes, (int)R, (int)Hq, (int)Hkv, (int)D, (int)c.c, split, scale, faithful, dtype_code(*ref), tune,
              next->data_ptr(), next->stride(0), (int)next->size(0), (int)next->size(1), stream),
          "mi_decode_step_attention_before_linear");
  } else if (fp8) {
    check(mi_decode_step_attention_fp8(qp, q_st, q_gst, kp, k_st, k_hst, vp, v_st, v_hst, ptr(qw), ptr(kw), eps, norm, ang.ptr,
                                       ang.stride, ang.rot, inter, mscale, (const int64_t*)ptr(pos), kc.data_ptr(), vc.data_ptr(),
                                       c.sc, c.st, c.sh, (float*)ks->data_ptr(), (float*)vs->data_ptr(), (float)as_float(a[26]),
                                       (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)lens.data_ptr(),
                                       out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes, (int)R, (int)Hq, (int)Hkv, (int)D, (int)c.c,
                                       split, scale, faithful, dtype_code(*ref), tune, stream),
          "mi_decode_step_attention_fp8");
  } else {
    check(mi_decode_step_attention(qp, q_st, q_gst, kp, k_st, k_hst, vp, v_st, v_hst, ptr(qw), ptr(kw), eps, norm, ang.ptr,
                                   ang.stride, ang.rot, inter, mscale, (const int64_t*)ptr(pos), kc.data_ptr(), vc.data_ptr(), c.sc,
                                   c.st, c.sh, (const int32_t*)table.data_ptr(), table.stride(0), (const int32_t*)lens.data_ptr(),
                                   out.data_ptr(), o3.sn, o3.sh, ws.ptr, ws.bytes, (int)R, (int)Hq, (int)Hkv, (int)D, (int)c.c,
                                   split, scale, faithful, dtype_code(*ref), tune, stream),
          "mi_decode_step_attention");
  }
  return a[21] == Py_None ? wrap(made) : same(a[21]);
}

PyObject* decode_step_attention(PyObject* const* a) { return decode_step(a, nullptr); }

// linear_decode(x, weight, bias|None, out|None, override|None)
PyObject* linear_decode(PyObject* const* a) {
  const Tensor &x = tensor(a[0], "x"), &w = tensor(a[1], "weight");
  const Tensor* bias = opt_tensor(a[2], "bias");
  REQUIRE(w.dim() == 2 && w.stride(1) == 1, "weight must be [N, K] with contiguous rows");
  const int64_t N = w.size(0), K = w.size(1), dims = x.dim();
  REQUIRE(dims >= 1 && x.size(dims - 1) == K && x.stride(dims - 1) == 1, "x must be [..., K] with a contiguous last dimension");
  REQUIRE(x.scalar_type() == w.scalar_type() && (!bias || bias->scalar_type() == x.scalar_type()), "x, weight and bias share one 16-bit type");
  // the leading dimensions as rows of one stride; a layout that is not one takes a copy
  int64_t T = 1, st = K;
  bool rows = true;
  for (int64_t i = dims - 2; i >= 0; --i) {
    if (x.size(i) != 1) {
      if (T == 1) st = x.stride(i);
      else rows = rows && x.stride(i) == st * T;
    }
    T *= x.size(i);
  }
  Tensor copy;
  if (!rows) {
    copy = x.reshape({T, K});
    st = copy.stride(0);
  }
  const Tensor& x2 = rows ? x : copy;
  Tensor made;
  if (a[3] == Py_None) made = with_width(x, N);
  const Tensor& out = a[3] == Py_None ? made : tensor(a[3], "out");
  int64_t o_st = N;
  if (a[3] != Py_None) {
    const Tensor o2 = out.view({-1, N});
    REQUIRE(o2.size(0) == T && o2.stride(1) == 1, "out must be [..., N] with a contiguous last dimension");
    o_st = T > 1 ? o2.stride(0) : N;
  }
  REQUIRE(!bias || (bias->numel() == N && bias->is_contiguous()), "bias must be a contiguous [N] vector");
  void* stream = stream_of(x);
  const int64_t need = mi_linear_decode_workspace_bytes((int)T, (int)N, (int)K);
  Tensor own;  // (the scratch is for results over an input; a use_workspace buffer sized for attention may lack the room)
  const bool fits = a[4] == Py_None || usable(tensor(a[4], "workspace"), x, need, 16);
  if (!fits) own = at::empty({need}, x.options().dtype(at::kByte));
  const Scratch ws = fits ? scratch(x, stream, need, Py_None, a[4]) : Scratch{own.data_ptr(), need};
  check(mi_linear_decode(x2.data_ptr(), st, w.data_ptr(), w.stride(0), ptr(bias), out.data_ptr(), o_st, ws.ptr, ws.bytes, (int)T,
                         (int)N, (int)K, dtype_code(x, "x"), stream),
        "mi_linear_decode");
  return a[3] == Py_None ? wrap(made) : same(a[3]);
}

// attention_layer_decode(hidden, qkv_weight, qkv_bias|None, proj_weight, proj_bias|None, num_query_heads, num_kv_heads,
//                        k_cache, v_cache, kv_lens, block_table, q_weight|None, k_weight|None, eps, norm_kind,
//                        rotary_emb|None, interleaved, softmax_scale|None, max_kv_len, k_scales|None, v_scales|None,
//                        headroom, tuning|None, override|None): the three calls of a decode step of a layer in a row
PyObject* attention_layer_decode(PyObject* const* a) {
  PyObject* const none = Py_None;
  PyObject* const linear_qkv[5] = {a[0], a[1], a[2], none, a[23]};
  PyObject* mixed = linear_decode(linear_qkv);
  struct Drop {
    PyObject* o;
    ~Drop() { Py_XDECREF(o); }
  };
  Drop d0{mixed}, d1{PyLong_FromLong(0)}, d2{PyFloat_FromDouble(1.0)};
  PyObject* const step[29] = {none, none, none, mixed, a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15],
                              none, a[16], d2.o, a[17], a[18], d1.o, none, none, Py_True, a[19], a[20], a[21], a[22], a[23]};
  // (a matrix that the projection below refuses is its to refuse; with an fp8 cache nothing is read ahead)
  const Tensor *proj = opt_tensor(a[3], "weight"), &cache = tensor(a[7], "k_cache");
  const bool fetchable = proj && cache.element_size() != 1 && proj->dim() == 2 && proj->stride(1) == 1 && is_16bit(*proj) && proj->device() == cache.device() &&
                         proj->size(0) > 0 && proj->size(0) % 16 == 0 && proj->size(1) > 0 && proj->size(1) % 32 == 0 &&
                         proj->stride(0) >= proj->size(1) && proj->stride(0) % 8 == 0 && proj->size(0) < (1 << 30) &&
                         proj->size(1) < (1 << 20) && (reinterpret_cast<uintptr_t>(proj->data_ptr()) & 15) == 0;
  PyObject* attn = decode_step(step, fetchable ? proj : nullptr);
  Drop d3{attn};
  const Tensor& o = THPVariable_Unpack(attn);   // [R, 1, Hq, d], contiguous
  Drop d4{wrap(o.view({o.size(0), 1, o.size(2) * o.size(3)}))};
  PyObject* const linear_proj[5] = {d4.o, a[3], a[4], none, a[23]};
  return linear_decode(linear_proj);
}

// sample_from_logits(logits, top_k, top_p, temperature, uniform|None, vocab_size, termination_id|None,
//                    kv_length_offsets|None, query_lengths|None, output_lengths|None, return_cut,
//                    override|None)
//   -> (samples, mask|None[, cut])
PyObject* sample_from_logits(PyObject* const* a) {
  const Tensor& logits = tensor(a[0], "logits");
  void* stream = stream_of(logits);
  REQUIRE(logits.dim() == 2 && logits.stride(1) == 1, "logits must be [R, V] with contiguous V");
  const int code = logits_code(logits);
  const int64_t R = logits.size(0), V = logits.size(1), top_k = as_int(a[1]);
  const Tensor* uniform = opt_tensor(a[4], "uniform");
  if (top_k != 1) {
    REQUIRE(uniform, "sampling needs one uniform number per row");
    REQUIRE(uniform->scalar_type() == at::kFloat && uniform->is_contiguous() && uniform->numel() >= R && uniform->device() == logits.device(),
            "uniform must be a contiguous fp32 row of at least R numbers");
  }
  const Tensor* lens[3] = {opt_tensor(a[7], "kv_length_offsets"), opt_tensor(a[8], "query_lengths"), opt_tensor(a[9], "output_lengths")};
  const bool masked = a[6] != Py_None;
  if (masked) {
    REQUIRE((!lens[0] && !lens[1] && !lens[2]) || (lens[0] && lens[1] && lens[2]), "the three request length rows go together");
    for (const Tensor* t : lens)
      REQUIRE(!t || (t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() >= R && t->device() == logits.device()),
              "request length rows must be contiguous int32 rows of at least R entries");
  } else {
    REQUIRE(!lens[0] && !lens[1] && !lens[2], "request lengths without a termination id");
  }
  Tensor samples = at::empty({R}, logits.options().dtype(at::kLong)), mask, cut;
  if (masked) mask = at::empty({R}, logits.options().dtype(at::kByte));
  const bool want_cut = as_bool(a[10]);
  if (want_cut) cut = at::empty({R}, logits.options().dtype(at::kFloat));
  const float top_p = (float)as_float(a[2]);
  // (sampling needs no workspace: a use_workspace buffer that does not serve the parts -- too small, on another device, off
  // a 256-byte line -- leaves the rows to one workgroup each)
  const int64_t need = mi_sample_workspace_bytes((int)R, (int)V, (int)top_k, top_p);
  Scratch ws;
  Tensor many;   // (scratch of a large batch belongs to the call, or to the graph that captures it: the stream's own is not for capture)
  if (a[11] == Py_None && R > 128 && need > 0) {
    many = at::empty({need}, logits.options().dtype(at::kByte));
    ws = {many.data_ptr(), need};
  } else if (a[11] == Py_None || usable(tensor(a[11], "workspace"), logits, need, 256)) {
    ws = scratch(logits, stream, need, Py_None, a[11]);
  }
  check(mi_sample_from_logits_ws(logits.data_ptr(), logits.stride(0), code, (int)R, (int)V, (int)top_k, top_p,
                              (float)as_float(a[3]), (const float*)ptr(uniform), (int)as_int(a[5]), (int64_t*)samples.data_ptr(),
                              want_cut ? (float*)cut.data_ptr() : nullptr, (const int32_t*)ptr(lens[0]), (const int32_t*)ptr(lens[1]),
                              (const int32_t*)ptr(lens[2]), masked ? as_int(a[6]) : -1, masked ? (uint8_t*)mask.data_ptr() : nullptr,
                                 ws.ptr, ws.bytes, stream),
        "mi_sample_from_logits");
  PyObject* m = masked ? wrap(mask) : same(Py_None);
  return want_cut ? Py_BuildValue("NNN", wrap(samples), m, wrap(cut)) : Py_BuildValue("NN", wrap(samples), m);
}

// selected_log_probs(logits, token_ids)
PyObject* selected_log_probs(PyObject* const* a) {
  const Tensor &logits = tensor(a[0], "logits"), &ids = tensor(a[1], "token_ids");
  void* stream = stream_of(logits);
  REQUIRE(logits.dim() == 2 && logits.stride(1) == 1, "logits must be [T, V] with contiguous V");
  const int code = logits_code(logits);
  const int64_t T = logits.size(0), V = logits.size(1);
  REQUIRE(ids.scalar_type() == at::kLong && ids.dim() == 1 && ids.numel() == T && ids.is_contiguous() && ids.device() == logits.device(),
          "token_ids must be a contiguous int64 row with one id per row of logits");
  Tensor out = at::empty({T}, logits.options().dtype(at::kFloat));
  check(mi_selected_log_probs(logits.data_ptr(), logits.stride(0), code, (int)T, (int)V, (const int64_t*)ids.data_ptr(),
                              (float*)out.data_ptr(), stream),
        "mi_selected_log_probs");
  return wrap(out);
}

// last_token_gather(rows, request_query_lengths, out|None)
PyObject* last_token_gather(PyObject* const* a) {
  const Tensor &rows = tensor(a[0], "rows"), &lens = tensor(a[1], "request_query_lengths");
  void* stream = stream_of(rows);
  REQUIRE(rows.dim() == 2 && rows.stride(1) == 1, "rows must be [T, E] with contiguous E");
  REQUIRE(rows.element_size() == 2 || rows.element_size() == 4, "rows must have 2- or 4-byte elements");
  REQUIRE(lens.scalar_type() == at::kInt && lens.dim() == 1 && lens.is_contiguous(), "request_query_lengths must be a contiguous int32 row");
  const int64_t R = lens.numel(), E = rows.size(1);
  Tensor made;
  if (a[2] == Py_None) made = at::empty({R, E}, rows.options());
  const Tensor& out = a[2] == Py_None ? made : tensor(a[2], "out");
  REQUIRE(out.scalar_type() == rows.scalar_type() && out.dim() == 2 && out.size(0) == R && out.size(1) == E && out.stride(1) == 1,
          "out must be [R, E]");
  check(mi_last_token_gather(rows.data_ptr(), rows.stride(0), out.data_ptr(), out.stride(0), (const int32_t*)lens.data_ptr(), (int)R,
                             (int)E, (int)rows.element_size(), stream),
        "mi_last_token_gather");
  return a[2] == Py_None ? wrap(made) : same(a[2]);
}

// ------------------------------------------------------------------------------------------ module
template <PyObject* (*fn)(PyObject* const*), int count>
PyObject* op(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != count) {
    PyErr_Format(PyExc_TypeError, "expected %d positional arguments, got %zd", count, n);
    return nullptr;
  }
  try {
    return fn(a);
  } catch (const PyFailure&) {
    return nullptr;
  } catch (const c10::OutOfMemoryError& e) {
    static PyObject* oom = nullptr;  // torch.OutOfMemoryError, as torch's own calls raise it
    if (!oom) {
      PyObject* torch = PyImport_ImportModule("torch");
      oom = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
      Py_XDECREF(torch);
    }
    PyErr_Clear();
    PyErr_SetString(oom ? oom : PyExc_RuntimeError, e.what_without_backtrace());
    return nullptr;
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// layer_views(buffer, layer, pair) -> new views of one layer: `buffer[0, layer]`, `buffer[1, layer]` of a buffer of keys and
// values, or `buffer[layer]`, None.  A decode step of a small batch asks for them in every layer, and indexing from Python
// takes 2-4 us a view, an operation of the dispatcher's 0.5 us: these are made below autograd, which has no business in a
// cache that kernels write (they take any write, and none makes the buffer itself require grad).
PyObject* layer_views(PyObject* const* a) {
  const Tensor& buffer = tensor(a[0], "buffer");
  const int lead = as_bool(a[2]) ? 2 : 1;
  int64_t layer = as_int(a[1]);
  const int64_t layers = buffer.dim() >= lead ? buffer.size(lead - 1) : 0;
  if (layer < -layers || layer >= layers) {
    PyErr_Format(PyExc_IndexError, "layer index %lld is out of range for %lld layers", (long long)layer, (long long)layers);
    throw PyFailure{};
  }
  if (layer < 0) layer += layers;
  const auto size = buffer.sizes().slice(lead), stride = buffer.strides().slice(lead);
  const int64_t at = buffer.storage_offset() + layer * buffer.stride(lead - 1);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor first = buffer.as_strided(size, stride, at);
  if (lead == 1) return Py_BuildValue("NO", wrap(first), Py_None);
  return Py_BuildValue("NN", wrap(first), wrap(buffer.as_strided(size, stride, at + buffer.stride(0))));
}

// watch(tensor, index, value, microseconds): whether element `index` of an int32 row in pinned host memory became
// anything but `value` within the time.  The interpreter lock is free meanwhile.
PyObject* watch(PyObject* const* a) {
  const Tensor& t = tensor(a[0], "row");
  const int64_t index = as_int(a[1]);
  REQUIRE(t.device().is_cpu() && t.scalar_type() == at::kInt && t.is_contiguous() && index >= 0 && index < t.numel(),
          "watch takes an int32 row in host memory");
  const int32_t* word = static_cast<const int32_t*>(t.data_ptr()) + index;
  const int32_t value = (int32_t)as_int(a[2]);
  const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(as_int(a[3]));
  bool changed = false;
  Py_BEGIN_ALLOW_THREADS
  for (;;) {
    for (int i = 0; i < 64 && !changed; ++i) {
      changed = __atomic_load_n(word, __ATOMIC_ACQUIRE) != value;
      if (!changed) __builtin_ia32_pause();
    }
    if (changed || std::chrono::steady_clock::now() > until) break;
  }
  Py_END_ALLOW_THREADS
  return PyBool_FromLong(changed);
}

// written_by_kernel(row, device index): a kernel about to go onto the device's current stream stores into `row`, pinned
// host memory of torch's allocator.  The allocator sees the copies it is told of, not a kernel's stores: noted here, the
// memory of a dropped `row` is handed out again only once the stream has got past this point.  Returns the stream's id.
PyObject* written_by_kernel(PyObject* const* a) {
  const Tensor& t = tensor(a[0], "row");
  const c10::Device device(c10::kCUDA, (c10::DeviceIndex)as_int(a[1]));
  REQUIRE(t.device().is_cpu(), "written_by_kernel takes a row in host memory");
  const c10::Stream stream = c10::impl::VirtualGuardImpl(c10::kCUDA).getStream(device);
  REQUIRE(at::getHostAllocator(c10::kCUDA)->record_event(t.data_ptr(), t.storage().data_ptr().get_context(), stream),
          "written_by_kernel takes a row in torch's pinned memory");
  return PyLong_FromLongLong(stream.id());
}

// as_defined(object, class|None, methods): whether `methods` (pairs of a name and the function its class defines) are what
// the object has: none overridden in a subclass, replaced on the class or on the object.  With a class also whether the
// object is one of exactly that class and, a torch module, has no hooks on its call.  (A decode step of a small batch asks
// this of four objects in every layer: 1.9 us from Python.)
PyObject* as_defined(PyObject* const* a) {
  static PyObject* const hooks[4] = {
      PyUnicode_InternFromString("_forward_hooks"), PyUnicode_InternFromString("_forward_pre_hooks"),
      PyUnicode_InternFromString("_backward_hooks"), PyUnicode_InternFromString("_backward_pre_hooks")};
  PyObject* const kind = (PyObject*)Py_TYPE(a[0]);
  if (a[1] != Py_None && kind != a[1]) Py_RETURN_FALSE;
  PyObject** const slot = _PyObject_GetDictPtr(a[0]);
  PyObject* const own = slot ? *slot : nullptr;
  REQUIRE(own && PyTuple_Check(a[2]), "as_defined takes an object with a dictionary and a tuple of pairs");
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(a[2]); ++i) {
    PyObject* const pair = PyTuple_GET_ITEM(a[2], i);
    REQUIRE(PyTuple_Check(pair) && PyTuple_GET_SIZE(pair) == 2, "as_defined takes pairs of a name and a function");
    const int replaced = PyDict_Contains(own, PyTuple_GET_ITEM(pair, 0));
    if (replaced < 0) throw PyFailure{};
    if (replaced) Py_RETURN_FALSE;
    PyObject* const function = PyObject_GetAttr(kind, PyTuple_GET_ITEM(pair, 0));
    if (!function) throw PyFailure{};
    Py_DECREF(function);  // (the class holds it)
    if (function != PyTuple_GET_ITEM(pair, 1)) Py_RETURN_FALSE;
  }
  if (a[1] != Py_None)
    for (PyObject* const name : hooks) {
      PyObject* const set = PyDict_GetItemWithError(own, name);
      if (!set && PyErr_Occurred()) throw PyFailure{};
      const int any = set ? PyObject_IsTrue(set) : 0;
      if (any < 0) throw PyFailure{};
      if (any) Py_RETURN_FALSE;
    }
  Py_RETURN_TRUE;
}

// setup(kernel_error_class, raw_stream(device index), grow(device index, stream, bytes))
PyObject* setup(PyObject* const* a) {
  for (int i = 0; i < 3; ++i) Py_INCREF(a[i]);
  g_kernel_error = a[0];
  g_raw_stream = a[1];
  g_grow = a[2];
  Py_RETURN_NONE;
}
// set_workspace(device index, stream, tensor) -> the tensor it replaces, or None
PyObject* set_workspace(PyObject* const* a) {
  const Key key{(int)as_int(a[0]), PyLong_AsVoidPtr(a[1])};
  const Tensor& t = tensor(a[2], "workspace");
  auto it = pool().find(key);
  PyObject* old = it == pool().end() ? same(Py_None) : wrap(it->second);
  pool()[key] = t;
  return old;
}

#define ABI(name) {"abi_" #name, (PyCFunction)(void (*)(void))Abi<decltype(&name), &name>::entry, METH_FASTCALL, nullptr}
#define OP(name, count) {#name, (PyCFunction)(void (*)(void))op<name, count>, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ABI(mi_kv_append_decode), ABI(mi_kv_quantize_chunks_fp8), ABI(mi_kv_append_decode_fp8), ABI(mi_decode_workspace_bytes),
    ABI(mi_prefill_workspace_bytes), ABI(mi_paged_decode_attention_noalloc),
    ABI(mi_update_requests), ABI(mi_update_requests_mask8), ABI(mi_update_requests_clearing),
    ABI(mi_add_request), ABI(mi_decode_attention_state), ABI(mi_step_attention_state),
    OP(kv_append, 6), OP(kv_append_fp8, 9), OP(paged_decode_attention, 14), OP(paged_mla_decode_attention, 10),
    OP(paged_prefill_attention, 14), OP(paged_prefill_attention_mla, 11), OP(norm_rope_append, 22), OP(qkv_norm_rope_append, 22), OP(qkv_key_append, 16),
    OP(qkv_prefill_attention, 18), OP(decode_step_attention, 29),
    OP(linear_decode, 5), OP(attention_layer_decode, 24), OP(sample_from_logits, 12), OP(selected_log_probs, 2), OP(last_token_gather, 3), OP(setup, 3),
    OP(set_workspace, 3), OP(layer_views, 3), OP(watch, 4), OP(written_by_kernel, 2), OP(as_defined, 3), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Host side of the per-layer calls.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&kModule); }
