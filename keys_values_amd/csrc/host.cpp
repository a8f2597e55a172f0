// Host path of the package: the Python functions and the cache object call these with tensors, and one call checks the
// arguments, allocates the outputs and the scratch, fills the C ABI's argument blocks (include/kvx.h) and launches.
//
// Why native: a generation loop calls the cache once per layer and token, and the kernels of such a step take 20 to 40 us
// on the device. Written in Python over ctypes (some eighty attribute stores per step, a device context, a stream and
// a workspace lookup per call) the same work took 45 us of host time for a step on a plain store and 85 us for one of the
// weighted policies: the device waited. Measured, one step: 1 sequence, 32 / 8 heads of 128, 4096 slots 44.2 -> 24.3 us;
// 2 sequences, 8 / 2 heads, 808 slots of 8-bit codes, errors weighed in, 77 -> 36 us; a 512-token first chunk 50 -> 22 us.
//
// Error behaviour is that of the Python functions this serves: ValueError for shapes, NotImplementedError for
// unsupported sizes and types, RuntimeError for tensors that are not on the device. Scratch comes from PyTorch's caching
// allocator per call, on the caller's stream, and goes back to it when the call returns: nothing outlives a call, and
// calls from several threads or streams share nothing. Python objects are read with the interpreter lock held; allocation
// and launch run without it (`unlocked`).
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <dlfcn.h>

#include <algorithm>
#include <array>
#include <optional>
#include <string>

#include "../../include/kvx.h"

namespace {

// ---- the C ABI, bound by bind(path) to the library the ctypes side loaded ------------------------------------------

#define KVX_HOST_SYMBOLS(X)                                                                                                 \
  X(kvx_last_error) X(kvx_sdpa_prefill) X(kvx_sdpa_prefill_workspace_bytes) X(kvx_score_sum) X(kvx_sdpa_prefill_weights)     \
  X(kvx_sdpa_prefill_copying) X(kvx_sdpa_prefill_copying_workspace_bytes)                                                    \
  X(kvx_sdpa_decode) X(kvx_sdpa_decode_workspace_bytes) X(kvx_h2o_decode_step) X(kvx_h2o_decode_step_workspace_bytes)        \
  X(kvx_quantize_blocks) X(kvx_dequantize_blocks) X(kvx_dequantize_rows_typed) X(kvx_cache_write) \
  X(kvx_h2o_update_select) X(kvx_h2o_workspace_bytes) X(kvx_rmsnorm_rows) X(kvx_add_rmsnorm_rows) X(kvx_swiglu_rows)         \
  X(kvx_qk_norm_rope)

struct Lib {
#define X(name) decltype(&::name) name = nullptr;
  KVX_HOST_SYMBOLS(X)
#undef X
  decltype(&::kvx_cache_write_first) kvx_cache_write_first = nullptr;  // libraries from before it bind too
  decltype(&::kvx_sdpa_prefill_first) kvx_sdpa_prefill_first = nullptr;  // likewise: the two calls it stands for
  bool bound = false;
} lib;

PyObject* kvx_error = nullptr;      // KvxError of the ctypes module
PyObject* memory_error = nullptr;   // torch.OutOfMemoryError

struct PyRaised {};  // a Python exception is set

template <typename... A>
[[noreturn]] void raise(PyObject* type, const char* fmt, A... args) {
  PyErr_Format(type, fmt, args...);
  throw PyRaised{};
}

void check(int rc) {
  if (rc == KVX_OK) return;
  if (rc == KVX_ERR_INVALID) raise(PyExc_ValueError, "%s", lib.kvx_last_error());
  if (rc == KVX_ERR_UNSUPPORTED) raise(PyExc_NotImplementedError, "%s", lib.kvx_last_error());
  raise(kvx_error, "kvx status %d: %s", rc, lib.kvx_last_error());
}

// f() without the interpreter lock: the allocator may have to free blocks and wait for the device, a launch for room in a
// hardware queue, and what they wait for may need Python (a host function in a stream). f touches no Python object and raises
// no Python error (its status goes to check() afterwards; C++ exceptions pass); tensors it uses are arguments of the call,
// which the caller holds, or held by the call itself.
template <typename F>
auto unlocked(F&& f) {
  struct Release {
    PyThreadState* state = PyEval_SaveThread();
    ~Release() { PyEval_RestoreThread(state); }
  } release;
  return f();
}

std::string shape_str(const at::Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

// ---- arguments ---------------------------------------------------------------------------------------------------

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "%s must be a tensor, not %s", name, Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
const at::Tensor* opt_tensor(PyObject* o, const char* name) { return o == Py_None ? nullptr : &tensor(o, name); }
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyRaised{};
  return v;
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyRaised{};
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyRaised{};
  return v != 0;
}
void require_args(Py_ssize_t n, Py_ssize_t want, const char* who) {
  if (n != want) raise(PyExc_TypeError, "%s takes %zd arguments, got %zd", who, want, n);
}
void require_gpu(const at::Tensor& t) {
  if (!t.is_cuda())
    raise(PyExc_RuntimeError, "keys_values_amd: tensor on %s; the HIP kernels need a ROCm device and there is no CPU fallback", t.device().str().c_str());
}

// Attributes of the cache object that are read per call, as interned names.
#define ATTRS(X)                                                                                                           \
  X(k) X(v) X(k_scale) X(k_zp) X(v_scale) X(v_zp) X(token_pos) X(scores) X(v_norm) X(q_errors) X(_next_flat) X(_next_count) \
  X(batch_size) X(n_query_groups) X(n_head) X(head_size) X(cache_length) X(current_length) X(prefill_length)              \
  X(grace_period) X(normalize_scores) X(combination_constant) X(scale_factor) X(_input_pos) X(_store_dtype) X(_store_quantized)
struct Names {
#define X(n) PyObject* n = nullptr;
  ATTRS(X)
#undef X
} names;

struct Ref {  // an owned reference
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {
    if (!o) throw PyRaised{};
  }
  Ref(const Ref&) = delete;
  Ref(Ref&& o) : p(o.p) { o.p = nullptr; }
  ~Ref() { Py_XDECREF(p); }
};
// int(o): positions and counts may be floats and the like
int64_t converted(PyObject* o) { return PyLong_Check(o) ? integer(o) : integer(Ref(PyNumber_Long(o)).p); }
Ref attr(PyObject* o, PyObject* name) { return Ref(PyObject_GetAttr(o, name)); }
int64_t attr_int(PyObject* o, PyObject* name) { return integer(attr(o, name).p); }
at::Tensor attr_tensor(PyObject* o, PyObject* name) { return tensor(attr(o, name).p, PyUnicode_AsUTF8(name)); }
std::optional<at::Tensor> attr_opt_tensor(PyObject* o, PyObject* name) {
  Ref r = attr(o, name);
  if (r.p == Py_None) return std::nullopt;
  return tensor(r.p, PyUnicode_AsUTF8(name));
}

// The cache's tensors that a call's argument block points into: another thread may give the object new ones meanwhile.
struct Held {
  std::array<at::Tensor, 16> tensors;  // eleven at most
  size_t n = 0;
  const at::Tensor& operator()(at::Tensor t) { return tensors.at(n++) = std::move(t); }
};

// Device and stream of a call: the tensors' device is made current if it is not.
struct Launch {
  c10::DeviceIndex dev;
  std::optional<c10::DeviceGuard> guard;
  void* stream;
  at::TensorOptions options;
  explicit Launch(const at::Tensor& t) : dev(t.device().index()), options(at::TensorOptions().device(t.device())) {
    if (c10::hip::current_device() != dev) guard.emplace(t.device());
    stream = (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev).stream();
  }
  at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const { return at::empty(sizes, options.dtype(type)); }
  at::Tensor scratch(size_t bytes) const { return bytes ? at::empty({(int64_t)bytes}, options.dtype(at::kByte)) : at::Tensor(); }
};
void* data(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

bool served_head_size(int64_t d) { return d == 64 || d == 128 || d == 256; }
int elem_dtype(at::ScalarType t) { return t == at::kHalf ? KVX_KV_F16 : KVX_KV_BF16; }
int quant_dtype(int bits, at::ScalarType t) {
  if (bits == 4) return t == at::kHalf ? KVX_KV_U4_F16 : KVX_KV_U4;
  return t == at::kHalf ? KVX_KV_U8_F16 : KVX_KV_U8;
}

void check_bhtd(const char* name, const at::Tensor& t) {
  if (t.dim() != 4) raise(PyExc_ValueError, "%s must be a 4D tensor, got shape %s", name, shape_str(t).c_str());
  if (t.stride(3) != 1) raise(PyExc_ValueError, "%s: the head dimension must be contiguous (stride %lld)", name, (long long)t.stride(3));
}

std::string dtype_name(at::ScalarType t) {
  const std::string s = c10::toString(t);
  return t == at::kBFloat16 ? "torch.bfloat16" : t == at::kHalf ? "torch.float16" : t == at::kByte ? "torch.uint8" : t == at::kFloat ? "torch.float32" : s;
}

// A QuantState, any object with its attributes, or a bare tuple in its order; keys_only: the state of V is not looked at.
struct Quant {
  at::Tensor ks, kz, vs, vz;
  explicit Quant(PyObject* o, bool keys_only = false) {
    const bool bare = PyTuple_CheckExact(o);
    if (bare && PyTuple_GET_SIZE(o) != 4) raise(PyExc_ValueError, "quant must be a QuantState");
    auto field = [&](int i, PyObject* name) { return bare ? tensor(PyTuple_GET_ITEM(o, i), PyUnicode_AsUTF8(name)) : attr_tensor(o, name); };
    ks = field(0, names.k_scale);
    kz = field(1, names.k_zp);
    vs = keys_only ? ks : field(2, names.v_scale);
    vz = keys_only ? kz : field(3, names.v_zp);
  }
};

void check_dtypes(const at::Tensor& q, const at::Tensor& k, const at::Tensor* v, bool quant) {
  const at::ScalarType qt = q.scalar_type();
  if (qt != at::kBFloat16 && qt != at::kHalf)
    raise(PyExc_NotImplementedError, "query.dtype must be torch.bfloat16 or torch.float16, got %s", dtype_name(qt).c_str());
  const at::ScalarType want = quant ? at::kByte : qt;
  const at::Tensor* ts[2] = {&k, v};
  for (int i = 0; i < 2; ++i)
    if (ts[i] && ts[i]->scalar_type() != want)
      raise(PyExc_NotImplementedError, "%s.dtype must be %s, got %s", i ? "value" : "key", dtype_name(want).c_str(), dtype_name(ts[i]->scalar_type()).c_str());
}

void set_q(kvx_sdpa_args& a, const at::Tensor& t) {
  a.q = t.data_ptr();
  a.q_stride_b = t.stride(0);
  a.q_stride_h = t.stride(1);
  a.q_stride_t = t.stride(2);
}
void set_k(kvx_sdpa_args& a, const at::Tensor& t) {
  a.k = t.data_ptr();
  a.k_stride_b = t.stride(0);
  a.k_stride_h = t.stride(1);
  a.k_stride_t = t.stride(2);
}
void set_v(kvx_sdpa_args& a, const at::Tensor& t) {
  a.v = t.data_ptr();
  a.v_stride_b = t.stride(0);
  a.v_stride_h = t.stride(1);
  a.v_stride_t = t.stride(2);
}

// Sizes, operands and quantiser state of an attention call (checked by the caller up to the state).
kvx_sdpa_args sdpa_args(const at::Tensor& q, const at::Tensor& k, const at::Tensor* v, double scale, int64_t input_pos, const Quant* qs, int64_t num_splits) {
  kvx_sdpa_args a{};
  const int64_t B = q.size(0), D = q.size(3), Hkv = k.size(1), T = k.size(2);
  a.B = (int32_t)B;
  a.Hq = (int32_t)q.size(1);
  a.Hkv = (int32_t)Hkv;
  a.q_len = (int32_t)q.size(2);
  a.kv_len = (int32_t)T;
  a.D = (int32_t)D;
  a.input_pos = (int32_t)input_pos;
  a.sm_scale = (float)scale;
  a.num_splits = (int32_t)num_splits;
  set_q(a, q);
  set_k(a, k);
  if (v) set_v(a, *v);
  if (!qs) {
    a.kv_dtype = elem_dtype(q.scalar_type());
    return a;
  }
  // rows of D bytes: 8-bit codes; rows of D / 2 bytes: the 4-bit store. The rows dequantise to the query's type.
  a.kv_dtype = quant_dtype(k.size(3) * 2 == D ? 4 : 8, q.scalar_type());
  for (const at::Tensor* t : {&qs->ks, &qs->kz, &qs->vs, &qs->vz})
    if (t->dim() != 3 || t->size(0) != B || t->size(1) != Hkv || t->size(2) != T || t->stride(2) != 1 || t->strides() != qs->ks.strides())
      raise(PyExc_ValueError, "quantisation state must be (B, Hkv, T) arrays sharing strides, last axis contiguous");
  if (qs->ks.scalar_type() != at::kFloat || qs->kz.scalar_type() != at::kInt)
    raise(PyExc_ValueError, "quantisation state must be float32 scales and int32 zero points");
  a.k_scale = (const float*)qs->ks.data_ptr();
  a.k_zp = (const int32_t*)qs->kz.data_ptr();
  a.v_scale = (const float*)qs->vs.data_ptr();
  a.v_zp = (const int32_t*)qs->vz.data_ptr();
  a.qs_stride_b = qs->ks.stride(0);
  a.qs_stride_h = qs->ks.stride(1);
  return a;
}

// token_positions as int32 with a contiguous last axis; `keep` holds a converted copy
void set_positions(kvx_sdpa_args& a, const at::Tensor* tp, at::Tensor& keep) {
  if (!tp) return;
  if (tp->dim() != 3 || tp->size(0) != a.B || tp->size(1) != a.Hkv || tp->size(2) != a.kv_len)
    raise(PyExc_ValueError, "token_positions.shape = %s, must be (%d, %d, %d)", shape_str(*tp).c_str(), a.B, a.Hkv, a.kv_len);
  if (tp->scalar_type() == at::kInt && tp->stride(2) == 1) keep = *tp;
  else keep = unlocked([&] {
    at::Tensor t = tp->to(at::kInt);
    return t.stride(2) == 1 ? t : t.contiguous();
  });
  a.token_positions = (const int32_t*)keep.data_ptr();
  a.tp_stride_b = keep.stride(0);
  a.tp_stride_h = keep.stride(1);
}

int64_t row_len(int64_t D, const at::Tensor& key, bool quant) { return quant && key.size(3) * 2 == D ? D / 2 : D; }

void check_kv(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool quant) {
  if (k.sizes() != v.sizes() || k.size(0) != q.size(0) || k.size(3) != row_len(q.size(3), k, quant))
    raise(PyExc_ValueError, "key.shape = %s, value.shape = %s do not fit query %s", shape_str(k).c_str(), shape_str(v).c_str(), shape_str(q).c_str());
}
void check_heads(int64_t Hq, int64_t Hkv) {
  if (Hkv <= 0 || Hq % Hkv != 0)
    raise(PyExc_ValueError, "n_head = %lld must be a positive multiple of n_query_groups = %lld", (long long)Hq, (long long)Hkv);
}
void check_head_size(int64_t D) {
  if (!served_head_size(D)) raise(PyExc_NotImplementedError, "head size %lld not in (64, 128, 256)", (long long)D);
}

void set_o(kvx_sdpa_args& a, const at::Tensor& o, int64_t sb, int64_t sh, int64_t st) {
  a.o = o.data_ptr();
  a.o_stride_b = sb;
  a.o_stride_h = sh;
  a.o_stride_t = st;
}

PyObject* wrap(const at::Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}
PyObject* three(const at::Tensor& x, const at::Tensor& y, const at::Tensor& z) {
  PyObject* r = PyTuple_New(3);
  if (!r) throw PyRaised{};
  PyTuple_SET_ITEM(r, 0, wrap(x));
  PyTuple_SET_ITEM(r, 1, wrap(y));
  PyTuple_SET_ITEM(r, 2, wrap(z));
  return r;
}

// ---- attention ------------------------------------------------------------------------------------------------------

struct AttnOut {
  at::Tensor out, w, lse;
};

// Whether the allocator can hand out `bytes`. Asked when it cannot, it first gives every cached block back and waits for
// the device, and would do so on every call of a program that fills the memory. What it holds but cannot give back are blocks
// in use and the rest of blocks it has split.
bool has_room(const Launch& L, size_t bytes) {
  namespace allocator = c10::hip::HIPCachingAllocator;
  constexpr size_t kAll = 0, kGranule = (size_t)2 << 20;  // CachingAllocator's StatType::AGGREGATE; large blocks are multiples of 2 MiB
  try {
    const auto s = allocator::getDeviceStats(L.dev);
    const size_t reserved = s.reserved_bytes[kAll].current, kept = s.active_bytes[kAll].current + s.inactive_split_bytes[kAll].current;
    if (kept + bytes + kGranule <= reserved) return true;
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return true;  // no queries while recording
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) return true;
    const size_t most = std::min(free + reserved, (size_t)(allocator::getMemoryFraction(L.dev) * (double)total));
    return kept + bytes + kGranule <= most;
  } catch (const c10::Error&) {
    return true;  // an allocator that keeps no such account
  }
}

// prefill attention on checked operands; `copy`: a quantised store may be dequantised into the scratch where that is faster
AttnOut run_prefill(kvx_sdpa_args& a, const Launch& L, at::ScalarType type, bool weights, bool want_lse, bool transposed, bool copy) {
  AttnOut r;
  check(unlocked([&] {
    if (transposed) {
      r.out = L.empty({a.B, a.q_len, a.Hq, a.D}, type);
      set_o(a, r.out, r.out.stride(0), r.out.stride(2), r.out.stride(1));
    } else {
      r.out = L.empty({a.B, a.Hq, a.q_len, a.D}, type);
      set_o(a, r.out, r.out.stride(0), r.out.stride(1), r.out.stride(2));
    }
    if (weights || want_lse) r.lse = L.empty({a.B, a.q_len, a.Hq}, at::kFloat);
    if (weights) r.w = L.empty({a.B, a.Hkv, a.kv_len}, at::kFloat);
    a.lse = (float*)data(r.lse);
    a.w = (float*)data(r.w);
    const size_t least = lib.kvx_sdpa_prefill_workspace_bytes(&a), most = copy ? lib.kvx_sdpa_prefill_copying_workspace_bytes(&a) : least;
    if (most > least) copy = has_room(L, most);  // not more where no copy pays, or where it spares as many partial results
    at::Tensor ws;
    try {
      ws = L.scratch(copy ? most : least);
    } catch (const c10::OutOfMemoryError&) {
      if (!copy) throw;
      copy = false;  // no room for a copy of a quantised store after all: the form that needs none
      ws = L.scratch(least);
    }
    a.workspace = data(ws);
    a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    return (copy ? lib.kvx_sdpa_prefill_copying : weights ? lib.kvx_sdpa_prefill_weights : lib.kvx_sdpa_prefill)(&a, L.stream);
  }));
  return r;
}

// prefill(query, key, value, scale, input_pos, token_positions, return_weights, return_lse, output_transposed, quant,
// num_splits, fused_dequant) -> (out, weights or None, lse or None)
PyObject* prefill(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 12, "prefill");
  const at::Tensor &q = tensor(args[0], "query"), &k = tensor(args[1], "key"), &v = tensor(args[2], "value");
  for (const at::Tensor* t : {&q, &k, &v}) require_gpu(*t);
  check_bhtd("query", q);
  check_bhtd("key", k);
  check_bhtd("value", v);
  std::optional<Quant> qs;
  if (args[9] != Py_None) qs.emplace(args[9]);
  check_dtypes(q, k, &v, qs.has_value());
  check_kv(q, k, v, qs.has_value());
  const int64_t q_len = q.size(2), T = k.size(2);
  if (!(0 < q_len && q_len <= T)) raise(PyExc_ValueError, "Must have 0 < q_len = %lld <= kv_len = %lld", (long long)q_len, (long long)T);
  check_heads(q.size(1), k.size(1));
  check_head_size(q.size(3));
  const Launch L(q);
  kvx_sdpa_args a = sdpa_args(q, k, &v, real(args[3]), converted(args[4]), qs ? &*qs : nullptr, converted(args[10]));
  at::Tensor keep;
  set_positions(a, opt_tensor(args[5], "token_positions"), keep);
  const bool want_lse = truth(args[7]);
  AttnOut r = run_prefill(a, L, q.scalar_type(), truth(args[6]), want_lse, truth(args[8]), qs && !truth(args[11]));
  return three(r.out, r.w, want_lse ? r.lse : at::Tensor());
}

// score_sum(query, key, lse, scale, input_pos, token_positions, quant) -> weights
PyObject* score_sum(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 7, "score_sum");
  const at::Tensor &q = tensor(args[0], "query"), &k = tensor(args[1], "key"), &lse = tensor(args[2], "lse");
  for (const at::Tensor* t : {&q, &k, &lse}) require_gpu(*t);
  check_bhtd("query", q);
  check_bhtd("key", k);
  std::optional<Quant> qs;
  if (args[6] != Py_None) qs.emplace(args[6], true);
  check_dtypes(q, k, nullptr, qs.has_value());
  const int64_t B = q.size(0), Hq = q.size(1), q_len = q.size(2);
  if (lse.dim() != 3 || lse.size(0) != B || lse.size(1) != q_len || lse.size(2) != Hq || lse.scalar_type() != at::kFloat || !lse.is_contiguous())
    raise(PyExc_ValueError, "lse must be contiguous float32 (%lld, %lld, %lld), got %s %s", (long long)B, (long long)q_len, (long long)Hq,
          shape_str(lse).c_str(), dtype_name(lse.scalar_type()).c_str());
  check_head_size(q.size(3));
  const Launch L(q);
  kvx_sdpa_args a = sdpa_args(q, k, nullptr, real(args[3]), converted(args[4]), qs ? &*qs : nullptr, 0);
  at::Tensor keep;
  set_positions(a, opt_tensor(args[5], "token_positions"), keep);
  a.lse = (float*)lse.data_ptr();
  at::Tensor w;
  check(unlocked([&] {
    const at::Tensor ws = L.scratch(lib.kvx_sdpa_prefill_workspace_bytes(&a));  // asked without w: no partials of an attention lie ahead of the sums
    w = L.empty({a.B, a.Hkv, a.kv_len}, at::kFloat);
    a.w = (float*)w.data_ptr();
    a.workspace = data(ws);
    a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    return lib.kvx_score_sum(&a, L.stream);
  }));
  return wrap(w);
}

// decode(query, key, value, scale, return_weights, return_lse, quant, num_splits, scratch_splits) -> (out, weights, lse)
PyObject* decode(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 9, "decode");
  const at::Tensor &q = tensor(args[0], "query"), &k = tensor(args[1], "key"), &v = tensor(args[2], "value");
  for (const at::Tensor* t : {&q, &k, &v}) require_gpu(*t);
  check_bhtd("query", q);
  check_bhtd("key", k);
  check_bhtd("value", v);
  std::optional<Quant> qs;
  if (args[6] != Py_None) qs.emplace(args[6]);
  check_dtypes(q, k, &v, qs.has_value());
  if (q.size(2) != 1) raise(PyExc_ValueError, "decode needs q_len == 1, got %lld", (long long)q.size(2));
  check_kv(q, k, v, qs.has_value());
  check_heads(q.size(1), k.size(1));
  check_head_size(q.size(3));
  const int64_t T = k.size(2);
  const Launch L(q);
  kvx_sdpa_args a = sdpa_args(q, k, &v, real(args[3]), T > 0 ? T - 1 : 0, qs ? &*qs : nullptr, converted(args[7]));
  if (const at::Tensor* s = opt_tensor(args[8], "scratch_splits")) {
    if (s->scalar_type() != at::kInt || s->numel() != 1 || s->device() != q.device())
      raise(PyExc_ValueError, "scratch_splits must be a one-element int32 tensor on the query's device");
    a.decode_scratch_splits = (uint32_t*)s->data_ptr();
  }
  const bool want_w = truth(args[4]), want_lse = truth(args[5]);
  AttnOut r;
  check(unlocked([&] {
    r.out = L.empty({a.B, a.Hq, a.D}, q.scalar_type());
    if (want_w) r.w = L.empty({a.B, a.Hkv, a.kv_len}, at::kFloat);
    if (want_lse) r.lse = L.empty({a.B, 1, a.Hq}, at::kFloat);
    set_o(a, r.out, (int64_t)a.Hq * a.D, a.D, a.D);
    a.w = (float*)data(r.w);
    a.lse = (float*)data(r.lse);
    const at::Tensor ws = L.scratch(lib.kvx_sdpa_decode_workspace_bytes(&a));
    a.workspace = data(ws);
    a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    return lib.kvx_sdpa_decode(&a, L.stream);
  }));
  return three(r.out, r.w, r.lse);
}

// ---- the cache object --------------------------------------------------------------------------------------------------

// check_qkv(query, key, value, n_head, n_query_groups, head_size) -> (batch, number of new tokens)
PyObject* check_qkv(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 6, "check_qkv");
  const at::Tensor &q = tensor(args[0], "query"), &k = tensor(args[1], "key"), &v = tensor(args[2], "value");
  for (const at::Tensor* t : {&q, &k, &v}) require_gpu(*t);
  if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes()) raise(PyExc_ValueError, "query, key, value must be 4D and key.shape == value.shape");
  const int64_t b = q.size(0), num = q.size(2), hq = integer(args[3]), hkv = integer(args[4]), d = integer(args[5]);
  if (k.size(0) != b || k.size(1) != hkv || k.size(2) != num || k.size(3) != d || q.size(1) != hq || q.size(3) != d)
    raise(PyExc_ValueError, "shapes %s, %s do not fit the cache", shape_str(q).c_str(), shape_str(k).c_str());
  return Py_BuildValue("LL", (long long)b, (long long)num);
}

void set_cache_tensors(kvx_cache_write_args& a, PyObject* cache, Held& held) {
  const at::Tensor &k = held(attr_tensor(cache, names.k)), &v = held(attr_tensor(cache, names.v));
  a.k_cache = k.data_ptr();
  a.kc_stride_b = k.stride(0);
  a.kc_stride_h = k.stride(1);
  a.kc_stride_t = k.stride(2);
  a.v_cache = v.data_ptr();
  a.vc_stride_b = v.stride(0);
  a.vc_stride_h = v.stride(1);
  a.vc_stride_t = v.stride(2);
  a.kv_dtype = (int32_t)attr_int(cache, names._store_dtype);
  const bool codes = truth(attr(cache, names._store_quantized).p);
  if (codes) {
    const at::Tensor& ks = held(attr_tensor(cache, names.k_scale));
    a.k_scale = (float*)ks.data_ptr();
    a.k_zp = (int32_t*)held(attr_tensor(cache, names.k_zp)).data_ptr();
    a.v_scale = (float*)held(attr_tensor(cache, names.v_scale)).data_ptr();
    a.v_zp = (int32_t*)held(attr_tensor(cache, names.v_zp)).data_ptr();
    a.qs_stride_b = ks.stride(0);
    a.qs_stride_h = ks.stride(1);
  }
  const at::Tensor &tp = held(attr_tensor(cache, names.token_pos)), &sc = held(attr_tensor(cache, names.scores));
  a.token_pos = (int32_t*)tp.data_ptr();
  a.tp_stride_b = tp.stride(0);
  a.tp_stride_h = tp.stride(1);
  a.scores = (float*)sc.data_ptr();
  a.sc_stride_b = sc.stride(0);
  a.sc_stride_h = sc.stride(1);
  if (auto t = attr_opt_tensor(cache, names.v_norm)) a.v_norm = (float*)held(*t).data_ptr();
  // a working buffer whose codes live elsewhere (blocks over the heads): the row-quantising write has no errors to give
  if (codes)
    if (auto t = attr_opt_tensor(cache, names.q_errors)) a.q_errors = (float*)held(*t).data_ptr();
}

// `t` as rows of `type`; `strided`: set where the head dimension is not contiguous in that type and a copy makes it so
at::Tensor rows_of(const at::Tensor& t, at::ScalarType type, bool& strided) {
  if (t.scalar_type() == type && t.stride(3) == 1) return t;
  return unlocked([&] {
    at::Tensor r = t.to(type);
    if (r.stride(3) == 1) return r;
    strided = true;
    return r.contiguous();
  });
}

struct WriteCall {
  kvx_cache_write_args a{};
  at::Tensor key, value;  // as handed to the kernel
  bool strided = false;   // copies of rows that lie strided
  Held held;
};
// key / value (B, Hkv, num, D) into the slots `index` (int32, strides for batch and head; NULL: the slots chosen last)
WriteCall write_args(PyObject* cache, const at::Tensor* index, const at::Tensor& key, const at::Tensor& value, int64_t input_pos, PyObject* ring, PyObject* log) {
  WriteCall w;
  kvx_cache_write_args& a = w.a;
  set_cache_tensors(a, cache, w.held);
  const at::ScalarType type =
      (a.kv_dtype == KVX_KV_F16 || a.kv_dtype == KVX_KV_U8_F16 || a.kv_dtype == KVX_KV_U4_F16) ? at::kHalf : at::kBFloat16;
  w.key = rows_of(key, type, w.strided);
  w.value = rows_of(value, type, w.strided);
  a.B = (int32_t)key.size(0);
  a.Hkv = (int32_t)key.size(1);
  a.num = (int32_t)key.size(2);
  a.D = (int32_t)key.size(3);
  a.cache_len = (int32_t)attr_int(cache, names.cache_length);
  a.input_pos = (int32_t)input_pos;
  if (index) {
    a.index = (const int32_t*)index->data_ptr();
    a.index_stride_b = index->stride(0);
    a.index_stride_h = index->stride(1);
  } else {
    const int64_t c = attr_int(cache, names._next_count);
    a.index = (const int32_t*)w.held(attr_tensor(cache, names._next_flat)).data_ptr();
    a.index_stride_b = a.Hkv * c;
    a.index_stride_h = c;
  }
  a.key = w.key.data_ptr();
  a.key_stride_b = w.key.stride(0);
  a.key_stride_h = w.key.stride(1);
  a.key_stride_t = w.key.stride(2);
  a.value = w.value.data_ptr();
  a.value_stride_b = w.value.stride(0);
  a.value_stride_h = w.value.stride(1);
  a.value_stride_t = w.value.stride(2);
  if (ring != Py_None) {
    const at::Tensor& r = tensor(ring, "ring");
    a.grace_num = (int32_t)r.numel();
    a.grace_period = (int32_t)attr_int(cache, names.grace_period);
    a.grace_slots = (const int32_t*)r.data_ptr();
  }
  if (log != Py_None) {  // (arena, blocksize, position of the first token)
    if (!PyTuple_Check(log) || PyTuple_GET_SIZE(log) != 3) raise(PyExc_TypeError, "log must be (arena, blocksize, position)");
    const at::Tensor& arena = tensor(PyTuple_GET_ITEM(log, 0), "arena");
    a.replay_log = (uint32_t*)arena.data_ptr();
    a.log_blocksize = (int32_t)integer(PyTuple_GET_ITEM(log, 1));
    a.log_pos = integer(PyTuple_GET_ITEM(log, 2));
    a.log_stride_block = arena.stride(0);
    a.log_stride_b = arena.stride(1);
    a.log_stride_h = arena.stride(2);
  }
  return w;
}

// cache_write(cache, index or None, key, value, input_pos, ring or None, log or None)
PyObject* cache_write(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 7, "cache_write");
  const at::Tensor &key = tensor(args[2], "key"), &value = tensor(args[3], "value");
  const Launch L(key);
  const WriteCall w = write_args(args[0], opt_tensor(args[1], "index"), key, value, integer(args[4]), args[5], args[6]);
  check(unlocked([&] { return lib.kvx_cache_write(&w.a, L.stream); }));
  Py_RETURN_NONE;
}

// cache_write_first(cache, index, key, value): the first chunk of a sequence; the other slots' scores, norms and errors become zero
PyObject* cache_write_first(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 4, "cache_write_first");
  if (!lib.kvx_cache_write_first) raise(PyExc_ImportError, "the bound library does not export kvx_cache_write_first");
  const at::Tensor &key = tensor(args[2], "key"), &value = tensor(args[3], "value");
  const Launch L(key);
  const WriteCall w = write_args(args[0], opt_tensor(args[1], "index"), key, value, 0, Py_None, Py_None);
  check(unlocked([&] { return lib.kvx_cache_write_first(&w.a, L.stream); }));
  Py_RETURN_NONE;
}

// prefill_first(cache, index, query, key, value, scale) -> out (B, num, Hq, D): the first chunk of a sequence into its slots, as cache_write_first, and its causal attention
PyObject* prefill_first(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 6, "prefill_first");
  const at::Tensor &q = tensor(args[2], "query"), &key = tensor(args[3], "key"), &value = tensor(args[4], "value");
  const Launch L(q);
  const WriteCall w = write_args(args[0], opt_tensor(args[1], "index"), key, value, 0, Py_None, Py_None);
  const bool fills = w.a.num == w.a.cache_len;  // no slots behind the chunk: an ordinary write
  if (!fills && !lib.kvx_cache_write_first) raise(PyExc_ImportError, "the bound library does not export kvx_cache_write_first");
  for (const at::Tensor* t : {&q, &w.key, &w.value}) require_gpu(*t);
  check_bhtd("query", q);
  if (w.strided) raise(PyExc_ValueError, "key, value: the head dimension must be contiguous");  // as for any attention over the caller's rows
  check_dtypes(q, w.key, &w.value, false);
  check_kv(q, w.key, w.value, false);
  check_heads(q.size(1), key.size(1));
  check_head_size(q.size(3));
  kvx_sdpa_args a = sdpa_args(q, w.key, &w.value, real(args[5]), 0, nullptr, 0);
  at::Tensor out;
  check(unlocked([&] {
    out = L.empty({a.B, a.q_len, a.Hq, a.D}, q.scalar_type());
    set_o(a, out, out.stride(0), out.stride(2), out.stride(1));
    const at::Tensor ws = L.scratch(lib.kvx_sdpa_prefill_workspace_bytes(&a));
    a.workspace = data(ws);
    a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    if (lib.kvx_sdpa_prefill_first) return lib.kvx_sdpa_prefill_first(&a, &w.a, L.stream);
    const int rc = (fills ? lib.kvx_cache_write : lib.kvx_cache_write_first)(&w.a, L.stream);
    return rc ? rc : lib.kvx_sdpa_prefill(&a, L.stream);
  }));
  return wrap(out);
}

// Arguments of the score update and the choice of k slots; `full`: the cache has no free slot (else nothing is chosen
// that anyone uses, and the smallest selection is run)
kvx_h2o_args h2o_args(PyObject* cache, bool full, int64_t k, int64_t input_pos, Held& held) {
  kvx_h2o_args a{};
  a.B = (int32_t)attr_int(cache, names.batch_size);
  a.Hkv = (int32_t)attr_int(cache, names.n_query_groups);
  a.kv_len = (int32_t)attr_int(cache, names.current_length);
  a.limit = full ? (int32_t)(attr_int(cache, names.cache_length) - attr_int(cache, names.grace_period)) : a.kv_len;
  a.k = full ? (int32_t)k : 1;
  a.normalize = full && truth(attr(cache, names.normalize_scores).p);
  a.input_pos = (int32_t)input_pos;
  a.prefill_len = (int32_t)attr_int(cache, names.prefill_length);
  const at::Tensor &sc = held(attr_tensor(cache, names.scores)), &tp = held(attr_tensor(cache, names.token_pos));
  a.scores = (float*)sc.data_ptr();
  a.sc_stride_b = sc.stride(0);
  a.sc_stride_h = sc.stride(1);
  a.token_pos = (const int32_t*)tp.data_ptr();
  a.tp_stride_b = tp.stride(0);
  a.tp_stride_h = tp.stride(1);
  if (auto t = attr_opt_tensor(cache, names.v_norm)) a.v_norm = (const float*)held(*t).data_ptr();
  if (full)  // only the selection reads the errors
    if (auto t = attr_opt_tensor(cache, names.q_errors)) a.q_errors = (const float*)held(*t).data_ptr();
  a.combination = real(attr(cache, names.combination_constant).p);
  return a;
}

// background: the choice runs beside the caller's other work and nobody waits for it. Then one workgroup per row is the
// better form, which is what a workspace without room for sorted lists selects: spread over the device the choice is
// over sooner but holds up the matrix products beside it (two layers of the long-context stack, 4096 slots: 5.60 ms
// against 5.88).
int run_update(kvx_h2o_args& a, const Launch& L, bool background) {
  size_t bytes = lib.kvx_h2o_workspace_bytes(&a);
  if (background) bytes = std::min(bytes, (size_t)a.B * a.Hkv * (8 + 16) + 32);  // a bound and four statistics per row
  const at::Tensor ws = L.scratch(bytes);
  a.workspace = data(ws);
  a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
  return lib.kvx_h2o_update_select(&a, L.stream);
}

// cache_update(cache, weights or None, query_length, k, full, background): scores += weights, then the next k slots into
// the cache's own buffer, on the current stream
PyObject* cache_update(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 6, "cache_update");
  PyObject* cache = args[0];
  const bool full = truth(args[4]);
  Held held;
  kvx_h2o_args a = h2o_args(cache, full, integer(args[3]), attr_int(cache, names._input_pos), held);
  const Launch L(held.tensors[0]);
  const at::Tensor* given = opt_tensor(args[1], "attn_weights");
  a.q_len = (int32_t)integer(args[2]);
  const bool background = truth(args[5]);
  at::Tensor next, w;
  if (full) next = attr_tensor(cache, names._next_flat);
  check(unlocked([&] {
    if (given) w = given->contiguous();
    if (!full) next = L.empty({(int64_t)a.B * a.Hkv}, at::kInt);
    a.w = (const float*)data(w);
    a.next_index = (int32_t*)next.data_ptr();
    return run_update(a, L, background);
  }));
  Py_RETURN_NONE;
}

// cache_decode_step(cache, query, key, value, index or None, input_pos, ring or None, log or None) -> output
// (B, 1, Hq * D): one new token into a full cache: slot write, attention over all slots, score update and the choice of
// the next slot.
PyObject* cache_decode_step(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 8, "cache_decode_step");
  PyObject* cache = args[0];
  const at::Tensor &q = tensor(args[1], "query"), &key = tensor(args[2], "key"), &value = tensor(args[3], "value");
  check_bhtd("query", q);
  const int64_t input_pos = integer(args[5]);
  const Launch L(q);
  const WriteCall w = write_args(cache, opt_tensor(args[4], "index"), key, value, input_pos, args[6], args[7]);
  const kvx_cache_write_args& c = w.a;
  kvx_sdpa_args a{};
  a.B = c.B;
  a.Hq = (int32_t)q.size(1);
  a.Hkv = c.Hkv;
  a.q_len = 1;
  a.kv_len = c.cache_len;
  a.D = c.D;
  a.input_pos = c.cache_len - 1;  // the new token is the newest: it sees every slot
  a.kv_dtype = c.kv_dtype;
  a.sm_scale = (float)real(attr(cache, names.scale_factor).p);
  const bool f16 = c.kv_dtype == KVX_KV_F16 || c.kv_dtype == KVX_KV_U8_F16 || c.kv_dtype == KVX_KV_U4_F16;
  if (q.scalar_type() != (f16 ? at::kHalf : at::kBFloat16))
    raise(PyExc_NotImplementedError, "query.dtype must be %s, got %s", f16 ? "torch.float16" : "torch.bfloat16", dtype_name(q.scalar_type()).c_str());
  set_q(a, q);
  a.k = c.k_cache;
  a.k_stride_b = c.kc_stride_b;
  a.k_stride_h = c.kc_stride_h;
  a.k_stride_t = c.kc_stride_t;
  a.v = c.v_cache;
  a.v_stride_b = c.vc_stride_b;
  a.v_stride_h = c.vc_stride_h;
  a.v_stride_t = c.vc_stride_t;
  a.k_scale = c.k_scale;
  a.k_zp = c.k_zp;
  a.v_scale = c.v_scale;
  a.v_zp = c.v_zp;
  a.qs_stride_b = c.qs_stride_b;
  a.qs_stride_h = c.qs_stride_h;
  Held held;
  kvx_h2o_args h = h2o_args(cache, true, 1, input_pos + 1, held);
  h.q_len = 1;
  h.next_index = (int32_t*)held(attr_tensor(cache, names._next_flat)).data_ptr();
  at::Tensor out;
  check(unlocked([&] {
    out = L.empty({a.B, 1, (int64_t)a.Hq * a.D}, q.scalar_type());
    set_o(a, out, (int64_t)a.Hq * a.D, a.D, a.D);
    const at::Tensor ws = L.scratch(lib.kvx_h2o_decode_step_workspace_bytes(&a, &h));
    a.workspace = data(ws);
    a.workspace_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    return lib.kvx_h2o_decode_step(&c, &a, &h, L.stream);
  }));
  return wrap(out);
}

// ---- quantiser --------------------------------------------------------------------------------------------------------------

// x, or a copy of it that the block kernels can address: rows 16-byte aligned, strides multiples of 8 and, for one block
// per row, the (batch, head) axes collapsible into one
at::Tensor block_view(const at::Tensor& x, bool over_heads) {
  bool ok = x.stride(3) == 1 && (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0;
  for (int i = 0; i < 3; ++i) ok = ok && x.stride(i) % 8 == 0;
  if (!over_heads && x.size(0) > 1) ok = ok && x.stride(0) == x.size(1) * x.stride(1);
  return ok ? x : unlocked([&] { return x.contiguous(); });
}

// quantize_blocks(x, start, codes, scales, zero_points, over_heads, bits) and dequantize_blocks: x (B, Hkv, num, D) of
// the source type, a block per row or, over_heads, per token over all heads; slots start .. of the buffers (first, L,
// final), (first, L), (first, L)
PyObject* blocks_call(PyObject* const* args, Py_ssize_t n, bool quantize) {
  require_args(n, 7, "quantize_blocks");
  const at::Tensor &given = tensor(args[0], "x"), &codes = tensor(args[2], "codes"), &scale = tensor(args[3], "scales"), &zp = tensor(args[4], "zero_points");
  const int64_t start = integer(args[1]);
  const bool over_heads = truth(args[5]);
  require_gpu(given);
  const Launch L(codes);
  const at::Tensor x = quantize ? block_view(given, over_heads) : given;  // dequantised rows: always contiguous
  kvx_block_quant_args a{};
  const int64_t b = x.size(0), hkv = x.size(1), num = x.size(2), d = x.size(3);
  a.x = x.data_ptr();
  if (over_heads) {
    a.n_outer = (int32_t)b;
    a.n_inner = (int32_t)num;
    a.nseg = (int32_t)hkv;
    a.x_stride_outer = x.stride(0);
    a.x_stride_inner = x.stride(2);
    a.x_stride_seg = x.stride(1);
  } else {
    a.n_outer = (int32_t)(b * hkv);
    a.n_inner = (int32_t)num;
    a.nseg = 1;
    a.x_stride_outer = x.stride(1);
    a.x_stride_inner = x.stride(2);
  }
  a.D = (int32_t)d;
  a.bits = (int32_t)integer(args[6]);
  a.elem_dtype = elem_dtype(x.scalar_type());
  a.codes = (uint8_t*)codes.data_ptr() + start * codes.stride(1);
  a.codes_stride_outer = codes.stride(0);
  a.scale = (float*)scale.data_ptr() + start;
  a.zp = (int32_t*)zp.data_ptr() + start;
  a.state_stride_outer = scale.stride(0);
  check(unlocked([&] { return (quantize ? lib.kvx_quantize_blocks : lib.kvx_dequantize_blocks)(&a, L.stream); }));
  Py_RETURN_NONE;
}
PyObject* quantize_blocks(PyObject* const* args, Py_ssize_t n) { return blocks_call(args, n, true); }
PyObject* dequantize_blocks(PyObject* const* args, Py_ssize_t n) { return blocks_call(args, n, false); }

// dequantize_rows(codes, scales, zero_points, bits, out): everything contiguous, rows of out's last axis
PyObject* dequantize_rows(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 5, "dequantize_rows");
  const at::Tensor &codes = tensor(args[0], "codes"), &scale = tensor(args[1], "scales"), &zp = tensor(args[2], "zero_points"), &out = tensor(args[4], "out");
  const Launch L(codes);
  const int64_t d = out.size(-1), bits = integer(args[3]);
  check(unlocked([&] {
    return lib.kvx_dequantize_rows_typed((const uint8_t*)codes.data_ptr(), (const float*)scale.data_ptr(), (const int32_t*)zp.data_ptr(), out.numel() / d,
                                         (int32_t)d, (int32_t)bits, elem_dtype(out.scalar_type()), out.data_ptr(), d, L.stream);
  }));
  Py_RETURN_NONE;
}

// ---- normalisation, activation, rotary encoding ----------------------------------------------------------------------------

at::Tensor rows2d(const at::Tensor& t, int64_t dim) {
  at::Tensor r = t.reshape({-1, dim});
  return r.stride(1) == 1 ? r : r.contiguous();
}

// rmsnorm(x, weight, eps, out or None) -> out
PyObject* rmsnorm(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 4, "rmsnorm");
  const at::Tensor &x = tensor(args[0], "x"), &weight = tensor(args[1], "weight");
  require_gpu(x);
  require_gpu(weight);
  if (x.scalar_type() != at::kBFloat16 || weight.scalar_type() != at::kFloat)
    raise(PyExc_ValueError, "rmsnorm takes bfloat16 rows and a float32 weight");
  const int64_t dim = x.dim() ? x.size(-1) : 0;
  if (weight.dim() != 1 || weight.size(0) != dim) raise(PyExc_ValueError, "weight.shape = %s, must be (%lld,)", shape_str(weight).c_str(), (long long)dim);
  const Launch L(x);
  const float eps = (float)real(args[2]);
  at::Tensor x2, out;
  if (args[3] != Py_None) out = tensor(args[3], "out");
  check(unlocked([&] {
    x2 = rows2d(x, dim);
    if (!out.defined()) out = L.empty(x.sizes(), x.scalar_type());
    const at::Tensor o2 = out.view({-1, dim});
    return lib.kvx_rmsnorm_rows(x2.data_ptr(), x2.stride(0), o2.data_ptr(), o2.stride(0), (const float*)weight.data_ptr(), x2.size(0), (int32_t)dim, eps,
                                L.stream);
  }));
  return wrap(out);
}

// add_rmsnorm(x, delta, weight, eps) -> normed rows; x += delta in place
PyObject* add_rmsnorm(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 4, "add_rmsnorm");
  const at::Tensor &x = tensor(args[0], "x"), &delta = tensor(args[1], "delta"), &weight = tensor(args[2], "weight");
  for (const at::Tensor* t : {&x, &delta, &weight}) require_gpu(*t);
  if (x.scalar_type() != at::kBFloat16 || delta.scalar_type() != at::kBFloat16 || weight.scalar_type() != at::kFloat)
    raise(PyExc_ValueError, "add_rmsnorm_ takes bfloat16 rows and a float32 weight");
  const int64_t dim = x.dim() ? x.size(-1) : 0;
  if (x.sizes() != delta.sizes() || weight.dim() != 1 || weight.size(0) != dim || !x.is_contiguous())
    raise(PyExc_ValueError, "x %s (contiguous), delta %s, weight %s do not fit", shape_str(x).c_str(), shape_str(delta).c_str(), shape_str(weight).c_str());
  const Launch L(x);
  const float eps = (float)real(args[3]);
  at::Tensor d2, out;
  check(unlocked([&] {
    d2 = rows2d(delta, dim);
    out = L.empty(x.sizes(), x.scalar_type());
    return lib.kvx_add_rmsnorm_rows(x.data_ptr(), dim, d2.data_ptr(), d2.stride(0), x.data_ptr(), dim, out.data_ptr(), dim, (const float*)weight.data_ptr(),
                                    x.numel() / dim, (int32_t)dim, eps, L.stream);
  }));
  return wrap(out);
}

// swiglu(gate_up) -> activation
PyObject* swiglu(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 1, "swiglu");
  const at::Tensor& g = tensor(args[0], "gate_up");
  require_gpu(g);
  if (g.scalar_type() != at::kBFloat16 || g.dim() == 0 || g.size(-1) % 16 != 0)
    raise(PyExc_ValueError, "swiglu takes bfloat16 rows of even width, a multiple of 16");
  const int64_t dim = g.size(-1) / 2;
  const Launch L(g);
  std::vector<int64_t> sizes = g.sizes().vec();
  sizes.back() = dim;
  at::Tensor g2, out;
  check(unlocked([&] {
    g2 = rows2d(g, 2 * dim);
    out = L.empty(sizes, g.scalar_type());
    return lib.kvx_swiglu_rows(g2.data_ptr(), g2.stride(0), out.data_ptr(), dim, g2.size(0), (int32_t)dim, L.stream);
  }));
  return wrap(out);
}

// qk_norm_rope(qkv, n_head, n_query_groups, head_size, q_weight or None, k_weight or None, eps, cos, sin, input_pos)
PyObject* qk_norm_rope(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 10, "qk_norm_rope");
  const at::Tensor &qkv = tensor(args[0], "qkv"), &cos = tensor(args[7], "cos"), &sin = tensor(args[8], "sin");
  for (const at::Tensor* t : {&qkv, &cos, &sin}) require_gpu(*t);
  if (qkv.scalar_type() != at::kBFloat16 || qkv.dim() != 3 || qkv.stride(2) != 1)
    raise(PyExc_ValueError, "qkv must be a bfloat16 (B, num, heads * head_size) tensor with a contiguous last axis");
  const int64_t hq = integer(args[1]), hkv = integer(args[2]), d = integer(args[3]);
  if (qkv.size(2) != (hq + 2 * hkv) * d)
    raise(PyExc_ValueError, "qkv.shape[-1] = %lld does not fit %lld + 2 * %lld heads of %lld", (long long)qkv.size(2), (long long)hq, (long long)hkv, (long long)d);
  if (cos.sizes() != sin.sizes() || cos.dim() != 2 || cos.size(1) != d / 2 || cos.scalar_type() != at::kFloat)
    raise(PyExc_ValueError, "cos / sin must be float32 (positions, head_size / 2) tables");
  const at::Tensor *qw = opt_tensor(args[4], "q_weight"), *kw = opt_tensor(args[5], "k_weight");
  const float eps = (float)real(args[6]);
  const int64_t input_pos = converted(args[9]);
  const Launch L(qkv);
  check(unlocked([&] {
    return lib.kvx_qk_norm_rope(qkv.data_ptr(), qkv.stride(0), qkv.stride(1), (int32_t)qkv.size(0), (int32_t)qkv.size(1), (int32_t)hq, (int32_t)hkv,
                                (int32_t)d, qw ? (const float*)qw->data_ptr() : nullptr, kw ? (const float*)kw->data_ptr() : nullptr, eps,
                                (const float*)cos.data_ptr(), (const float*)sin.data_ptr(), (int32_t)cos.size(0), (int32_t)input_pos, L.stream);
  }));
  Py_RETURN_NONE;
}

// ---- module -------------------------------------------------------------------------------------------------------------------

// bind(path, KvxError, torch.OutOfMemoryError): take the entry points from the library at `path` (already loaded by ctypes: the same handle)
PyObject* bind(PyObject* const* args, Py_ssize_t n) {
  require_args(n, 3, "bind");
  const char* path = PyUnicode_AsUTF8(args[0]);
  if (!path) throw PyRaised{};
  void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!h) raise(PyExc_ImportError, "%s", dlerror());
  Lib l;
#define X(name)                                    \
  l.name = (decltype(l.name))dlsym(h, #name);      \
  if (!l.name) raise(PyExc_ImportError, "%s does not export %s", path, #name);
  KVX_HOST_SYMBOLS(X)
#undef X
  l.kvx_cache_write_first = (decltype(l.kvx_cache_write_first))dlsym(h, "kvx_cache_write_first");
  l.kvx_sdpa_prefill_first = (decltype(l.kvx_sdpa_prefill_first))dlsym(h, "kvx_sdpa_prefill_first");
  l.bound = true;
  lib = l;
  Py_XSETREF(kvx_error, Py_NewRef(args[1]));
  Py_XSETREF(memory_error, Py_NewRef(args[2]));
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject* const*, Py_ssize_t), bool NEEDS_LIB = true>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  try {
    if (NEEDS_LIB && !lib.bound) raise(PyExc_ImportError, "the kernel library is not bound");
    return F(args, n);
  } catch (const PyRaised&) {
    return nullptr;
  } catch (const c10::OutOfMemoryError& e) {
    PyErr_SetString(memory_error, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))entry<name>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))entry<bind, false>, METH_FASTCALL, nullptr},
    METHOD(prefill), METHOD(score_sum), METHOD(decode), METHOD(check_qkv), METHOD(cache_write), METHOD(cache_write_first), METHOD(prefill_first), METHOD(cache_update), METHOD(cache_decode_step),
    METHOD(quantize_blocks), METHOD(dequantize_blocks), METHOD(dequantize_rows), METHOD(rmsnorm), METHOD(add_rmsnorm),
    METHOD(swiglu), METHOD(qk_norm_rope), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Native host path of the kernels (see csrc/host.cpp).", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
#define X(n) \
  if (!(names.n = PyUnicode_InternFromString(#n))) return nullptr;
  ATTRS(X)
#undef X
  return PyModule_Create(&module_def);
}
