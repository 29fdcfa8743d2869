// Native half of the Python op layer: argument checks on torch tensors and the calls into libkvq_hip.so.
//
// A decode step of a small batch is 15 - 35 us of GPU work in three to five launches, and the Python that checked its
// tensors and marshalled some thirty ctypes arguments per call took longer than that (27 us for one short sequence,
// 37 us for a small MLA step).  Here a call reads the tensors through torch's C++ interface: one GQA step is two
// calls of about a microsecond each beside the launches themselves.  Checks and messages are the op layer's; nothing
// is remembered between calls.
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdarg>
#include <cstdio>

#include "kvq.h"

namespace {

struct Raised {};   // a Python error is set

[[noreturn]] void raise(PyObject* type, const char* fmt, ...) {
  char msg[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(msg, sizeof(msg), fmt, ap);
  va_end(ap);
  PyErr_SetString(type, msg);
  throw Raised{};
}
#define NEED(cond, ...) \
  do {                  \
    if (!(cond)) raise(PyExc_RuntimeError, __VA_ARGS__); \
  } while (0)

// ---- arguments ----------------------------------------------------------------------------------------------------

typedef const at::Tensor* Ten;

struct Args {
  PyObject* const* a;
  Py_ssize_t n, i = 0;
  Args(PyObject* const* args, Py_ssize_t nargs, Py_ssize_t want, const char* op) : a(args), n(nargs) {
    if (nargs != want) raise(PyExc_TypeError, "%s: %zd arguments, %zd expected", op, nargs, want);
  }
  Ten opt() {
    PyObject* o = a[i++];
    if (o == Py_None) return nullptr;
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "a tensor was expected, got %s", Py_TYPE(o)->tp_name);
    return &THPVariable_Unpack(o);
  }
  const at::Tensor& ten() {
    Ten t = opt();
    if (t == nullptr) raise(PyExc_TypeError, "a tensor was expected, got None");
    return *t;
  }
  int64_t num() {
    const long long v = PyLong_AsLongLong(a[i++]);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
  }
  double real() {
    const double v = PyFloat_AsDouble(a[i++]);
    if (v == -1.0 && PyErr_Occurred()) throw Raised{};
    return v;
  }
  template <class T>
  const T* addr() { return reinterpret_cast<const T*>(static_cast<uintptr_t>(num())); }
};

void* ptr(const at::Tensor& t) { return t.data_ptr(); }
void* ptr(Ten t) { return t == nullptr ? nullptr : t->data_ptr(); }

int dtype_code(const at::Tensor& t, const char* what) {
  switch (t.scalar_type()) {
    case at::kFloat: return KVQ_F32;
    case at::kBFloat16: return KVQ_BF16;
    case at::kHalf: return KVQ_F16;
    default: break;
  }
  raise(PyExc_RuntimeError, "%s: unsupported dtype %s", what, c10::toString(t.scalar_type()));
}

// absmax floor of the quantisers: 1e-10 in the source dtype, as a float
float eps_of(int code) {
  switch (code) {
    case KVQ_BF16: return static_cast<float>(c10::BFloat16(1e-10f));
    case KVQ_F16: return static_cast<float>(c10::Half(1e-10f));
    default: return 1e-10f;
  }
}

// The device all of a call's tensors lie on.
struct Device {
  int index = -1;
  void add(const at::Tensor& t) {
    NEED(t.is_cuda(), "int8 KV-cache ops need GPU tensors (there is no CPU path)");
    const int d = t.get_device();
    if (index < 0) index = d;
    else NEED(d == index, "tensors on different devices: cuda:%d vs cuda:%d", index, d);
  }
  void add(Ten t) {
    if (t != nullptr) add(*t);
  }
};
template <class... T>
int device_of(const T&... t) {
  Device d;
  (d.add(t), ...);
  return d.index;
}

// The interpreter's lock given up, and a device made current, until the end of the block.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
struct OnDevice {
  int before;
  OnDevice(int device, const char* op) : before(device) {
    NEED(hipGetDevice(&before) == hipSuccess, "%s: no current device", op);
    if (before == device) before = -1;
    else NEED(hipSetDevice(device) == hipSuccess, "%s: cannot select device %d", op, device);
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// Calls f, an entry of the library, with the tensors' device current, on its current stream and without the
// interpreter's lock (a launch may wait for room in the queue).  The arguments are plain values, taken from the tensors
// by the caller, who holds the lock: a tensor without storage raises there (and may run Python to do so).
template <class F, class... A>
void call(int device, const char* op, F f, A... args) {
  int rc;
  char why[512] = "";
  {
    const OnDevice on(device, op);
    const kvq_stream_t s = reinterpret_cast<kvq_stream_t>(c10::hip::getCurrentHIPStream(device).stream());
    const Unlocked unlocked;
    rc = f(args..., s);
    if (rc != 0) snprintf(why, sizeof(why), "%s", kvq_last_error());
  }
  NEED(rc == 0, "%s failed (status %d): %s", op, rc, why);
}

// A query or output operand: [rows, heads, head_size], or the layer's flat [rows, heads * head_size].
struct Rows {
  int64_t rows, heads, dim, stride_t, stride_h, stride_d;
};
Rows rows_of(const at::Tensor& t, int64_t heads, int64_t dim, const char* what) {
  if (t.dim() == 3) return {t.size(0), t.size(1), t.size(2), t.stride(0), t.stride(1), t.stride(2)};
  NEED(heads > 0 && t.dim() == 2 && t.size(1) == heads * dim, "%s", what);
  return {t.size(0), heads, dim, t.stride(0), dim * t.stride(1), t.stride(1)};
}

void check_heads(Ten t, int64_t heads, int device, const char* what) {
  if (t == nullptr) return;
  NEED(t->scalar_type() == at::kFloat && t->is_contiguous() && t->dim() == 1 && t->size(0) == heads && t->is_cuda() &&
           t->get_device() == device,
       "%s must be a contiguous float32 [num_q_heads] tensor on the device of q", what);
}

bool shape_is(const at::Tensor& t, std::initializer_list<int64_t> want) {
  return t.sizes() == c10::IntArrayRef(want.begin(), want.size());
}

// ---- GQA ----------------------------------------------------------------------------------------------------------

// (key, value, cache, slot_mapping, geom, base)
PyObject* cache_update(Args& in) {
  const at::Tensor &key = in.ten(), &value = in.ten(), &cache = in.ten(), &slots = in.ten();
  const auto* g = in.addr<kvq_cache_geom>();
  void* base = const_cast<void*>(in.addr<void>());
  const int dev = device_of(key, value, cache, slots);
  NEED(key.dim() == 3 && value.sizes() == key.sizes() && key.scalar_type() == value.scalar_type(),
       "key/value must be [num_tokens, num_kv_heads, head_size] of one dtype");
  NEED(key.size(1) == g->num_kv_heads && key.size(2) == g->head_size,
       "key shape (%ld, %ld, %ld) does not match cache (Hkv=%d, D=%d)", (long)key.size(0), (long)key.size(1),
       (long)key.size(2), g->num_kv_heads, g->head_size);
  NEED(key.stride(2) == 1 && value.stride(2) == 1, "key/value head dim must be contiguous");
  NEED(slots.scalar_type() == at::kLong && slots.dim() == 1 && slots.is_contiguous(),
       "slot_mapping must be a contiguous 1-D int64 tensor");
  NEED(slots.size(0) <= key.size(0), "slot_mapping is longer than key");
  const int dt = dtype_code(key, "key");
  call(dev, "reshape_and_cache_flash_per_token_head_quant", kvq_reshape_and_cache_int8, ptr(key), ptr(value), dt,
       key.stride(0), key.stride(1), value.stride(0), value.stride(1), base, g, static_cast<const int64_t*>(ptr(slots)),
       slots.size(0), eps_of(dt));
  Py_RETURN_NONE;
}

// The flag that tells the library of a batch of short sequences.  A launch that is being captured is replayed on whatever
// lengths the buffers hold then, and a replay cannot change the launch: there only what the block table can hold counts
// (one sequence captured at 300 tokens, 8 kv heads: replayed at 4000 26.8 us with a workgroup per kv head, 12.0 cut, at
// 100 000 483 and 40 us; replayed at 300 8.5 and 9.4).
int short_context(int64_t max_k, const at::Tensor& table, const kvq_cache_geom* g, int64_t num_seqs, int device) {
  if (max_k > KVQ_SHORT_CONTEXT) return 0;
  const int limit = kvq_short_context_tokens(g, (int)num_seqs);
  if (max_k > limit) return 0;
  if (table.size(1) * g->block_size > limit) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream(device).stream(), &status) != hipSuccess) {
      (void)hipGetLastError();   // the legacy stream while another one captures: no capture of this call
      status = hipStreamCaptureStatusNone;
    }
    if (status != hipStreamCaptureStatusNone) return 0;
  }
  return KVQ_ATTN_SHORT_CONTEXT;
}

// (q, out, rows, num_q_heads, cache, geom, base, cu_seqlens_q, seqused_k, block_table, max_seqlen_q, max_seqlen_k, scale,
//  flags, window, softcap, sinks, alibi, lse, workspace, splits); rows < 0: all rows of q; num_q_heads: of flat q / out
PyObject* paged_attention(Args& in) {
  const at::Tensor &q = in.ten(), &out = in.ten();
  const int64_t limit = in.num(), flat_heads = in.num();
  const at::Tensor& cache = in.ten();
  const auto* g = in.addr<kvq_cache_geom>();
  const void* base = in.addr<void>();
  const at::Tensor &cu = in.ten(), &lens = in.ten(), &table = in.ten();
  const int64_t max_q = in.num(), max_k = in.num();
  const double scale = in.real();
  const int asked = (int)in.num(), window = (int)in.num();
  const double softcap = in.real();
  const Ten sinks = in.opt(), alibi = in.opt(), lse = in.opt(), ws = in.opt();
  const int splits = (int)in.num();
  const int dev = device_of(q, cache, out, cu, lens, table, ws, lse);
  const char* qwhat = "q/out must be [num_tokens, num_q_heads, head_size] matching the cache head size";
  Rows rq = rows_of(q, flat_heads, g->head_size, qwhat), ro = rows_of(out, flat_heads, g->head_size, qwhat);
  if (limit >= 0) {
    NEED(rq.rows >= limit && ro.rows >= limit, "%s", qwhat);
    rq.rows = ro.rows = limit;
  }
  NEED(rq.rows == ro.rows && rq.heads == ro.heads && rq.dim == ro.dim && rq.dim == g->head_size, "%s", qwhat);
  NEED(rq.stride_d == 1 && ro.stride_d == 1, "q/out head dim must be contiguous");
  NEED(lens.scalar_type() == at::kInt && cu.scalar_type() == at::kInt && table.scalar_type() == at::kInt,
       "seqused_k, cu_seqlens_q and block_table must be int32");
  const int64_t B = lens.size(0);
  NEED(cu.size(0) == B + 1 && table.size(0) >= B && table.stride(1) == 1,
       "cu_seqlens_q must have num_seqs+1 entries and block_table num_seqs contiguous rows");
  NEED(lens.is_contiguous() && cu.is_contiguous(), "seqused_k and cu_seqlens_q must be contiguous");
  NEED(table.size(1) * g->block_size >= max_k, "block_table rows are too short for max_seqlen_k");
  if (B == 0 || rq.rows == 0) Py_RETURN_NONE;
  check_heads(sinks, rq.heads, dev, "sinks");
  check_heads(alibi, rq.heads, dev, "alibi_slopes");
  if (lse != nullptr)
    NEED(lse->scalar_type() == at::kFloat && lse->is_contiguous() && shape_is(*lse, {rq.rows, rq.heads}),
         "lse must be a contiguous float32 [num_tokens, num_q_heads] tensor");
  const int odt = dtype_code(out, "out"), qdt = dtype_code(q, "q");
  const auto *bt = static_cast<const int32_t*>(ptr(table)), *sl = static_cast<const int32_t*>(ptr(lens)),
             *cq = static_cast<const int32_t*>(ptr(cu));
  const auto *sk = static_cast<const float*>(ptr(sinks)), *al = static_cast<const float*>(ptr(alibi));
  auto* ls = static_cast<float*>(ptr(lse));
  const char* op = "unified_attention";
  const int flags = asked | short_context(max_k, table, g, B, dev);
  if (ws == nullptr)   // the states live in the library's own array
    call(dev, op, kvq_paged_attn_int8_static_scratch, ptr(out), odt, ro.stride_t, ro.stride_h, ptr(q), qdt, rq.stride_t,
         rq.stride_h, base, g, bt, table.stride(0), sl, cq, (int)B, (int)rq.heads, (int)max_q, (float)scale, flags, window,
         (float)softcap, sk, al, ls);
  else if (splits > 1 && max_q > 1)
    call(dev, op, kvq_paged_attn_int8_split_prefill, ptr(out), odt, ro.stride_t, ro.stride_h, ptr(q), qdt, rq.stride_t,
         rq.stride_h, base, g, bt, table.stride(0), sl, cq, (int)B, (int)rq.heads, (int)max_q, (float)scale, flags, window,
         (float)softcap, sk, al, ls, (int)rq.rows, splits, ptr(ws), ws->nbytes());
  else
    call(dev, op, kvq_paged_attn_int8, ptr(out), odt, ro.stride_t, ro.stride_h, ptr(q), qdt, rq.stride_t, rq.stride_h, base,
         g, bt, table.stride(0), sl, cq, (int)B, (int)rq.heads, (int)max_q, (float)scale, flags, window, (float)softcap, sk,
         al, ls, ptr(ws), ws->nbytes());
  Py_RETURN_NONE;
}

// (q, key, value, out, rows, num_q_heads, cache, geom, base, seqused_k, block_table, max_seqlen_k, scale, window, softcap,
//  sinks, alibi, lse, workspace, slot_mapping); flat q / out / key / value as above
PyObject* decode_with_update(Args& in) {
  const at::Tensor &q = in.ten(), &key = in.ten(), &value = in.ten(), &out = in.ten();
  const int64_t limit = in.num(), flat_heads = in.num();
  const at::Tensor& cache = in.ten();
  const auto* g = in.addr<kvq_cache_geom>();
  const void* base = in.addr<void>();
  const at::Tensor &lens = in.ten(), &table = in.ten();
  const int64_t max_k = in.num();
  const double scale = in.real();
  const int window = (int)in.num();
  const double softcap = in.real();
  const Ten sinks = in.opt(), alibi = in.opt(), lse = in.opt();
  const at::Tensor& ws = in.ten();
  const Ten slots = in.opt();
  const int dev = device_of(q, key, value, cache, out, lens, table, ws, lse, slots);
  const char* qwhat = "q/out must be [num_seqs, num_q_heads, head_size] matching the cache head size";
  const char* kwhat = "key/value must be [num_seqs, num_kv_heads, head_size] of one dtype";
  const int64_t B = lens.size(0), flat_kv = flat_heads > 0 ? g->num_kv_heads : 0;
  Rows rq = rows_of(q, flat_heads, g->head_size, qwhat), ro = rows_of(out, flat_heads, g->head_size, qwhat);
  Rows rk = rows_of(key, flat_kv, g->head_size, kwhat), rv = rows_of(value, flat_kv, g->head_size, kwhat);
  if (limit >= 0) {
    NEED(rq.rows >= limit && ro.rows >= limit, "%s", qwhat);
    NEED(rk.rows >= limit && rv.rows >= limit, "%s", kwhat);
    rq.rows = ro.rows = rk.rows = rv.rows = limit;
  }
  NEED(rq.rows == ro.rows && rq.heads == ro.heads && rq.dim == ro.dim && rq.dim == g->head_size && rq.rows == B, "%s", qwhat);
  NEED(rq.stride_d == 1 && ro.stride_d == 1, "q/out head dim must be contiguous");
  NEED(rk.rows == rv.rows && rk.heads == rv.heads && rk.dim == rv.dim && key.scalar_type() == value.scalar_type() &&
           rk.rows >= B,
       "%s", kwhat);
  NEED(rk.heads == g->num_kv_heads && rk.dim == g->head_size,
       "key shape (%ld, %ld, %ld) does not match cache (Hkv=%d, D=%d)", (long)rk.rows, (long)rk.heads, (long)rk.dim,
       g->num_kv_heads, g->head_size);
  NEED(rk.stride_d == 1 && rv.stride_d == 1, "key/value head dim must be contiguous");
  NEED(lens.scalar_type() == at::kInt && table.scalar_type() == at::kInt && lens.is_contiguous(),
       "seqused_k (contiguous) and block_table must be int32");
  NEED(table.size(0) >= B && table.stride(1) == 1, "block_table needs num_seqs contiguous rows");
  NEED(table.size(1) * g->block_size >= max_k, "block_table rows are too short for max_seqlen_k");
  if (slots != nullptr)
    NEED(slots->scalar_type() == at::kLong && slots->dim() == 1 && slots->size(0) >= B && slots->is_contiguous(),
         "slot_mapping must be a contiguous int64 tensor with one entry per sequence");
  if (B == 0) Py_RETURN_NONE;
  if (lse != nullptr)
    NEED(lse->scalar_type() == at::kFloat && lse->is_contiguous() && shape_is(*lse, {B, rq.heads}),
         "lse must be a contiguous float32 [num_seqs, num_q_heads] tensor");
  check_heads(sinks, rq.heads, dev, "sinks");
  check_heads(alibi, rq.heads, dev, "alibi_slopes");
  const int odt = dtype_code(out, "out"), qdt = dtype_code(q, "q"), kdt = dtype_code(key, "key");
  call(dev, "decode_attention_with_cache_update", kvq_paged_attn_int8_fused_write_flags, ptr(out), odt, ro.stride_t, ro.stride_h,
       ptr(q), qdt, rq.stride_t, rq.stride_h, ptr(key), ptr(value), kdt, rk.stride_t, rk.stride_h, rv.stride_t, rv.stride_h,
       eps_of(kdt), const_cast<void*>(base), g, static_cast<const int32_t*>(ptr(table)), table.stride(0),
       static_cast<const int32_t*>(ptr(lens)), static_cast<const int64_t*>(ptr(slots)), (int)B, (int)rq.heads, (float)scale,
       window, (float)softcap, static_cast<const float*>(ptr(sinks)), static_cast<const float*>(ptr(alibi)),
       static_cast<float*>(ptr(lse)), ptr(ws), ws.nbytes(), short_context(max_k, table, g, B, dev));
  Py_RETURN_NONE;
}

// ---- MLA ----------------------------------------------------------------------------------------------------------

// (kv_c, k_pe, cache, slot_mapping, geom, base, layer_form); layer_form: k_pe may be [T, 1, P], as the layer holds it
PyObject* mla_cache_update(Args& in) {
  const at::Tensor &kv_c = in.ten(), &k_pe = in.ten(), &cache = in.ten(), &slots = in.ten();
  const auto* g = in.addr<kvq_mla_geom>();
  void* base = const_cast<void*>(in.addr<void>());
  const bool layer_form = in.num() != 0;
  const int dev = device_of(kv_c, k_pe, cache, slots);
  const bool three = layer_form && k_pe.dim() == 3 && k_pe.size(1) == 1;
  NEED(kv_c.dim() == 2 && (k_pe.dim() == 2 || three) && kv_c.scalar_type() == k_pe.scalar_type(),
       "kv_c [T, R] and k_pe [T, P] must be 2-D of one dtype");
  NEED(kv_c.size(1) == g->kv_lora_rank && k_pe.size(-1) == g->rope_dim, "kv_c / k_pe widths do not match the cache entry");
  NEED(kv_c.stride(1) == 1 && k_pe.stride(-1) == 1, "kv_c / k_pe rows must be contiguous");
  NEED(slots.scalar_type() == at::kLong && slots.is_contiguous(), "slot_mapping must be contiguous int64");
  const int64_t T = slots.size(0);
  NEED(T <= kv_c.size(0) && T <= k_pe.size(0), "slot_mapping is longer than kv_c / k_pe");
  const int dt = dtype_code(kv_c, "kv_c");
  call(dev, "concat_and_cache_mla", kvq_concat_and_cache_mla_int8, ptr(kv_c), ptr(k_pe), dt, kv_c.stride(0),
       k_pe.stride(0), base, g, static_cast<const int64_t*>(ptr(slots)), T, eps_of(dt));
  Py_RETURN_NONE;
}

// (q_nope, W_UK_T, q_pe, cache, o, lse, layer_form, block_table, seq_lens, scale, workspace, geom, base);
// layer_form: o / lse may have more rows than q_nope (a buffer for the largest batch)
PyObject* mla_decode_absorb(Args& in) {
  const at::Tensor &q = in.ten(), &w = in.ten(), &q_pe = in.ten(), &cache = in.ten(), &o = in.ten();
  const Ten lse = in.opt();
  const bool layer_form = in.num() != 0;
  const at::Tensor &table = in.ten(), &lens = in.ten();
  const double scale = in.real();
  const at::Tensor& ws = in.ten();
  const auto* g = in.addr<kvq_mla_geom>();
  const void* base = in.addr<void>();
  const int dev = device_of(q, w, q_pe, cache, o, lse, table, lens, ws);
  NEED(q.dim() == 3, "q_nope must be [B, H, P]");
  const int64_t B = q.size(0), H = q.size(1), P = q.size(2);
  NEED(shape_is(w, {H, P, g->kv_lora_rank}) && shape_is(q_pe, {B, H, g->rope_dim}),
       "W_UK_T must be [H, P, R] and q_pe [B, H, rope]");
  NEED(q.scalar_type() == w.scalar_type() && q.scalar_type() == q_pe.scalar_type(),
       "q_nope, W_UK_T and q_pe must share a dtype");
  NEED(q.stride(2) == 1 && w.stride(2) == 1 && q_pe.stride(2) == 1, "last dims must be contiguous");
  NEED(o.dim() == 3 && (layer_form ? o.size(0) >= B : o.size(0) == B) && o.size(1) == H && o.size(2) == g->kv_lora_rank &&
           o.is_contiguous(),
       "o must be contiguous [B, H, R]");
  NEED(lens.scalar_type() == at::kInt && table.scalar_type() == at::kInt && table.stride(1) == 1,
       "seq_lens and block_table must be int32");
  if (lse != nullptr)
    NEED(lse->scalar_type() == at::kFloat && lse->dim() == 2 && (layer_form ? lse->size(0) >= B : lse->size(0) == B) &&
             lse->size(1) == H && lse->is_contiguous(),
         "lse must be contiguous float32 [B, H]");
  const int odt = dtype_code(o, "o"), qdt = dtype_code(q, "q_nope");
  call(dev, "mla_decode_absorb_int8", kvq_mla_decode_absorb_int8, ptr(o), odt, static_cast<float*>(ptr(lse)), ptr(q), qdt,
       q.stride(0), q.stride(1), (int)P, ptr(w), w.stride(0), w.stride(1), ptr(q_pe), q_pe.stride(0), q_pe.stride(1), base,
       g, static_cast<const int32_t*>(ptr(table)), table.stride(0), static_cast<const int32_t*>(ptr(lens)), (int)B, (int)H,
       (float)scale, ptr(ws), ws.nbytes());
  Py_RETURN_NONE;
}

// (x, rows, W_UV, out); rows < 0: all rows of x
PyObject* mla_v_up_proj(Args& in) {
  const at::Tensor& x = in.ten();
  const int64_t limit = in.num();
  const at::Tensor &w = in.ten(), &out = in.ten();
  const int dev = device_of(x, w, out);
  NEED(x.dim() == 3 && w.dim() == 3, "mla_v_up_proj takes x [B, H, L] and W_UV [H, L, V]");
  NEED(limit <= x.size(0), "mla_v_up_proj: x has fewer rows than asked for");
  const int64_t B = limit < 0 ? x.size(0) : limit, H = x.size(1), L = x.size(2), V = w.size(2);
  NEED(shape_is(w, {H, L, V}), "W_UV must be [H, L, V]");
  const bool flat = out.dim() == 2;
  if (flat)
    NEED(shape_is(out, {B, H * V}) && out.stride(1) == 1, "out must be [B, H * V] with a contiguous last dim");
  else
    NEED(shape_is(out, {B, H, V}) && out.stride(2) == 1, "out must be [B, H, V] with a contiguous last dim");
  NEED(x.scalar_type() == w.scalar_type() && x.scalar_type() == out.scalar_type(), "x, W_UV and out must share a dtype");
  NEED(x.stride(2) == 1 && w.stride(2) == 1, "last dims must be contiguous");
  if (B == 0) Py_RETURN_NONE;
  const int dt = dtype_code(x, "x");
  call(dev, "mla_v_up_proj", kvq_mla_v_up_proj, ptr(out), out.stride(0), flat ? V : out.stride(1), ptr(x), dt, x.stride(0),
       x.stride(1), ptr(w), w.stride(0), w.stride(1), (int)B, (int)H, (int)L, (int)V);
  Py_RETURN_NONE;
}

// ---- cache identity -----------------------------------------------------------------------------------------------

// A tensor's identity as a cache: storage, address, shape and strides.
struct CacheRef {
  const c10::StorageImpl* storage;
  const void* data;
  int64_t dim, sizes[5], strides[5];
};

CacheRef ref_of(const at::Tensor& t) {
  CacheRef r{};
  NEED(t.dim() <= 5, "a cache tensor of more than five dimensions");
  r.storage = t.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl();
  r.data = t.data_ptr();
  r.dim = t.dim();
  for (int64_t i = 0; i < r.dim; ++i) {
    r.sizes[i] = t.size(i);
    r.strides[i] = t.stride(i);
  }
  return r;
}

const char* kRefName = "kvq cache identity";
void drop_ref(PyObject* c) { delete static_cast<CacheRef*>(PyCapsule_GetPointer(c, kRefName)); }

// (cache) -> an object that is_cache compares tensors with
PyObject* cache_ref(Args& in) {
  return PyCapsule_New(new CacheRef(ref_of(in.ten())), kRefName, drop_ref);
}

// (ref or None, cache) -> whether the tensor is the one the reference was made from, or another view that is the same
PyObject* is_cache(Args& in) {
  PyObject* c = in.a[in.i++];
  const at::Tensor& t = in.ten();
  if (c == Py_None) Py_RETURN_FALSE;
  const auto* want = static_cast<const CacheRef*>(PyCapsule_GetPointer(c, kRefName));
  if (want == nullptr) throw Raised{};
  bool same = t.dim() == want->dim && t.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl() == want->storage &&
              t.data_ptr() == want->data;
  for (int64_t i = 0; same && i < want->dim; ++i) same = t.size(i) == want->sizes[i] && t.stride(i) == want->strides[i];
  return PyBool_FromLong(same);
}

template <PyObject* (*F)(Args&), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  try {
    Args in(args, nargs, N, "kvq_torch");
    return F(in);
  } catch (const Raised&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

#define METHOD(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(cache_update, 6),       METHOD(paged_attention, 21), METHOD(decode_with_update, 20),
                         METHOD(mla_cache_update, 7),   METHOD(mla_decode_absorb, 13), METHOD(mla_v_up_proj, 4),
                         METHOD(cache_ref, 1),          METHOD(is_cache, 2),         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kvq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_kvq_torch(void) { return PyModule_Create(&module); }
