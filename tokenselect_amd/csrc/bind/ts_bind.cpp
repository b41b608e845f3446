// The per-call host work of ops.DecodeLayer and ops.PrefillChunk in native code: checks the
// tensors, fills the structs of include/tokenselect.h and calls the library on the current
// stream.
//
// A layer call is a few microseconds of kernel launches; the same checks and ctypes structs
// in Python took 25 us around them, longer than the kernels of a short context run (8 layers
// of a 2003-token request, 16 calls: 577 us a pass, of which the GPU was busy 290).  Nothing
// is computed here and nothing is kept between calls but the buffers the object owns and the
// layout its workspace was last left clean for.
//
// Built with the host compiler against PyTorch's headers; the library's entry points are
// handed over as addresses by _lib.py, so that there is one loaded copy of it.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <exception>
#include <optional>
#include <string>

#include "../../../include/tokenselect.h"

namespace {

// A Python exception is set; unwinds to the method's end.
struct Raised {};
[[noreturn]] void raise(PyObject* type, const std::string& text) {
  PyErr_SetString(type, text.c_str());
  throw Raised{};
}
[[noreturn]] void bad_value(const std::string& text) { raise(PyExc_ValueError, text); }

// An owned reference.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {
    if (!p) throw Raised{};
  }
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

const char* dtype_name(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return "torch.bfloat16";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    default: return at::toString(t);
  }
}

std::string shape_text(const at::Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, std::string(name) + " must be a torch.Tensor");
  return THPVariable_Unpack(o);
}

// A tensor on the GPU of the given type; ndim < 0: any number of dims.
const at::Tensor& need(PyObject* o, const char* name, at::ScalarType dtype, int ndim = -1) {
  const at::Tensor& t = tensor(o, name);
  if (t.scalar_type() != dtype)
    raise(PyExc_TypeError, std::string(name) + " must be " + dtype_name(dtype) + ", got " + dtype_name(t.scalar_type()));
  if (!t.is_cuda())
    bad_value(std::string(name) + " must live on the GPU (got " + t.device().str() + "); there is no CPU path");
  if (!t.is_contiguous()) bad_value(std::string(name) + " must be contiguous");
  if (ndim >= 0 && t.dim() != ndim)
    bad_value(std::string(name) + " must have " + std::to_string(ndim) + " dims, got shape " + shape_text(t));
  return t;
}

// Attribute names of Batch, SelectionCache and PagePool, interned once.
#define TS_NAMES(X)                                                                              \
  X(seq_lens) X(table) X(max_seq_len) X(k_per_req) X(fault) X(host_seq_lens) X(hint)             \
  X(separate_kernels) X(rerun) X(wait_us) X(absent_workgroups) X(workspace_clean)                \
  X(q_cache) X(topk_cache) X(cache_len) X(counters) X(threshold)                                 \
  X(free_pages) X(free_count) X(ticket)
#define TS_DECLARE(n) PyObject* n_##n;
TS_NAMES(TS_DECLARE)
#undef TS_DECLARE

bool intern_names() {
#define TS_INTERN(n) \
  if (!(n_##n = PyUnicode_InternFromString(#n))) return false;
  TS_NAMES(TS_INTERN)
#undef TS_INTERN
  return true;
}

PyObject* attr(PyObject* o, PyObject* name) {
  PyObject* v = PyObject_GetAttr(o, name);
  if (!v) throw Raised{};
  return v;
}
long as_long(PyObject* o) {
  if (!PyLong_Check(o)) {  // (what int() takes: a numpy integer, a one-element tensor)
    const Ref number(PyNumber_Long(o));
    return as_long(number.p);
  }
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw Raised{};
  return v;
}
long long_attr(PyObject* o, PyObject* name) {
  const Ref v(attr(o, name));
  return as_long(v.p);
}
bool bool_attr(PyObject* o, PyObject* name) {
  const Ref v(attr(o, name));
  const int b = PyObject_IsTrue(v.p);
  if (b < 0) throw Raised{};
  return b != 0;
}

using StepFn = int (*)(const ts_config*, const ts_batch*, const ts_new_kv*, const void*, int32_t, int32_t,
                       const float*, const float*, void*, void*, int64_t, const ts_selcache*, void*, int32_t*, int32_t*, int64_t, int32_t*,
                       void*, size_t, ts_stream_t);
using LayerFn = int (*)(const ts_config*, const ts_batch*, const void*, const float*, const float*, const void*,
                        const void*, int64_t, const ts_selcache*, void*, int32_t*, int32_t*, int64_t, int32_t*,
                        void*, size_t, ts_stream_t);
using ChunkStepFn = int (*)(const ts_config*, const ts_batch*, const ts_new_kv*, const void*, int32_t, int32_t,
                            int32_t, const float*, const float*, int64_t, void*, void*, int64_t, void*, int32_t*, int32_t*, int64_t,
                            int32_t*, void*, size_t, ts_stream_t);
using ChunkFn = int (*)(const ts_config*, const ts_batch*, const void*, int32_t, const float*, const float*, int64_t,
                        const void*, const void*, int64_t, void*, int32_t*, int32_t*, int64_t, int32_t*, void*,
                        size_t, ts_stream_t);
using PromptFn = int (*)(const ts_config*, const ts_batch*, const ts_new_kv*, const void*, int32_t, int32_t, int32_t,
                         int32_t, const float*, const float*, int64_t, void*, void*, int64_t, void*, void*, size_t,
                         ts_stream_t);
using PromptBytesFn = size_t (*)(const ts_config*, int32_t, int32_t, int32_t);
using LayoutFn = int64_t (*)(const ts_config*, int32_t, int32_t);
LayoutFn decode_layer_layout;
StepFn decode_step;
LayerFn decode_layer;
ChunkStepFn prefill_step;
ChunkFn prefill_chunk;
PromptFn prefill_prompt;
PromptBytesFn prefill_prompt_bytes;

// What a DecodeLayer (max_rows == 0) or a PrefillChunk owns.
struct Owned {
  ts_config cfg;
  at::Tensor workspace, cos, sin, out, sel, sel_pos, sel_len, fault;
  int64_t batch, max_seq_len, max_rows;
  // (batch, max_seq_len) that the selection's counters in the workspace are clean for, -1: none.
  int64_t clean_batch = -1, clean_len = -1;
  int64_t clean_layout = -1;  // ts_decode_layer_layout of that call
  // The workspace has users that the object does not see: the replays of a graph into which a
  // call on it was recorded, or a shallow copy of the object.  They may have used it since any
  // call that is remembered, so from then on none is.
  bool shared = false;
  void forget_clean() { clean_batch = clean_len = clean_layout = -1; }
};

struct Runner {
  PyObject_HEAD
  Owned* own;
};

uint32_t fault_of(const Owned& o) { return *(const volatile uint32_t*)o.fault.data_ptr(); }

const at::Tensor& check_pool(const ts_config& cfg, PyObject* o, const char* name) {
  const at::Tensor& t = need(o, name, at::kBFloat16, 3);
  if (t.size(1) != cfg.num_kv_heads || t.size(2) != cfg.head_dim)
    bad_value(std::string(name) + " must be [rows, " + std::to_string(cfg.num_kv_heads) + ", " +
              std::to_string(cfg.head_dim) + "], got " + shape_text(t));
  return t;
}

// The options of a call, from a Batch and the object's own state.
struct Call {
  ts_batch bt{};
  int64_t table_tokens = 0;
};

void fill_batch(const Owned& o, PyObject* b, bool separate, bool rerun, Call* call) {
  ts_batch& c = call->bt;
  const Ref lens_ref(attr(b, n_seq_lens)), table_ref(attr(b, n_table)), k_ref(attr(b, n_k_per_req)),
      fault_ref(attr(b, n_fault)), host_ref(attr(b, n_host_seq_lens)), hint_ref(attr(b, n_hint));
  // (the Batch holds the tensors: the references below outlive this function)
  const at::Tensor& lens = need(lens_ref.p, "seq_lens", at::kInt, 1);
  const at::Tensor& table = need(table_ref.p, "table", at::kInt, 2);
  const int64_t B = lens.size(0);
  const int64_t max_len = long_attr(b, n_max_seq_len);
  if (table.size(0) != B) bad_value("table must have one row per request");
  if (table.size(1) * o.cfg.page_size < max_len)
    bad_value("table row of " + std::to_string(table.size(1)) + " pages (page_size " +
              std::to_string(o.cfg.page_size) + ") cannot address max_seq_len " + std::to_string(max_len));
  c.batch = (int32_t)B;
  c.max_seq_len = (int32_t)max_len;
  c.seq_lens = (const int32_t*)lens.data_ptr();
  c.table = (const int32_t*)table.data_ptr();
  c.table_stride = table.stride(0);
  if (k_ref.p != Py_None) {
    const at::Tensor& k = need(k_ref.p, "k_per_req", at::kInt, 1);
    if (k.size(0) != B) bad_value("k_per_req must have one entry per request");
    c.k_per_req = (const int32_t*)k.data_ptr();
  }
  if (fault_ref.p == Py_None) {
    c.fault = (uint32_t*)o.fault.data_ptr();
  } else {
    const at::Tensor& f = tensor(fault_ref.p, "fault");
    if (f.scalar_type() != at::kInt || f.numel() != 1 || !(f.is_cuda() || f.is_pinned()))
      bad_value("fault must be one int32 word of device or pinned host memory");
    c.fault = (uint32_t*)f.data_ptr();
  }
  if (host_ref.p != Py_None) {
    const at::Tensor& h = tensor(host_ref.p, "host_seq_lens");
    if (h.scalar_type() != at::kInt || h.is_cuda() || h.dim() != 1 || h.size(0) != B || !h.is_contiguous())
      bad_value("host_seq_lens must be a contiguous [B] int32 tensor on the CPU");
    c.host_seq_lens = (const int32_t*)h.data_ptr();
  }
  if (hint_ref.p != Py_None) {
    const at::Tensor& h = need(hint_ref.p, "hint", at::kInt, 1);
    if (h.size(0) != B) bad_value("hint must have one entry per request");
    c.threshold_hint = (int32_t*)h.data_ptr();
  }
  c.separate_kernels = (separate || bool_attr(b, n_separate_kernels)) ? 1 : 0;
  c.rerun = (rerun || bool_attr(b, n_rerun)) ? 1 : 0;
  c.wait_us = (uint32_t)long_attr(b, n_wait_us);
  c.absent_workgroups = rerun ? 0 : (int32_t)long_attr(b, n_absent_workgroups);
  c.workspace_clean = bool_attr(b, n_workspace_clean) ? 1 : 0;
  if (B > o.batch || max_len > o.max_seq_len) {
    if (o.max_rows > 0) bad_value("one request, within the sizes this PrefillChunk was built for");
    bad_value("batch / max_seq_len exceed what this DecodeLayer was sized for");
  }
  call->table_tokens = table.size(1) * o.cfg.page_size;
}

void fill_cache(const ts_config& cfg, PyObject* cache, int64_t B, ts_selcache* c) {
  const Ref q_ref(attr(cache, n_q_cache)), top_ref(attr(cache, n_topk_cache)), len_ref(attr(cache, n_cache_len)),
      cnt_ref(attr(cache, n_counters)), thr_ref(attr(cache, n_threshold));
  const at::Tensor& q = need(q_ref.p, "q_cache", at::kBFloat16, 2);
  const at::Tensor& top = need(top_ref.p, "topk_cache", at::kInt, 2);
  const at::Tensor& len = need(len_ref.p, "cache_len", at::kInt, 1);
  const at::Tensor& cnt = need(cnt_ref.p, "counters", at::kLong, 2);
  if (q.size(0) != B || q.size(1) != (int64_t)cfg.num_heads * cfg.head_dim || top.size(0) != B ||
      top.size(1) != cfg.top_k || len.size(0) != B || cnt.size(0) != B || cnt.size(1) != 2)
    bad_value("selection cache arrays do not match batch / config");
  const double threshold = PyFloat_AsDouble(thr_ref.p);
  if (threshold == -1.0 && PyErr_Occurred()) throw Raised{};
  *c = ts_selcache{q.data_ptr(), (int32_t*)top.data_ptr(), (int32_t*)len.data_ptr(), (int64_t*)cnt.data_ptr(),
                   (float)threshold};
}

void fill_pages(PyObject* pages, ts_page_pool* c) {
  const Ref list_ref(attr(pages, n_free_pages)), count_ref(attr(pages, n_free_count)), ticket_ref(attr(pages, n_ticket));
  *c = ts_page_pool{(const int32_t*)need(list_ref.p, "free_pages", at::kInt, 1).data_ptr(),
                    (int32_t*)need(count_ref.p, "free_count", at::kInt, 1).data_ptr(),
                    (uint32_t*)need(ticket_ref.p, "ticket", at::kInt, 1).data_ptr()};
}

// Rows of bf16 as the library takes them: at `ptr`, `stride` elements apart.
struct Rows {
  const void* ptr;
  int64_t stride;
  std::optional<at::Tensor> copy;  // of rows that do not lie so
};
// `count` rows of `width` elements, rows [from, from + count) of `t` (the part of a fused QKV
// projection, as a split leaves it: read where it lies).
Rows rows_of(PyObject* obj, const char* name, int64_t from, int64_t count, int64_t width, bool packed) {
  const at::Tensor& t = tensor(obj, name);
  if (t.scalar_type() != at::kBFloat16 || !t.is_cuda()) need(obj, name, at::kBFloat16);  // (raises)
  if (t.dim() < 2 || t.numel() != t.size(0) * width || from + count > t.size(0))
    bad_value(std::string(name) + " must hold rows of " + std::to_string(width) + " elements, got shape " + shape_text(t));
  bool dense = true;  // within a row
  int64_t step = 1;
  for (int64_t d = t.dim() - 1; d > 0; --d) {
    dense = dense && (t.size(d) == 1 || t.stride(d) == step);
    step *= t.size(d);
  }
  const int64_t stride = t.size(0) > 1 ? t.stride(0) : width;
  if (dense && !packed && stride >= width && stride <= INT32_MAX && stride % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0)
    return Rows{(const char*)t.data_ptr() + 2 * from * stride, stride, std::nullopt};
  at::Tensor c = t.narrow(0, from, count).contiguous();
  if ((uintptr_t)c.data_ptr() % 16 != 0) c = c.clone();
  const void* at = c.data_ptr();
  return Rows{at, width, std::move(c)};
}

// The slots of rows [from, from + count), next to each other: a part of a strided tensor is
// copied together.
Rows slots_of(PyObject* obj, int64_t from, int64_t count) {
  const at::Tensor& t = tensor(obj, "out_cache_loc");
  if (t.scalar_type() != at::kInt || !t.is_cuda() || t.dim() != 1) need(obj, "out_cache_loc", at::kInt, 1);  // (raises)
  if (t.size(0) < from + count) bad_value("out_cache_loc does not match the rows");
  if (t.is_contiguous()) return Rows{(const int32_t*)t.data_ptr() + from, 1, std::nullopt};
  at::Tensor c = t.narrow(0, from, count).contiguous();
  const void* at = c.data_ptr();
  return Rows{at, 1, std::move(c)};
}

// Whether what is launched on the current stream is recorded into a graph instead of run.
bool capturing() {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream().stream(), &status) != hipSuccess) {
    (void)hipGetLastError();  // (the legacy stream beside a capture on another one)
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

// The first B rows, as a tensor of its own.  (As narrow() makes it, without the dispatcher: four
// of them are made per call, 2 us of the 17 that a dense step of 2003 tokens takes.)
PyObject* row_view(const at::Tensor& t, int64_t B) {
  at::Tensor rows = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(t.storage()),
                                                             t.key_set(), t.dtype());
  c10::SmallVector<int64_t, 4> sizes(t.sizes().begin(), t.sizes().end());
  sizes[0] = B;
  rows.unsafeGetTensorImpl()->set_storage_offset(t.storage_offset());
  rows.unsafeGetTensorImpl()->set_sizes_and_strides(sizes, t.strides());
  PyObject* v = THPVariable_Wrap(std::move(rows));
  if (!v) throw Raised{};
  return v;
}

// The library's call on the current stream, with the object's buffers.  kv: the tokens to store
// first, or NULL.  q_stride, kv_stride: elements between the rows of a step (0: next to each
// other).  rows: of the chunk.
int call_library(Owned& o, ts_batch* bt, const ts_new_kv* kv, const void* q, int32_t q_stride, int32_t kv_stride,
                 int64_t rows, const at::Tensor& k_pool, const at::Tensor& v_pool, const ts_selcache* cache, void* out,
                 bool rerun = false) {
  // The attention kernel of a plain call leaves the selection's counters zero for the next
  // one of the same layout.
  const bool chunk = o.max_rows > 0;
  // (While a graph is captured the object states nothing: the recorded flag would hold for
  // every replay, whatever used the workspace before it.)
  if (!chunk && !o.shared) o.shared = capturing();
  const bool plain = !chunk && !cache && !bt->separate_kernels && !rerun && !o.shared;
  // (By the layout and not by the length, which grows with every token: it is the same for
  // some 64 steps, and each of them starts with the selection instead of with a launch that
  // rotates and clears: 2 layers of a 128K request, two steps, 296 -> 292 us; a 31599-token
  // prompt with 16 tokens 4615 -> 4513.)
  const int64_t layout = plain ? decode_layer_layout(&o.cfg, bt->batch, bt->max_seq_len) : -1;
  if (layout >= 0 && o.clean_batch == bt->batch && o.clean_layout == layout) bt->workspace_clean = 1;
  o.forget_clean();
  const ts_stream_t stream = (ts_stream_t)c10::hip::getCurrentHIPStream().stream();
  const float *cos = (const float*)o.cos.data_ptr(), *sin = (const float*)o.sin.data_ptr();
  int32_t *sel = (int32_t*)o.sel.data_ptr(), *sel_pos = (int32_t*)o.sel_pos.data_ptr(),
          *sel_len = (int32_t*)o.sel_len.data_ptr();
  const int64_t sel_stride = o.sel.size(1), table_rows = o.cos.size(0), pool_rows = k_pool.size(0);
  void *kp = k_pool.data_ptr(), *vp = v_pool.data_ptr(), *ws = o.workspace.data_ptr();
  const size_t ws_bytes = (size_t)o.workspace.numel();
  const ts_config* cfg = &o.cfg;
  int code;
  Py_BEGIN_ALLOW_THREADS
  if (chunk)
    code = kv ? prefill_step(cfg, bt, kv, q, q_stride, kv_stride, (int32_t)rows, cos, sin, table_rows, kp, vp,
                             pool_rows, out, sel, sel_pos, sel_stride, sel_len, ws, ws_bytes, stream)
              : prefill_chunk(cfg, bt, q, (int32_t)rows, cos, sin, table_rows, kp, vp, pool_rows, out, sel, sel_pos,
                              sel_stride, sel_len, ws, ws_bytes, stream);
  else
    code = kv ? decode_step(cfg, bt, kv, q, q_stride, kv_stride, cos, sin, kp, vp, pool_rows, cache, out, sel, sel_pos, sel_stride, sel_len,
                            ws, ws_bytes, stream)
              : decode_layer(cfg, bt, q, cos, sin, kp, vp, pool_rows, cache, out, sel, sel_pos, sel_stride, sel_len, ws,
                             ws_bytes, stream);
  Py_END_ALLOW_THREADS
  if (code == TS_OK && plain) {
    o.clean_batch = bt->batch;
    o.clean_len = bt->max_seq_len;
    o.clean_layout = layout;
  }
  return code;
}

// run(q, k, v, out_cache_loc, k_pool, v_pool, bt, cache, out, pages, store, separate, rerun):
// the layer (store false) or the step; None when an earlier call's selection gave up (not with
// rerun), an error code of the library as an int, or (out, sel, sel_pos, sel_len).
PyObject* run(Runner* self, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 13) raise(PyExc_TypeError, "run() takes 13 arguments");
  Owned& o = *self->own;
  PyObject *q_o = args[0], *k_o = args[1], *v_o = args[2], *loc_o = args[3], *kp_o = args[4], *vp_o = args[5],
           *bt_o = args[6], *cache_o = args[7], *out_o = args[8], *pages_o = args[9];
  const bool store = args[10] == Py_True, separate = args[11] == Py_True, rerun = args[12] == Py_True;
  if (!rerun && fault_of(o) != 0) Py_RETURN_NONE;
  const bool chunk = o.max_rows > 0;
  const ts_config& cfg = o.cfg;
  const int64_t width = (int64_t)cfg.num_heads * cfg.head_dim, row = (int64_t)cfg.num_kv_heads * cfg.head_dim;

  Call call;
  fill_batch(o, bt_o, separate, rerun, &call);
  ts_batch& bt = call.bt;
  const int64_t B = bt.batch;
  const at::Tensor& q = need(q_o, "q", at::kBFloat16, chunk ? 2 : -1);
  int64_t rows = B;
  if (chunk) {
    rows = q.size(0);
    if (B != 1 || rows > o.max_rows) bad_value("one request, within the sizes this PrefillChunk was built for");
    if (q.size(1) != width) bad_value("q must be [rows, H*D]");
  } else if (q.numel() != B * width) {
    bad_value("q must hold B*H*D elements");
  }
  const at::Tensor& k_pool = check_pool(cfg, kp_o, "k_pool");
  const at::Tensor& v_pool = check_pool(cfg, vp_o, "v_pool");
  if (!chunk && k_pool.size(0) != v_pool.size(0)) bad_value("k_pool and v_pool must have the same shape");

  ts_new_kv kv{};
  ts_page_pool pool{};
  if (store) {
    const at::Tensor& k = need(k_o, "k", at::kBFloat16);
    const at::Tensor& v = need(v_o, "v", at::kBFloat16);
    int64_t slots = rows;
    if (pages_o != Py_None) {
      fill_pages(pages_o, &pool);
      kv.pages = &pool;
    } else {
      if (cfg.page_size != 1) bad_value("page_size " + std::to_string(cfg.page_size) + " needs a PagePool");
      const at::Tensor& loc = need(loc_o, "out_cache_loc", at::kInt, 1);
      slots = loc.size(0);
      kv.out_cache_loc = (const int32_t*)loc.data_ptr();
    }
    if (k.numel() != rows * row || v.numel() != rows * row || slots != rows)
      bad_value(chunk ? "k / v / out_cache_loc / table do not match the chunk"
                      : "k / v / out_cache_loc / table do not match the batch");
    kv.k = k.data_ptr();
    kv.v = v.data_ptr();
    kv.max_tokens = (int32_t)call.table_tokens;
  }

  ts_selcache cache{};
  const bool cached = cache_o != Py_None;
  if (cached) fill_cache(cfg, cache_o, B, &cache);

  PyObject* out_py;
  void* out_ptr;
  if (out_o != Py_None) {
    const at::Tensor& t = need(out_o, "out", at::kBFloat16);
    if (t.numel() != q.numel()) bad_value(chunk ? "out must hold rows*H*D elements" : "out must hold B*H*D elements");
    out_ptr = t.data_ptr();
    out_py = out_o;
    Py_INCREF(out_py);
  } else if (chunk) {
    at::Tensor t = at::empty_like(q);
    out_ptr = t.data_ptr();
    out_py = THPVariable_Wrap(std::move(t));
    if (!out_py) throw Raised{};
  } else {
    out_ptr = o.out.data_ptr();
    out_py = row_view(o.out, B);
  }
  const Ref out_ref(out_py);

  const int code = call_library(o, &bt, store ? &kv : nullptr, q.data_ptr(), 0, 0, rows, k_pool, v_pool,
                                cached ? &cache : nullptr, out_ptr, rerun);
  if (code != TS_OK) return PyLong_FromLong(code);
  // (tensors of the call's own: a caller may reshape or resize them in place)
  const Ref sel(row_view(o.sel, B)), sel_pos(row_view(o.sel_pos, B)), sel_len(row_view(o.sel_len, B));
  return PyTuple_Pack(4, out_py, sel.p, sel_pos.p, sel_len.p);
}

// serve(q, k, v, out_cache_loc, k_pool, v_pool, bt, cache, out, from, rows, separate): the step of a
// serving stack whose q, k and v are parts of one projection.  A DecodeLayer: one row per
// request, the output a fresh tensor.  A PrefillChunk: `rows` rows of the prompt part from
// `from` on, written to the same rows of `out`.  Returns as run() does, but the output alone.
PyObject* serve(Runner* self, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 12) raise(PyExc_TypeError, "serve() takes 12 arguments");
  Owned& o = *self->own;
  if (fault_of(o) != 0) Py_RETURN_NONE;
  const bool chunk = o.max_rows > 0, separate = args[11] == Py_True;
  const ts_config& cfg = o.cfg;
  const int64_t width = (int64_t)cfg.num_heads * cfg.head_dim, row = (int64_t)cfg.num_kv_heads * cfg.head_dim;
  Call call;
  fill_batch(o, args[6], separate, false, &call);
  ts_batch& bt = call.bt;
  const int64_t from = chunk ? as_long(args[9]) : 0;
  int64_t rows = bt.batch;
  if (chunk) {
    rows = as_long(args[10]);
    if (bt.batch != 1 || rows > o.max_rows) bad_value("one request, within the sizes this PrefillChunk was built for");
    if (from < 0 || rows < 1) bad_value("a chunk has at least one row");
  }
  // (a prompt's k and v may have rows after those of q, which are not read)
  if (!chunk && (tensor(args[1], "k").numel() != rows * row || tensor(args[2], "v").numel() != rows * row))
    bad_value("k / v do not match the batch");
  const Rows q = rows_of(args[0], "q", from, rows, width, false);
  Rows k = rows_of(args[1], "k", from, rows, row, false), v = rows_of(args[2], "v", from, rows, row, false);
  if (k.stride != v.stride) {
    if (k.stride != row) k = rows_of(args[1], "k", from, rows, row, true);
    if (v.stride != row) v = rows_of(args[2], "v", from, rows, row, true);
  }
  const at::Tensor& k_pool = check_pool(cfg, args[4], "k_pool");
  const at::Tensor& v_pool = check_pool(cfg, args[5], "v_pool");
  if (k_pool.size(0) != v_pool.size(0)) bad_value("k_pool and v_pool must have the same shape");
  if (cfg.page_size != 1) bad_value("page_size " + std::to_string(cfg.page_size) + " needs a PagePool");
  const Rows loc = slots_of(args[3], from, rows);
  ts_new_kv kv{k.ptr, v.ptr, (const int32_t*)loc.ptr, nullptr,
               (int32_t)call.table_tokens};
  ts_selcache cache{};
  const bool cached = args[7] != Py_None;
  if (cached) fill_cache(cfg, args[7], bt.batch, &cache);
  at::Tensor out;
  if (chunk) {
    out = need(args[8], "out", at::kBFloat16);
    if (out.dim() < 1 || out.numel() != out.size(0) * width || out.size(0) < from + rows)
      bad_value("out must hold the rows of q");
  } else {
    out = at::empty({rows, width}, o.out.options());
  }
  const int code = call_library(o, &bt, &kv, q.ptr, (int32_t)q.stride, (int32_t)k.stride, rows, k_pool, v_pool, cached ? &cache : nullptr,
                                (char*)out.data_ptr() + 2 * from * width);
  if (code != TS_OK) return PyLong_FromLong(code);
  if (chunk) {
    Py_INCREF(args[8]);
    return args[8];
  }
  return THPVariable_Wrap(std::move(out));
}

// prompt(q, k, v, out_cache_loc, k_pool, v_pool, bt, out, from, rows, chunk_rows): `rows` rows of a prompt
// part from `from` on, in chunks of chunk_rows, as serve() does them one by one.  The workspace is
// the call's own, in the order of the stream: a prompt's is larger than what a request would keep.
// False, and nothing done, where the memory for it (or for a copy of rows that lie otherwise) is not to be had.
PyObject* prompt(Runner* self, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 11) raise(PyExc_TypeError, "prompt() takes 11 arguments");
  Owned& o = *self->own;
  if (fault_of(o) != 0) Py_RETURN_NONE;
  const ts_config& cfg = o.cfg;
  const int64_t width = (int64_t)cfg.num_heads * cfg.head_dim, row = (int64_t)cfg.num_kv_heads * cfg.head_dim;
  Call call;
  fill_batch(o, args[6], false, false, &call);
  ts_batch& bt = call.bt;
  const int64_t from = as_long(args[8]), rows = as_long(args[9]), chunk_rows = as_long(args[10]);
  if (o.max_rows < 1 || bt.batch != 1 || chunk_rows > o.max_rows)
    bad_value("one request, within the sizes this PrefillChunk was built for");
  if (from < 0 || rows < 1 || rows > INT32_MAX || chunk_rows < 1) bad_value("a chunk has at least one row");
  const at::Tensor& k_pool = check_pool(cfg, args[4], "k_pool");
  const at::Tensor& v_pool = check_pool(cfg, args[5], "v_pool");
  if (k_pool.size(0) != v_pool.size(0)) bad_value("k_pool and v_pool must have the same shape");
  if (cfg.page_size != 1) bad_value("page_size " + std::to_string(cfg.page_size) + " needs a PagePool");
  const at::Tensor& out = need(args[7], "out", at::kBFloat16);
  if (out.dim() < 1 || out.numel() != out.size(0) * width || out.size(0) < from + rows)
    bad_value("out must hold the rows of q");
  Rows q, k, v, loc;
  const size_t bytes = prefill_prompt_bytes(&cfg, (int32_t)rows, (int32_t)chunk_rows, bt.max_seq_len);
  at::Tensor workspace;
  try {
    q = rows_of(args[0], "q", from, rows, width, false);
    k = rows_of(args[1], "k", from, rows, row, false), v = rows_of(args[2], "v", from, rows, row, false);
    if (k.stride != v.stride) {
      if (k.stride != row) k = rows_of(args[1], "k", from, rows, row, true);
      if (v.stride != row) v = rows_of(args[2], "v", from, rows, row, true);
    }
    loc = slots_of(args[3], from, rows);
    workspace = at::empty({(int64_t)bytes}, o.workspace.options());
  } catch (const c10::OutOfMemoryError&) {
    Py_RETURN_FALSE;
  }
  const ts_new_kv kv{k.ptr, v.ptr, (const int32_t*)loc.ptr, nullptr, (int32_t)call.table_tokens};
  const ts_stream_t stream = (ts_stream_t)c10::hip::getCurrentHIPStream().stream();
  int code;
  Py_BEGIN_ALLOW_THREADS
  code = prefill_prompt(&cfg, &bt, &kv, q.ptr, (int32_t)q.stride, (int32_t)k.stride, (int32_t)rows, (int32_t)chunk_rows,
                        (const float*)o.cos.data_ptr(), (const float*)o.sin.data_ptr(), o.cos.size(0),
                        k_pool.data_ptr(), v_pool.data_ptr(), k_pool.size(0),
                        (char*)out.data_ptr() + 2 * from * width, workspace.data_ptr(), bytes, stream);
  Py_END_ALLOW_THREADS
  if (code != TS_OK) return PyLong_FromLong(code);
  Py_INCREF(args[7]);
  return args[7];
}

// Runs `f`, with C++ exceptions turned into Python's.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const Raised&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

PyObject* runner_run(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&] { return run((Runner*)self, args, nargs); });
}

PyObject* runner_serve(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&] { return serve((Runner*)self, args, nargs); });
}

PyObject* runner_prompt(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&] { return prompt((Runner*)self, args, nargs); });
}

PyObject* runner_new(PyTypeObject* type, PyObject* args, PyObject*) {
  Py_buffer cfg;
  PyObject *ws, *cos, *sin, *out, *sel, *sel_pos, *sel_len, *fault;
  long long batch, max_seq_len, max_rows;
  if (!PyArg_ParseTuple(args, "y*OOOOOOOOLLL", &cfg, &ws, &cos, &sin, &out, &sel, &sel_pos, &sel_len, &fault, &batch,
                        &max_seq_len, &max_rows))
    return nullptr;
  PyObject* made = guarded([&]() -> PyObject* {
    if (cfg.len != (Py_ssize_t)sizeof(ts_config)) bad_value("config of another size");
    Ref self(type->tp_alloc(type, 0));
    Owned* o = new Owned();
    ((Runner*)self.p)->own = o;
    memcpy(&o->cfg, cfg.buf, sizeof(ts_config));
    const ts_config& c = o->cfg;
    const int64_t width = (int64_t)c.num_heads * c.head_dim, max_sel = (int64_t)c.n_init + c.top_k + c.n_local;
    o->workspace = need(ws, "workspace", at::kByte);
    o->cos = need(cos, "cos", at::kFloat, 2);
    o->sin = need(sin, "sin", at::kFloat, 2);
    if (o->cos.sizes() != o->sin.sizes() || o->cos.size(0) < 1 || o->cos.size(1) != c.head_dim)
      bad_value("cos / sin must both be [rows, head_dim]");
    if (out != Py_None) {
      o->out = need(out, "out", at::kBFloat16, 2);
      if (o->out.size(0) < batch || o->out.size(1) != width) bad_value("out must hold the batch's rows of H*D elements");
    }
    o->sel = need(sel, "sel", at::kInt, 2);
    o->sel_pos = need(sel_pos, "sel_pos", at::kInt, 2);
    o->sel_len = need(sel_len, "sel_len", at::kInt, 1);
    if (o->sel.size(0) < batch || o->sel.size(1) < max_sel || o->sel_pos.sizes() != o->sel.sizes() ||
        o->sel_len.size(0) < batch)
      bad_value("sel / sel_pos / sel_len must hold the batch's lists of " + std::to_string(max_sel));
    o->fault = tensor(fault, "fault");
    if (o->fault.scalar_type() != at::kInt || o->fault.numel() != 1 || !o->fault.is_pinned())
      bad_value("fault must be one int32 word of pinned host memory");
    o->batch = batch;
    o->max_seq_len = max_seq_len;
    o->max_rows = max_rows;
    Py_INCREF(self.p);
    return self.p;
  });
  PyBuffer_Release(&cfg);
  return made;
}

void runner_dealloc(PyObject* self) {
  Owned* o = ((Runner*)self)->own;
  delete o;
  PyTypeObject* type = Py_TYPE(self);
  type->tp_free(self);
  Py_DECREF(type);
}

PyObject* get_clean(PyObject* self, void*) {
  const Owned& o = *((Runner*)self)->own;
  if (o.clean_batch < 0) Py_RETURN_NONE;
  return Py_BuildValue("(LL)", (long long)o.clean_batch, (long long)o.clean_len);
}
int set_clean(PyObject* self, PyObject* value, void*) {
  Owned& o = *((Runner*)self)->own;
  long long b = -1, n = -1;
  if (value != Py_None && !(value && PyArg_ParseTuple(value, "LL", &b, &n))) return -1;
  if (value == Py_None) {  // other calls use the workspace from here on
    o.shared = o.shared || capturing();
    o.forget_clean();
    return 0;
  }
  o.clean_batch = b;
  o.clean_len = n;
  o.clean_layout = b >= 1 && n >= 1 ? decode_layer_layout(&o.cfg, (int32_t)b, (int32_t)n) : -1;
  return 0;
}

PyObject* get_shared(PyObject* self, void*) { return PyBool_FromLong(((Runner*)self)->own->shared); }
int set_shared(PyObject* self, PyObject* value, void*) {
  const int yes = value ? PyObject_IsTrue(value) : 0;
  if (yes < 0) return -1;
  ((Runner*)self)->own->shared = yes != 0;
  return 0;
}

PyMethodDef runner_methods[] = {
    {"run", (PyCFunction)(void (*)(void))runner_run, METH_FASTCALL, nullptr},
    {"serve", (PyCFunction)(void (*)(void))runner_serve, METH_FASTCALL, nullptr},
    {"prompt", (PyCFunction)(void (*)(void))runner_prompt, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef runner_getset[] = {{"clean", get_clean, set_clean, nullptr, nullptr},
                               {"shared", get_shared, set_shared, nullptr, nullptr},
                               {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyType_Slot runner_slots[] = {{Py_tp_new, (void*)runner_new}, {Py_tp_dealloc, (void*)runner_dealloc},
                              {Py_tp_methods, runner_methods}, {Py_tp_getset, runner_getset}, {0, nullptr}};
PyType_Spec runner_spec = {"_ts_bind.Runner", sizeof(Runner), 0, Py_TPFLAGS_DEFAULT, runner_slots};

// connect(addresses): the library's entry points, in this order (the last two stay where they are
// not given).
PyObject* connect(PyObject*, PyObject* args) {
  unsigned long long a, b, c, d, e, f = (uintptr_t)prefill_prompt, g = (uintptr_t)prefill_prompt_bytes;
  if (!PyArg_ParseTuple(args, "KKKKK|KK", &a, &b, &c, &d, &e, &f, &g)) return nullptr;
  prefill_prompt = (PromptFn)(uintptr_t)f;
  prefill_prompt_bytes = (PromptBytesFn)(uintptr_t)g;
  decode_layer = (LayerFn)(uintptr_t)a;
  decode_step = (StepFn)(uintptr_t)b;
  prefill_chunk = (ChunkFn)(uintptr_t)c;
  prefill_step = (ChunkStepFn)(uintptr_t)d;
  decode_layer_layout = (LayoutFn)(uintptr_t)e;
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {{"connect", connect, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ts_bind", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ts_bind(void) {
  if (!intern_names()) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  PyObject* type = m ? PyType_FromSpec(&runner_spec) : nullptr;
  if (!type || PyModule_AddObject(m, "Runner", type) < 0) {
    Py_XDECREF(type);
    Py_XDECREF(m);
    return nullptr;
  }
  return m;
}
