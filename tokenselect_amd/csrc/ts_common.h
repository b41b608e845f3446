// Shared host/device helpers for libtokenselect_hip.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tokenselect.h"
#include "ts_share.h"

namespace ts {

// ---------------------------------------------------------------- host side
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);
int validate_config(const ts_config* cfg);
int validate_batch(const ts_config* cfg, const ts_batch* bt);
// A row stride in elements: 0 (contiguous rows of `width`), or a multiple of 8 of at least `width`.
int check_row_stride(int64_t stride, int64_t width, const char* who);
bool group_supported(int num_kv_heads, int group);

#define TS_REQUIRE(cond, code, ...)                     \
  do {                                                  \
    if (!(cond)) return ::ts::fail((code), __VA_ARGS__); \
  } while (0)

#define TS_TRY(expr)            \
  do {                          \
    int _rc = (expr);           \
    if (_rc != TS_OK) return _rc; \
  } while (0)

// Device buffers are read and written with 16-byte vector accesses and 8-byte atomics:
// what hipMalloc and the framework allocators return is aligned far beyond that, a view
// at an odd offset is not, and would fault the device instead of failing a call.
#define TS_REQUIRE_ALIGNED(ptr, bytes, what)                                                   \
  TS_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & ((bytes)-1)) == 0, TS_EINVAL,                  \
             "%s must be aligned to %d bytes", what, (int)(bytes))

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }
static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Candidate rows per workgroup of the scoring pass, shared by the launcher,
// the statistics merge and the workspace query.
int score_tokens_per_block(int64_t total_candidates, int num_heads);

// Words the rotation kernel clears on the side: `count` pieces of `words` 32-bit
// words, `stride` words apart (all zero: nothing to clear).
struct ZeroRegion {
  uint32_t* base = nullptr;
  int64_t stride = 0;
  int words = 0;
  int count = 0;
};
// What one such launch clears: up to four regions.
constexpr int kZeroRegions = 4;
struct ZeroSet {
  ZeroRegion r[kZeroRegions];
  int used = 0;
  bool overflow = false;  // a region did not fit: the launchers refuse such a set
  void add(const ZeroRegion& region) {
    if (region.count <= 0 || region.words <= 0) return;
    if (used < kZeroRegions)
      r[used++] = region;
    else
      overflow = true;
  }
  int64_t total() const {
    int64_t t = 0;
    for (int i = 0; i < used; ++i) t += (int64_t)r[i].count * r[i].words;
    return t;
  }
};
// Wavefront `wave` of `waves` clears its share of a region: word by word (16 bytes at a time)
// where the pieces touch, else a wavefront per piece, beginning with wavefront `from`.  No index is divided by the length of a
// piece: with a 64-bit division and remainder per word the 0.3 MB of one request's selection cost
// every workgroup of the launch some 600 instructions ahead of its first load.
__device__ __forceinline__ void clear_region(const ZeroRegion& z, uint32_t wave, uint32_t waves, uint32_t from) {
  const uint32_t lane = threadIdx.x & 63u;
  if (z.count == 1 || z.stride == z.words) {
    const int64_t total = (int64_t)z.count * z.words, step = (int64_t)waves * 64;
    int64_t done = 0;
    if (((uintptr_t)z.base & 15u) == 0) {
      done = total & ~(int64_t)3;
      for (int64_t w = (int64_t)wave * 64 + lane; w < done >> 2; w += step)
        *(uint4*)(z.base + 4 * w) = make_uint4(0u, 0u, 0u, 0u);
    }
    for (int64_t w = done + (int64_t)wave * 64 + lane; w < total; w += step) z.base[w] = 0u;
  } else {
    uint32_t first = wave + from;
    first -= first >= waves ? waves : 0u;
    for (uint32_t piece = first; piece < (uint32_t)z.count; piece += waves) {
      uint32_t* const at = z.base + (int64_t)piece * z.stride;
      for (int w = (int)lane; w < z.words; w += 64) at[w] = 0u;
    }
  }
}
__device__ __forceinline__ void clear_regions(const ZeroSet& zero, uint32_t wave, uint32_t waves) {
#pragma unroll
  for (int i = 0; i < kZeroRegions; ++i) {
    if (i >= zero.used) break;
    // (another first wavefront per region: a piece each, not all of them to the same few)
    clear_region(zero.r[i], wave, waves, (uint32_t)i * (waves >> 2));
  }
}
// Chunk fingerprint (ts_prefill.hip) with the same side job as launch_rope: the
// regions are cleared by the same launch.
// The K/V rows of a prefill chunk, stored by the fingerprint launch on the side (as
// kv_store_chunk_kernel stores them): slots chosen by the caller, one per row.
struct ChunkStore {
  const uint4* k;  // [rows, Hkv*D] bf16 as 16-byte pieces
  const uint4* v;
  const int32_t* loc;
  uint4* k_pool;
  uint4* v_pool;
  int64_t pool_rows;
  int32_t* table;    // the request's row
  int32_t* seq_len;  // the request's length word
  int rows, row_vec, max_tokens;
  int kv_stride;     // 16-byte pieces between rows of k, and of v
  int workgroups;    // of the launch that store (set by the launcher)
};
int launch_fingerprint(const ts_config* cfg, const void* q, int q_stride, int32_t rows, const float* cos_table,
                       const float* sin_table, int64_t table_rows, void* qf, const ZeroSet& zero,
                       hipStream_t stream, const ChunkStore* store = nullptr);
// The new token's K/V rows of a decode step, for whatever launch stores them (store_step): slots
// chosen by the caller, one per request.
struct StepStore {
  const uint4* k;  // [B, Hkv*D] bf16 as 16-byte pieces
  const uint4* v;
  const int32_t* loc;
  uint4* k_pool;
  uint4* v_pool;
  int64_t pool_rows;
  int32_t* table;
  int64_t table_stride;
  int32_t* seq_lens;
  int row_vec;     // 16-byte pieces per row
  int kv_stride;   // 16-byte pieces between rows of k, and of v
  int max_tokens;
  // With a page pool (free_pages != NULL; loc is not read): the slots come from the table and
  // the pool by the plan of the batch (ts_pages.h).
  const int32_t* free_pages;
  int32_t* free_count;
  uint32_t* ticket;
  int page_shift;
};
// Whether a request's new token is stored: a slot of the pool, and a table with room at that length.
// (Asked by everyone who places one: what a call does must not depend on which launch that is.)
// (Both bounds are below 2^31: a negative one of the two is beyond them.)
__device__ __forceinline__ bool append_fits(int slot, int len, int64_t pool_rows, int max_tokens) {
  return (uint32_t)slot < (uint32_t)pool_rows && (uint32_t)len < (uint32_t)max_tokens;
}
// What a step's store leaves to be written when nobody reads the lengths any more: one per request,
// noted by the selection that stored the rows and knows the length (ts_score.hip), written by
// the attention after it.
struct StepCommit {
  int4* notes;  // [B] (length or -1: nothing, table index, table entry or -1: none, pages taken by the launch)
  int batch;    // 0: nothing to write
  int32_t* table;
  int64_t table_stride;
  int32_t* seq_lens;
  int32_t* free_count;  // NULL: no page pool
};
constexpr int kCommitBatch = 64;  // requests that one wavefront writes for

// x_stride: elements between the rows of x (out is contiguous).  store: rides in the launch.  zero, more: what it
// clears, `more` in one piece (words == 0: nothing).
int launch_rope(const void* x, int64_t x_stride, void* out, const float* cos_table, const float* sin_table,
                const int64_t* position_ids, int64_t table_rows, int64_t rows, int heads, int dim,
                const ZeroSet& zero, hipStream_t stream, const StepStore* store = nullptr, int store_batch = 0,
                const ZeroRegion& more = ZeroRegion{});

// Selection-cache decision (ts_selcache.hip); gave_up_len: see ts_batch.rerun (NULL: an
// ordinary step).
int launch_selcache(const ts_config* cfg, const ts_batch* bt, const void* qf, const ts_selcache* cache,
                    int32_t* hit, const int32_t* gave_up_len, hipStream_t stream);

// The fingerprint rotation of a decode step (one query row per request, q_cos / q_sin the
// [D] table rows of its position) and the cache decision in one launch, which also clears
// the regions of `zero`.
int launch_rope_selcache(const ts_config* cfg, const ts_batch* bt, const void* q, int q_stride, void* qf,
                         const float* q_cos, const float* q_sin, const ts_selcache* cache, int32_t* hit,
                         const int32_t* gave_up_len, const ZeroSet& zero, hipStream_t stream,
                         const StepStore* store = nullptr);

// The selection of a call whose every request attends to all its tokens, written by the store
// that precedes it (per-token tables only): sel and sel_pos of all positions, the new ones
// included, and sel_len; and the attention's tickets cleared.
struct DenseList {
  int32_t* sel;  // NULL: no list
  int32_t* sel_pos;
  int64_t sel_stride;
  int32_t* sel_len;
  uint32_t* clear;
  int clear_per_req;
  int max_seq_len;
};

// What ts_kv_store requires of its arguments.
int check_kv_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride, const int32_t* out_cache_loc,
                   const ts_page_pool* pages, const void* k_pool, const void* v_pool, int64_t pool_rows,
                   const int32_t* table, int64_t table_stride, const int32_t* seq_lens, int32_t batch,
                   int32_t max_tokens);
StepStore step_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                     const int32_t* out_cache_loc, const ts_page_pool* pages, void* k_pool, void* v_pool,
                     int64_t pool_rows, int32_t* table, int64_t table_stride, int32_t* seq_lens, int32_t max_tokens);
int launch_kv_store(const StepStore& st, int32_t batch, hipStream_t stream, const DenseList* list = nullptr);
// ts_kv_store_chunk for rows of k and v that lie row_stride elements apart.
int launch_kv_store_chunk(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                          const int32_t* out_cache_loc, const ts_page_pool* pages, int32_t rows, void* k_pool,
                          void* v_pool, int64_t pool_rows, int32_t* table, int32_t* seq_len, int32_t max_tokens,
                          hipStream_t stream);
// What it requires of its arguments, and the rows for whatever launch stores them.
int check_kv_store_chunk(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                         const int32_t* out_cache_loc, const ts_page_pool* pages, int32_t rows, const void* k_pool,
                         const void* v_pool, int64_t pool_rows, const int32_t* table, const int32_t* seq_len,
                         int32_t max_tokens);
ChunkStore chunk_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                       const int32_t* out_cache_loc, int32_t rows, void* k_pool, void* v_pool, int64_t pool_rows,
                       int32_t* table, int32_t* seq_len, int32_t max_tokens);
// What launch_fingerprint requires of its arguments.
int check_fingerprint(const void* q, int32_t rows, const float* cos_table, const float* sin_table,
                      int64_t table_rows, const void* qf, int32_t n_local);
// A chunk that attends to all tokens: its gather reads the table, and stores the chunk's rows and
// writes the list itself; the attention after it, which reads neither, writes the length.
struct PrefillDense {
  const int32_t* table;  // in pages of 1 << page_shift
  int page_shift;
  int32_t* seq_len;      // before the append, where there is one
  int32_t* sel;          // the selection that is left behind
  int32_t* sel_pos;
  int32_t* sel_len;
  int list_bound;        // entries that are there to be read, and the most that are listed
  ChunkStore store;      // k == NULL: no append, the length counts the chunk already
};
// Several chunks of a prompt: of chunk_rows rows each, the last one of what is left.
struct PromptChunks {
  int rows, chunk_rows, chunks;
  int32_t* lens;         // [chunks] the length after each, written by the fingerprints' launch
  uint32_t* counters;    // what their selections count into, cleared by it
  size_t counters_stride;
  int counter_words;
};
// Their fingerprints [chunks, H, D], and the store of all their rows (lengths left alone).
int launch_prompt_fingerprint(const ts_config* cfg, const void* q, int q_stride, const float* cos_table,
                              const float* sin_table, int64_t table_rows, void* qf, const PromptChunks& pc,
                              const ChunkStore& store, hipStream_t stream);
// ts_sparse_prefill_attn for several chunks, each over its list; workspace: a chunk's after the other.
int launch_prefill_attn_chunks(const ts_config* cfg, const void* q, int q_stride, int32_t rows, int32_t chunk_rows,
                               const void* k_pool, const void* v_pool, int64_t pool_rows, const int32_t* sel,
                               int64_t sel_stride, const int32_t* sel_len, int32_t max_sel_len, void* out,
                               void* workspace, size_t workspace_bytes, hipStream_t stream,
                               const PrefillDense* dense = nullptr, void* cut_space = nullptr);
// ts_sparse_prefill_attn for query rows that lie q_stride elements apart.
int launch_prefill_attn(const ts_config* cfg, const void* q, int q_stride, int32_t rows, const void* k_pool,
                        const void* v_pool, int64_t pool_rows, const int32_t* sel, const int32_t* sel_len,
                        int32_t max_sel_len, void* out, void* workspace, size_t workspace_bytes, hipStream_t stream,
                        const PrefillDense* dense = nullptr, void* cut_space = nullptr);
// Space for the pieces of jobs that the attention's workgroups of 256 columns share (ts_prefill_shared.hip), and
// whether so many rows over so many keys would use it.
size_t prefill_cut_bytes();
bool prefill_cuts_pay(int num_heads, int num_kv_heads, int rows, int chunk_rows, int keys);

// Sparse decode attention (ts_attn.hip).  The kernel counts its workgroups in per
// (request, KV head) tickets inside the workspace, which must be zero at launch:
// tickets_clear = false makes the launcher clear them first, true says an earlier
// kernel of the stream already did (attn_tickets() tells it where they are).
uint32_t* attn_tickets(void* workspace);
size_t attn_workspace_bytes(const ts_config* cfg, int batch, int max_sel_len);
// Tickets per request (the words to clear).
int attn_tickets_per_request(const ts_config* cfg);
// clear_after: regions that the kernel clears on the side (the counters of the stream's
// next selection), or NULL.
// dense: a decode step whose requests attend to all their tokens, in this launch alone; `sel` is
// then the table in pages of cfg's size and sel_len the lengths before the step's append.
struct AttnDense {
  int32_t* sel;      // the selection that is left behind: every position, the new one included
  int32_t* sel_pos;
  int64_t sel_stride;
  int32_t* sel_len;
  int list_bound;    // entries that are there to be read, whatever the length
  // The new tokens (loc == NULL: none, the lengths count them already), one per request.
  const int32_t* loc;
  const uint16_t* k;  // [B, Hkv*128] bf16, rows kv_stride elements apart
  const uint16_t* v;
  int64_t k_from_pool, v_from_pool;  // elements from the pools to them
  int kv_stride;
  int32_t* table;    // sel and sel_len of the launch, to be written
  int32_t* seq_lens;
  int max_tokens;
};
// How a call's splits are shared on the current device, with words in `bytes` bytes (words == NULL: not at all).
AttnShare attn_share(const ts_config* cfg, int batch, int max_sel_len, void* words, size_t bytes);
int launch_attn(const ts_config* cfg, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                int64_t pool_rows, const int32_t* sel, int64_t sel_stride, const int32_t* sel_len,
                int batch, int max_sel_len, void* out, void* workspace, bool tickets_clear,
                hipStream_t stream, const ZeroSet* clear_after = nullptr, const AttnDense* dense = nullptr,
                const StepCommit* commit = nullptr, const AttnShare* share = nullptr);

constexpr float kNegBig = -3.0e38f;  // finite stand-in for -inf in running maxima

// -------------------------------------------------------------- device side
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// Round-to-nearest-even, NaN kept quiet: the rounding torch applies on .to(bfloat16).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// Two floats to packed bf16, round to nearest even, in one v_cvt_pk_bf16_f32.
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
constexpr int kRowRor1 = 0x121, kRowRor2 = 0x122, kRowRor4 = 0x124, kRowRor8 = 0x128;

// Sum over the 16 lanes of a DPP row; every lane of the row gets the total.
__device__ __forceinline__ float row16_sum(float x) {
  x += dpp_move<kRowRor8>(x);
  x += dpp_move<kRowRor4>(x);
  x += dpp_move<kRowRor2>(x);
  x += dpp_move<kRowRor1>(x);
  return x;
}

// sin and cos of an angle of up to some 1e5 radians: two-constant reduction by
// 2 pi (hi + lo parts, each product exact inside the FMA), then the hardware
// functions on [-pi, pi].
__device__ __forceinline__ void sincos_reduced(float x, float& sn, float& cs) {
  const float k = rintf(x * 0.15915494309189535f);
  float r = fmaf(-k, 6.2831854820251465f, x);
  r = fmaf(-k, -1.7484555e-07f, r);
  sn = __sinf(r);
  cs = __cosf(r);
}

// One element of the scoring query's rotation (RotaryEmbedding.apply_rotary_pos_emb,
// tr.py:98-107): own * cos + (+-other) * sin, where `other` is the element 64 dims away and
// enters negated for the lower half.  Products and the sum are rounded one by one (no FMA
// contraction), which is what the reference's elementwise torch expression does.
__device__ __forceinline__ float rotate_element(float own, float other, float cs, float sn, bool lower) {
#pragma clang fp contract(off)
  const float a = own * cs;
  const float b = (lower ? -other : other) * sn;
  return a + b;
}

// Merge two (max, sum-of-exp) softmax partials.
__device__ __forceinline__ void softmax_merge(float& m, float& l, float m2, float l2) {
  float mm = fmaxf(m, m2);
  l = l * __expf(m - mm) + l2 * __expf(m2 - mm);
  m = mm;
}

__device__ __forceinline__ void row16_softmax_merge(float& m, float& l) {
  softmax_merge(m, l, dpp_move<kRowRor8>(m), dpp_move<kRowRor8>(l));
  softmax_merge(m, l, dpp_move<kRowRor4>(m), dpp_move<kRowRor4>(l));
  softmax_merge(m, l, dpp_move<kRowRor2>(m), dpp_move<kRowRor2>(l));
  softmax_merge(m, l, dpp_move<kRowRor1>(m), dpp_move<kRowRor1>(l));
}

// Per-request geometry of the selection, evaluated on the device so that no
// host synchronisation is needed (tr.py:376-378, 424-426).
struct ReqGeom {
  int seq_len;  // L
  int k;        // per-request top-k
  int n;        // candidates = L - n_init - n_local (0 when dense)
  bool dense;   // n_init + k + n_local >= L
};

// seq_lens[b] is clamped to the host's max_seq_len, the bound every buffer and
// grid was sized for.
__device__ __forceinline__ ReqGeom geometry_of_length(int length, const int32_t* k_per_req, int b, int n_init,
                                                      int n_local, int top_k, int max_seq_len) {
  ReqGeom g;
  g.seq_len = min(max(length, 0), max_seq_len);
  int k = k_per_req ? k_per_req[b] : top_k;
  g.k = k < 0 ? 0 : (k > top_k ? top_k : k);
  g.dense = (n_init + g.k + n_local >= g.seq_len);
  g.n = g.dense ? 0 : g.seq_len - n_init - n_local;
  return g;
}

__device__ __forceinline__ ReqGeom request_geometry(const int32_t* seq_lens, const int32_t* k_per_req,
                                                    int b, int n_init, int n_local, int top_k,
                                                    int max_seq_len) {
  return geometry_of_length(seq_lens[b], k_per_req, b, n_init, n_local, top_k, max_seq_len);
}

// Logical position -> physical KV slot through the (paged) table; page sizes are
// powers of two.  The slot is clamped to the pool so that a corrupt table cannot
// fault the GPU.
__device__ __forceinline__ uint32_t lookup_slot(const int32_t* tab, int pos, int page_size,
                                                int page_shift, uint32_t pool_rows) {
  const uint32_t slot =
      ((uint32_t)tab[pos >> page_shift] << page_shift) + (uint32_t)(pos & (page_size - 1));
  return slot < pool_rows ? slot : pool_rows - 1;
}

static inline int page_shift_of(int page_size) {
  if (page_size <= 0 || (page_size & (page_size - 1))) return -1;
  int s = 0;
  while ((1 << s) < page_size) ++s;
  return s;
}

}  // namespace ts
