// KV store and token-table append for a decode step
// (patched_radix_attention_store_kv_cache tr.py:844-854, add_k_cache tr.py:332-336).
#include "ts_pages.h"
#include "ts_store.h"

namespace ts {

__global__ __launch_bounds__(256) void kv_store_kernel(StepStore st) { store_step(st, blockIdx.x, gridDim.x); }

// One workgroup per request: the same, at a slot that the caller chose, and (where every request of
// the step attends to all its tokens) the request's selection (list), the table itself.  Bound by
// three dependent memory round trips (length and slot, stores, the length's store); the table
// entries are asked for with the first.  A dense step then has two launches, this (2.2 us) and the attention, where it had
// a store (1.7), a selection kernel or a rotation and a list (3.3 to 4.6) and the attention:
// 8 layers of a 2003-token request, two steps, 320 -> 261 us; 2 layers of a 300-token prompt
// with 8 tokens 430 -> 368 us.  (Once the caller can say that the attention's tickets are zero, the
// attention stores the row and writes the list itself, and this form serves the calls before.)
constexpr int kListThreads = 1024;  // one request's few thousand entries in a handful of steps
constexpr int kListAhead = 4;       // table entries a thread asks for before it knows the length

__global__ __launch_bounds__(kListThreads) void kv_store_list_kernel(StepStore st, DenseList list) {
  const uint4 *k = st.k, *v = st.v;
  uint4 *k_pool = st.k_pool, *v_pool = st.v_pool;
  const int64_t pool_rows = st.pool_rows;
  const int row_vec = st.row_vec, kv_stride = st.kv_stride, max_tokens = st.max_tokens;
  const int b = blockIdx.x;
  // The new rows are asked for together with the slot and the length, not after them: the
  // kernel is two memory round trips long instead of three.
  const int first = threadIdx.x;
  uint4 k0 = make_uint4(0u, 0u, 0u, 0u), v0 = k0;
  if (first < row_vec) {
    k0 = k[(size_t)b * kv_stride + first];
    v0 = v[(size_t)b * kv_stride + first];
  }
  const int slot = st.loc[b];
  const int len = st.seq_lens[b];
  int32_t* const tab = st.table + (int64_t)b * st.table_stride;
  int32_t ahead[kListAhead];
  const int known = min(list.max_seq_len, max_tokens);  // entries there to be read: a table holds max_tokens
#pragma unroll
  for (int i = 0; i < kListAhead; ++i) {
    const int pos = first + i * kListThreads;
    ahead[i] = pos < known ? tab[pos] : 0;
  }
  const bool ok = append_fits(slot, len, pool_rows, max_tokens);
  if (ok) {
    if (first < row_vec) {
      k_pool[(size_t)slot * row_vec + first] = k0;
      v_pool[(size_t)slot * row_vec + first] = v0;
    }
    for (int i = first + blockDim.x; i < row_vec; i += blockDim.x) {
      k_pool[(size_t)slot * row_vec + i] = k[(size_t)b * kv_stride + i];
      v_pool[(size_t)slot * row_vec + i] = v[(size_t)b * kv_stride + i];
    }
  }
  const int L = min(max(ok ? len + 1 : len, 0), list.max_seq_len);
  int32_t* const sel = list.sel + (int64_t)b * list.sel_stride;
  int32_t* const sel_pos = list.sel_pos + (int64_t)b * list.sel_stride;
  auto emit = [&](int pos, int32_t entry) {
    const uint32_t s = (uint32_t)(ok && pos == len ? slot : entry);
    sel_pos[pos] = pos;
    sel[pos] = (int32_t)(s < (uint32_t)pool_rows ? s : (uint32_t)pool_rows - 1);
  };
#pragma unroll
  for (int i = 0; i < kListAhead; ++i) {
    const int pos = first + i * kListThreads;
    if (pos < L) emit(pos, pos < known ? ahead[i] : (ok && pos == len ? slot : tab[pos]));
  }
  for (int pos = first + kListAhead * kListThreads; pos < L; pos += kListThreads)
    emit(pos, ok && pos == len ? slot : tab[pos]);
  for (int i = first; i < list.clear_per_req; i += kListThreads)
    list.clear[(size_t)b * list.clear_per_req + i] = 0u;
  if (first == 0) list.sel_len[b] = L;
  __syncthreads();
  if (threadIdx.x == 0 && ok) {
    tab[len] = slot;
    st.seq_lens[b] = len + 1;
  }
}

// Chunked prefill (tr.py:725-733): ts_store.h has the counted form's body, which the
// fingerprint launch of a chunk can also run on the side.
constexpr int kChunkRowsPerWg = 256 / kChunkThreadsPerRow;  // few workgroups, few counts on one word

template <bool COUNTED>
__global__ __launch_bounds__(256) void kv_store_chunk_kernel(ChunkStore cs) {
  store_chunk_rows<COUNTED>(cs, (int)blockIdx.x, 256);
}

__global__ void seq_len_add_kernel(int32_t* seq_len, int rows, int max_tokens) {
  const int len = *seq_len + rows;
  *seq_len = len > max_tokens ? max_tokens : len;
}


// Where row r of a chunk goes when the request's table is paged: positions
// len .. len + rows - 1 fill the request's last page and then fresh pages from the
// top of the free list, in order.  The same arithmetic serves every workgroup and
// the commit.
struct ChunkPlan {
  int len, count;
  int first_new;  // first page index of the table that does not exist yet
  int stored;     // rows that fit the table and the pages left
  int taken;      // pages taken from the list
};

__device__ __forceinline__ ChunkPlan make_chunk_plan(const int32_t* seq_len, const PagePool& pool,
                                                     int rows, int max_tokens, int page_shift) {
  ChunkPlan c;
  c.len = min(max(*seq_len, 0), max_tokens);
  c.count = max(*pool.free_count, 0);
  const int page = 1 << page_shift;
  c.first_new = (c.len + page - 1) >> page_shift;
  const int fit = min(rows, max_tokens - c.len);
  const int wanted = fit > 0 ? ((c.len + fit - 1) >> page_shift) - c.first_new + 1 : 0;
  c.taken = min(max(wanted, 0), c.count);
  c.stored = c.taken == max(wanted, 0) ? fit : max(((c.first_new + c.taken) << page_shift) - c.len, 0);
  return c;
}

__global__ __launch_bounds__(256) void kv_store_chunk_paged_kernel(
    const uint4* __restrict__ k, const uint4* __restrict__ v, uint4* __restrict__ k_pool,
    uint4* __restrict__ v_pool, uint32_t pool_rows, int32_t* table, int32_t* seq_len, int rows,
    int row_vec, int kv_stride, int max_tokens, int page_shift, PagePool pool) {
  const int r = blockIdx.x;
  const ChunkPlan c = make_chunk_plan(seq_len, pool, rows, max_tokens, page_shift);
  if (r < c.stored) {
    const int at = c.len + r;
    const int pg = at >> page_shift;
    const bool fresh = pg >= c.first_new;
    const int32_t page = fresh ? pool.free_pages[c.count - 1 - (pg - c.first_new)] : table[pg];
    uint32_t slot = ((uint32_t)page << page_shift) + (uint32_t)(at & ((1 << page_shift) - 1));
    slot = slot < pool_rows ? slot : pool_rows - 1;
    for (int i = threadIdx.x; i < row_vec; i += blockDim.x) {
      k_pool[(size_t)slot * row_vec + i] = k[(size_t)r * kv_stride + i];
      v_pool[(size_t)slot * row_vec + i] = v[(size_t)r * kv_stride + i];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 &&
      __hip_atomic_fetch_add(pool.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
          gridDim.x) {
    for (int j = 0; j < c.taken; ++j) table[c.first_new + j] = pool.free_pages[c.count - 1 - j];
    *seq_len = c.len + c.stored;
    *pool.free_count = c.count - c.taken;
    __hip_atomic_store(pool.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

static int check_pool_arg(const ts_config* cfg, const int32_t* out_cache_loc, const ts_page_pool* pages,
                          const char* who) {
  if (pages) {
    TS_REQUIRE(pages->free_pages && pages->free_count && pages->ticket, TS_EINVAL,
               "%s: page pool has a NULL array", who);
    return TS_OK;
  }
  TS_REQUIRE(cfg->page_size == 1, TS_EINVAL,
             "%s: page_size %d needs a page pool (without one the caller's out_cache_loc is appended to "
             "a per-token table, page_size 1)",
             who, cfg->page_size);
  TS_REQUIRE(out_cache_loc != nullptr, TS_EINVAL, "%s: NULL out_cache_loc and no page pool", who);
  return TS_OK;
}

int check_kv_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride, const int32_t* out_cache_loc,
                   const ts_page_pool* pages, const void* k_pool, const void* v_pool, int64_t pool_rows,
                   const int32_t* table, int64_t table_stride, const int32_t* seq_lens, int32_t batch,
                   int32_t max_tokens) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(k && v && k_pool && v_pool && table && seq_lens, TS_EINVAL,
             "ts_kv_store: NULL tensor argument");
  TS_REQUIRE_ALIGNED(k, 16, "k");
  TS_REQUIRE_ALIGNED(v, 16, "v");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(v_pool, 16, "v_pool");
  TS_TRY(check_pool_arg(cfg, out_cache_loc, pages, "ts_kv_store"));
  TS_REQUIRE(batch >= 1 && pool_rows >= 1 && pool_rows <= 0x7fffffffLL && max_tokens >= 1, TS_EINVAL,
             "ts_kv_store: batch=%d pool_rows=%lld max_tokens=%d out of range", batch,
             (long long)pool_rows, max_tokens);
  TS_REQUIRE(batch == 1 || table_stride * (int64_t)cfg->page_size >= max_tokens, TS_EINVAL,
             "ts_kv_store: table_stride %lld x page_size %d < max_tokens %d", (long long)table_stride,
             cfg->page_size, max_tokens);
  return check_row_stride(row_stride, (int64_t)cfg->num_kv_heads * cfg->head_dim, "ts_kv_store");
}

StepStore step_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                     const int32_t* out_cache_loc, const ts_page_pool* pages, void* k_pool, void* v_pool,
                     int64_t pool_rows, int32_t* table, int64_t table_stride, int32_t* seq_lens, int32_t max_tokens) {
  StepStore st{};
  st.k = (const uint4*)k;
  st.v = (const uint4*)v;
  st.loc = out_cache_loc;
  st.k_pool = (uint4*)k_pool;
  st.v_pool = (uint4*)v_pool;
  st.pool_rows = pool_rows;
  st.table = table;
  st.table_stride = table_stride;
  st.seq_lens = seq_lens;
  st.row_vec = cfg->num_kv_heads * cfg->head_dim * 2 / 16;
  st.kv_stride = row_stride ? (int)(row_stride / 8) : st.row_vec;
  st.max_tokens = max_tokens;
  if (pages) {
    st.free_pages = pages->free_pages;
    st.free_count = pages->free_count;
    st.ticket = pages->ticket;
    st.page_shift = page_shift_of(cfg->page_size);
  }
  return st;
}

int launch_kv_store(const StepStore& st, int32_t batch, hipStream_t stream, const DenseList* list) {
  TS_REQUIRE(list == nullptr || st.free_pages == nullptr, TS_EINVAL, "internal: a list needs a per-token table");
  if (list)
    hipLaunchKernelGGL(kv_store_list_kernel, dim3((unsigned)batch), dim3(kListThreads), 0, stream, st, *list);
  else
    hipLaunchKernelGGL(kv_store_kernel, dim3((unsigned)batch), dim3(256), 0, stream, st);
  return check_launch("kv_store_kernel");
}

int check_kv_store_chunk(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                         const int32_t* out_cache_loc, const ts_page_pool* pages, int32_t rows, const void* k_pool,
                         const void* v_pool, int64_t pool_rows, const int32_t* table, const int32_t* seq_len,
                         int32_t max_tokens) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(k && v && k_pool && v_pool && table && seq_len, TS_EINVAL,
             "ts_kv_store_chunk: NULL tensor argument");
  TS_REQUIRE_ALIGNED(k, 16, "k");
  TS_REQUIRE_ALIGNED(v, 16, "v");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(v_pool, 16, "v_pool");
  TS_TRY(check_pool_arg(cfg, out_cache_loc, pages, "ts_kv_store_chunk"));
  TS_REQUIRE(rows >= 0 && pool_rows >= 1 && pool_rows <= 0x7fffffffLL && max_tokens >= 1, TS_EINVAL,
             "ts_kv_store_chunk: rows=%d pool_rows=%lld max_tokens=%d out of range", rows,
             (long long)pool_rows, max_tokens);
  return check_row_stride(row_stride, (int64_t)cfg->num_kv_heads * cfg->head_dim, "ts_kv_store_chunk");
}

ChunkStore chunk_store(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                       const int32_t* out_cache_loc, int32_t rows, void* k_pool, void* v_pool, int64_t pool_rows,
                       int32_t* table, int32_t* seq_len, int32_t max_tokens) {
  ChunkStore cs{};
  cs.k = (const uint4*)k;
  cs.v = (const uint4*)v;
  cs.loc = out_cache_loc;
  cs.k_pool = (uint4*)k_pool;
  cs.v_pool = (uint4*)v_pool;
  cs.pool_rows = pool_rows;
  cs.table = table;
  cs.seq_len = seq_len;
  cs.rows = rows;
  cs.row_vec = cfg->num_kv_heads * cfg->head_dim * 2 / 16;
  cs.kv_stride = row_stride ? (int)(row_stride / 8) : cs.row_vec;
  cs.max_tokens = max_tokens;
  return cs;
}

int launch_kv_store_chunk(const ts_config* cfg, const void* k, const void* v, int64_t row_stride,
                          const int32_t* out_cache_loc, const ts_page_pool* pages, int32_t rows, void* k_pool,
                          void* v_pool, int64_t pool_rows, int32_t* table, int32_t* seq_len, int32_t max_tokens,
                          hipStream_t stream) {
  TS_TRY(check_kv_store_chunk(cfg, k, v, row_stride, out_cache_loc, pages, rows, k_pool, v_pool, pool_rows, table,
                              seq_len, max_tokens));
  if (rows == 0) return TS_OK;
  const int row_vec = cfg->num_kv_heads * cfg->head_dim * 2 / 16;
  const int kv_stride = row_stride ? (int)(row_stride / 8) : row_vec;
  if (pages) {
    hipLaunchKernelGGL(kv_store_chunk_paged_kernel, dim3((unsigned)rows), dim3(256), 0,
                       stream, (const uint4*)k, (const uint4*)v, (uint4*)k_pool,
                       (uint4*)v_pool, (uint32_t)pool_rows, table, seq_len, rows, row_vec, kv_stride, max_tokens,
                       page_shift_of(cfg->page_size), page_pool_of(pages));
    return check_launch("kv_store_chunk_paged_kernel");
  }
  const unsigned wgs = (unsigned)ceil_div(rows, kChunkRowsPerWg);
  ChunkStore cs = chunk_store(cfg, k, v, row_stride, out_cache_loc, rows, k_pool, v_pool, pool_rows, table, seq_len,
                              max_tokens);
  cs.workgroups = (int)wgs;
  if (wgs <= (unsigned)kChunkCountedWgs && max_tokens <= kLenMask) {
    hipLaunchKernelGGL(kv_store_chunk_kernel<true>, dim3(wgs), dim3(256), 0, stream, cs);
    return check_launch("kv_store_chunk_kernel");
  }
  hipLaunchKernelGGL(kv_store_chunk_kernel<false>, dim3(wgs), dim3(256), 0, stream, cs);
  TS_TRY(check_launch("kv_store_chunk_kernel"));
  hipLaunchKernelGGL(seq_len_add_kernel, dim3(1), dim3(1), 0, stream, seq_len, rows,
                     max_tokens);
  return check_launch("seq_len_add_kernel");
}

}  // namespace ts

using namespace ts;

extern "C" {

int ts_kv_store(const ts_config* cfg, const void* k, const void* v, const int32_t* out_cache_loc,
                const ts_page_pool* pages, void* k_pool, void* v_pool, int64_t pool_rows, int32_t* table,
                int64_t table_stride, int32_t* seq_lens, int32_t batch, int32_t max_tokens, ts_stream_t stream) {
  TS_TRY(check_kv_store(cfg, k, v, 0, out_cache_loc, pages, k_pool, v_pool, pool_rows, table, table_stride, seq_lens,
                        batch, max_tokens));
  return launch_kv_store(step_store(cfg, k, v, 0, out_cache_loc, pages, k_pool, v_pool, pool_rows, table, table_stride,
                                    seq_lens, max_tokens),
                         batch, (hipStream_t)stream);
}

int ts_kv_store_chunk(const ts_config* cfg, const void* k, const void* v, const int32_t* out_cache_loc,
                      const ts_page_pool* pages, int32_t rows, void* k_pool, void* v_pool, int64_t pool_rows,
                      int32_t* table, int32_t* seq_len, int32_t max_tokens, ts_stream_t stream) {
  return launch_kv_store_chunk(cfg, k, v, 0, out_cache_loc, pages, rows, k_pool, v_pool, pool_rows, table, seq_len,
                               max_tokens, (hipStream_t)stream);
}

}  // extern "C"
