// Several chunks of a prompt at once (patched_radix_attention_extend_forward_flashinfer,
// tr.py:716-773, which takes them one after the other).
//
// What a chunk selects from is the context before it and its own rows, and what it attends to are
// rows of that: once all rows are stored no chunk needs another one's result.  A chunk on its own
// is four launches that are chains of round trips (fingerprint 7 us, selection 23 to 60 with its
// workgroups waiting for each other, gather 6.5, attention 25); together they are seven launches
// for all of them, of which only the attention is long:
//
//   fingerprints    of all chunks, the store of all their rows, every chunk's length
//   statistics      per (chunk, head) maximum and sum of exponentials of the scores, by blocks of tokens
//   votes           the scores once more, as votes (tr.py:361), and the first histogram of the top-k
//   [max-pool]      tr.py:366-369
//   mark, final     the ragged top-k, a chunk as a request
//   gather, attention
//
// Nobody waits for anybody.  The scores are computed twice instead of kept: for one chunk the keys
// are the cost (the single launch streams them once and holds the scores in LDS), for four chunks
// that a workgroup serves together they are read for all of them, and 16 query rows fill the
// matrix instruction's tile.  A prompt of 31599 tokens with 16 more, 28 heads on 4: 4112 -> 2584 us;
// three of 700 to 5200 tokens, 32 heads on 8, two layers: 2343 -> 2126.
#include <algorithm>

#include "ts_topk.h"

namespace ts {

typedef __attribute__((ext_vector_type(8))) __bf16 pr_bf16x8;
typedef __attribute__((ext_vector_type(4))) float pr_f32x4;

constexpr int kPrThreads = 256;
constexpr int kPrChunks = 4;    // chunks of a workgroup: lane group l / 16 of a product's result has chunk l / 16
constexpr int kPrTiles = 4;     // tiles of 16 tokens of a wavefront's step
constexpr int kPrTokens = kPrThreads / 64 * kPrTiles * 16;  // tokens of a workgroup's step

struct PromptScoreArgs {
  const uint16_t* qf;  // [chunks, H, 128] bf16 fingerprints
  const uint4* k_pool;
  uint32_t pool_rows;
  const int32_t* table;
  int page_size, page_shift;
  const int32_t* lens;  // [chunks]
  int chunks, sets;     // sets of kPrChunks
  int n_init, n_local, top_k, max_seq_len, num_heads, head_map;
  int blocks, tokens_per_block;
  float2* partials;     // [chunk][head slot][block] (max, sum exp); head slot: KV head x G + g
  int32_t* seq_len;     // the request's length, advanced by the first of the two
  float* votes;
  int64_t vote_stride;
  uint32_t* hist_ws;    // top-k workspace, or NULL: no histogram
  size_t hist_ws_stride;
};

// Workgroup -> (block of tokens, set of chunks): the sets of a block eight workgroups apart, so that
// they run on one XCD and the keys come from its L2 for all but the first.
__device__ __forceinline__ void prompt_workgroup(const PromptScoreArgs& a, int& block, int& set) {
  const int per = 8 * a.sets, q = (int)blockIdx.x / per, r = (int)blockIdx.x % per;
  set = r / 8;
  block = q * 8 + r % 8;
}

// The query rows of a set as A operands in LDS: operand (KV head, block of four heads, k-step), lane l
// row l % 16, dims 32 ks + 8 (l / 16) + [0, 8).  Row 4 c + i is chunk c's head 4 nb + i of the KV
// head's G (zeros where there is none), so that a lane of the result holds heads of one chunk.
template <int HKV, int NB>
__device__ __forceinline__ void stage_queries(const PromptScoreArgs& a, int set, uint4* to) {
  const int G = a.num_heads / HKV;
  for (int i = threadIdx.x; i < HKV * NB * 4 * 64; i += kPrThreads) {
    const int lane = i & 63, ks = (i >> 6) & 3, nb = (i >> 8) % NB, kvh = (i >> 8) / NB;
    const int chunk = set * kPrChunks + ((lane & 15) >> 2), g = 4 * nb + (lane & 3);
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (chunk < a.chunks && g < G) {
      const int h = a.head_map == TS_HEADMAP_MOD ? kvh + HKV * g : kvh * G + g;
      v = *(const uint4*)(a.qf + ((size_t)chunk * a.num_heads + h) * kHeadDim + 32 * ks + 8 * (lane >> 4));
    }
    to[i] = v;
  }
}

// What a workgroup's set and block are: candidates of each chunk, rows of the pool per token.
struct PromptBlock {
  int set, base, steps;  // steps of kPrTokens tokens that hold candidates of the last chunk
  int n;                 // candidates of this lane's chunk (0: attends to everything, or no chunk)
};
__device__ __forceinline__ int candidates(const PromptScoreArgs& a, int chunk) {
  if (chunk >= a.chunks) return 0;
  return request_geometry(a.lens, nullptr, chunk, a.n_init, a.n_local, a.top_k, a.max_seq_len).n;
}
// false: nothing to do.  rows: tokens_per_block words of LDS.
__device__ __forceinline__ bool prompt_block(const PromptScoreArgs& a, PromptBlock& pb, uint32_t* rows) {
  int block;
  prompt_workgroup(a, block, pb.set);
  if (block >= a.blocks) return false;
  pb.base = block * a.tokens_per_block;
  // (lengths do not fall from chunk to chunk)
  const int most = candidates(a, min(pb.set * kPrChunks + kPrChunks, a.chunks) - 1);
  if (pb.base >= most) return false;
  pb.n = candidates(a, pb.set * kPrChunks + ((int)(threadIdx.x & 63) >> 4));
  const int end = min(a.tokens_per_block, most - pb.base);
  pb.steps = (end + kPrTokens - 1) / kPrTokens;
  for (int i = threadIdx.x; i < pb.steps * kPrTokens; i += kPrThreads)
    rows[i] = lookup_slot(a.table, a.n_init + pb.base + min(i, end - 1), a.page_size, a.page_shift, a.pool_rows);
  return true;
}

// A wavefront's 64 tokens of a step: lane (token l % 16, l / 16) has dims 32 ks + 8 (l / 16) + [0, 8).
struct KeyTiles {
  uint4 k[kPrTiles][4];
};
template <int HKV>
__device__ __forceinline__ void load_keys(const PromptScoreArgs& a, const uint32_t (&row)[kPrTiles], int kvh, KeyTiles& t) {
  const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int j = 0; j < kPrTiles; ++j) {
    const uint4* const at = a.k_pool + ((size_t)row[j] * HKV + kvh) * (kHeadDim / 8) + g4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) t.k[j][ks] = at[4 * ks];
  }
}
__device__ __forceinline__ void step_rows(const uint32_t* rows, int step, uint32_t (&row)[kPrTiles]) {
  const int first = step * kPrTokens + ((int)threadIdx.x >> 6) * (16 * kPrTiles) + (int)(threadIdx.x & 15);
#pragma unroll
  for (int j = 0; j < kPrTiles; ++j) row[j] = rows[first + 16 * j];
}
// s[j][r]: the score of token 16 j + l % 16 and head 4 nb + r of chunk l / 16.
__device__ __forceinline__ void score_tiles(const uint4* queries, int at, const KeyTiles& t, pr_f32x4 (&s)[kPrTiles]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const pr_bf16x8 q = __builtin_bit_cast(pr_bf16x8, queries[(at * 4 + ks) * 64 + (threadIdx.x & 63)]);
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) {
      const pr_f32x4 c = ks == 0 ? pr_f32x4{0.f, 0.f, 0.f, 0.f} : s[j];
      s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q, __builtin_bit_cast(pr_bf16x8, t.k[j][ks]), c, 0, 0, 0);
    }
  }
}

template <int HKV, int NB>
constexpr size_t prompt_query_bytes() { return (size_t)HKV * NB * 4 * 64 * 16; }

// Per (chunk, head) and block of tokens: the largest score and the sum of the exponentials.
template <int HKV, int NB>
__global__ __launch_bounds__(kPrThreads, 2) void prompt_stats_kernel(PromptScoreArgs a) {
  extern __shared__ __attribute__((aligned(16))) char pr_lds[];
  uint4* const queries = (uint4*)pr_lds;
  float2* const stats = (float2*)(pr_lds + prompt_query_bytes<HKV, NB>());  // [wavefront][KV head, nb][16]
  uint32_t* const rows = (uint32_t*)(stats + 4 * HKV * NB * 16);
  // (the launch before this one has stored the rows; nobody reads the length from here on)
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.seq_len = a.lens[a.chunks - 1];
  PromptBlock pb;
  if (!prompt_block(a, pb, rows)) return;
  stage_queries<HKV, NB>(a, pb.set, queries);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = a.num_heads / HKV;
  const int token0 = pb.base + wave * (16 * kPrTiles) + (lane & 15);
  uint32_t row[kPrTiles];
  KeyTiles now, next;
  step_rows(rows, 0, row);
  load_keys<HKV>(a, row, 0, now);
  for (int kvh = 0; kvh < HKV; ++kvh) {
    float m[NB][4], l[NB][4];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        m[nb][r] = kNegBig;
        l[nb][r] = 0.f;
      }
    for (int step = 0; step < pb.steps; ++step) {
      const bool last = step + 1 == pb.steps;
      if (!last || kvh + 1 < HKV) {
        step_rows(rows, last ? 0 : step + 1, row);
        load_keys<HKV>(a, row, last ? kvh + 1 : kvh, next);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        pr_f32x4 s[kPrTiles];
        score_tiles(queries, kvh * NB + nb, now, s);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float top = m[nb][r];
#pragma unroll
          for (int j = 0; j < kPrTiles; ++j) {
            s[j][r] = token0 + step * kPrTokens + 16 * j < pb.n ? s[j][r] : -INFINITY;
            top = fmaxf(top, s[j][r]);
          }
          float sum = l[nb][r] * __expf(m[nb][r] - top);
#pragma unroll
          for (int j = 0; j < kPrTiles; ++j) sum += __expf(s[j][r] - top);
          m[nb][r] = top;
          l[nb][r] = sum;
        }
      }
      now = next;
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        row16_softmax_merge(m[nb][r], l[nb][r]);
        if ((lane & 15) == 0) stats[(wave * HKV * NB + kvh * NB + nb) * 16 + 4 * (lane >> 4) + r] = make_float2(m[nb][r], l[nb][r]);
      }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < HKV * NB * 16; i += kPrThreads) {
    const int chunk = pb.set * kPrChunks + ((i & 15) >> 2), nb = (i >> 4) % NB, kvh = (i >> 4) / NB, g = 4 * nb + (i & 3);
    if (chunk >= a.chunks || g >= G) continue;
    float mm = kNegBig, ll = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float2 p = stats[w * HKV * NB * 16 + i];
      softmax_merge(mm, ll, p.x, p.y);
    }
    a.partials[((size_t)chunk * a.num_heads + kvh * G + g) * a.blocks + pb.base / a.tokens_per_block] = make_float2(mm, ll);
  }
}

// The votes of a block of tokens for a set of chunks, and their share of the top-k's first histogram.
template <int HKV, int NB>
__global__ __launch_bounds__(kPrThreads, 2) void prompt_votes_kernel(PromptScoreArgs a) {
  extern __shared__ __attribute__((aligned(16))) char pr_lds[];
  uint4* const queries = (uint4*)pr_lds;
  float2* const stats = (float2*)(pr_lds + prompt_query_bytes<HKV, NB>());  // [KV head, nb][16]: maximum, 1 / sum
  uint32_t* const hist = (uint32_t*)(stats + HKV * NB * 16);                // [chunk][bin]
  uint32_t* const rows = hist + (a.hist_ws ? kPrChunks * kTopkBins : 0);
  PromptBlock pb;
  if (!prompt_block(a, pb, rows)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = a.num_heads / HKV;
  stage_queries<HKV, NB>(a, pb.set, queries);
  if (a.hist_ws)
    for (int i = threadIdx.x; i < kPrChunks * kTopkBins; i += kPrThreads) hist[i] = 0u;
  __syncthreads();
  uint32_t row[kPrTiles];
  KeyTiles now, next;
  step_rows(rows, 0, row);
  load_keys<HKV>(a, row, 0, now);
  // The statistics of the set's chunks and heads, a wavefront a row at a time, a lane a block.
  for (int i0 = wave; i0 < HKV * NB * 16; i0 += 4 * 4) {
    float2 p[4][2];
    int blocks[4];
    size_t at[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int i = i0 + 4 * x;
      const int chunk = pb.set * kPrChunks + ((i & 15) >> 2), nb = (i >> 4) % NB, kvh = (i >> 4) / NB, g = 4 * nb + (i & 3);
      const bool there = i < HKV * NB * 16 && chunk < a.chunks && g < G;
      blocks[x] = there ? (candidates(a, chunk) + a.tokens_per_block - 1) / a.tokens_per_block : 0;
      at[x] = there ? ((size_t)chunk * a.num_heads + kvh * G + g) * a.blocks : 0;
#pragma unroll
      for (int y = 0; y < 2; ++y)
        p[x][y] = lane + 64 * y < blocks[x] ? a.partials[at[x] + lane + 64 * y] : make_float2(kNegBig, 0.f);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      float m = p[x][0].x, l = p[x][0].y;
      softmax_merge(m, l, p[x][1].x, p[x][1].y);
      for (int y = lane + 128; y < blocks[x]; y += 64) {
        const float2 more = a.partials[at[x] + y];
        softmax_merge(m, l, more.x, more.y);
      }
      row16_softmax_merge(m, l);
      softmax_merge(m, l, __shfl_xor(m, 16), __shfl_xor(l, 16));
      softmax_merge(m, l, __shfl_xor(m, 32), __shfl_xor(l, 32));
      const int i = i0 + 4 * x;
      // (a row without a head: its scores are zero, and so is its share of the vote)
      if (lane == 0 && i < HKV * NB * 16) stats[i] = blocks[x] > 0 ? make_float2(m, 1.0f / l) : make_float2(0.f, 0.f);
    }
  }
  __syncthreads();
  const int chunk = pb.set * kPrChunks + (lane >> 4);
  for (int step = 0; step < pb.steps; ++step) {
    float vote[kPrTiles];
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) vote[j] = 0.f;
    for (int kvh = 0; kvh < HKV; ++kvh) {
      const bool last = kvh + 1 == HKV;
      if (!last || step + 1 < pb.steps) {
        if (last) step_rows(rows, step + 1, row);
        load_keys<HKV>(a, row, last ? 0 : kvh + 1, next);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        pr_f32x4 s[kPrTiles];
        score_tiles(queries, kvh * NB + nb, now, s);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float2 st = stats[(kvh * NB + nb) * 16 + 4 * (lane >> 4) + r];
#pragma unroll
          for (int j = 0; j < kPrTiles; ++j) vote[j] += __expf(s[j][r] - st.x) * st.y;
        }
      }
      now = next;
    }
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) {
      const int t = pb.base + step * kPrTokens + wave * (16 * kPrTiles) + 16 * j + (lane & 15);
      if (t < pb.n) {
        a.votes[(size_t)chunk * a.vote_stride + t] = vote[j];
        if (a.hist_ws) atomicAdd(&hist[(lane >> 4) * kTopkBins + key_bin0(vote_key(vote[j]))], 1u);
      }
    }
  }
  if (!a.hist_ws) return;
  __syncthreads();
  for (int i = threadIdx.x; i < kPrChunks * kTopkBins; i += kPrThreads)
    if (hist[i])  // (of a chunk that is there: others count nothing)
      atomicAdd(&topk_ws(a.hist_ws, a.hist_ws_stride, pb.set * kPrChunks + i / kTopkBins)[kTopkHist0 + i % kTopkBins], hist[i]);
}

// --------------------------------------------------------------------------------- host
// Chunks that one round of launches takes, at most: the launches' fixed cost is shared by then, and the
// staged keys and values of a round (11 MB a chunk at 8 KV heads) stay below the last-level cache.
constexpr int kPrGroup = 20;
// Blocks of tokens: enough for two workgroups per CU, few enough for their statistics to be merged by
// every workgroup of the votes on its own (128 of four chunks' 28 heads: 110 KB from L2, 1 us).
constexpr int kPrBlocks = 128;

// Workspace of a round, carved in this order (256-byte aligned pieces).
struct PromptWorkspace {
  size_t qf, lens, sel, sel_pos, sel_len, votes, pooled, partials, topk, stage, total;
  int64_t vote_stride;
  int max_sel, blocks, tokens_per_block;
};

static PromptWorkspace prompt_workspace(const ts_config* cfg, int chunks, int32_t max_seq_len) {
  PromptWorkspace w;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align_up(bytes, 256);
    return at;
  };
  const size_t C = (size_t)chunks, H = (size_t)cfg->num_heads;
  const int max_n = std::max(max_seq_len - cfg->n_init - cfg->n_local, 1);
  w.vote_stride = ts_score_stride(max_n);
  w.max_sel = cfg->n_init + cfg->top_k + cfg->n_local;
  w.tokens_per_block = (int)ceil_div(max_n, (int64_t)kPrBlocks * kPrTokens) * kPrTokens;
  w.blocks = (int)ceil_div(max_n, w.tokens_per_block);
  w.qf = take(C * H * kHeadDim * 2);
  w.lens = take(C * 4);
  w.sel = take(C * w.max_sel * 4);
  w.sel_pos = take(C * w.max_sel * 4);
  w.sel_len = take(C * 4);
  w.votes = take(C * w.vote_stride * 4);
  w.pooled = take(cfg->pool_kernel > 0 ? C * w.vote_stride * 4 : 0);
  w.partials = take(C * H * kPrBlocks * sizeof(float2));  // (fewer tokens can be more blocks)
  w.topk = take(ts_topk_workspace_bytes(cfg, chunks, max_seq_len));
  w.stage = take(C * ts_prefill_attn_workspace_bytes(cfg, w.max_sel));
  w.total = off;
  return w;
}

template <int HKV, int NB>
static int launch_prompt_scores(const PromptScoreArgs& a, hipStream_t stream) {
  const size_t queries = prompt_query_bytes<HKV, NB>(), rows = (size_t)a.tokens_per_block * 4;
  const size_t stats_lds = queries + 4 * HKV * NB * 16 * sizeof(float2) + rows;
  const size_t votes_lds = queries + HKV * NB * 16 * sizeof(float2) + (a.hist_ws ? kPrChunks * kTopkBins * 4 : 0) + rows;
  // (2^20 candidates in kPrBlocks blocks: 32 KB of rows, and at most 104 KB of the others)
  constexpr int kMostLds = 160 * 1024;
  static const hipError_t ok1 = hipFuncSetAttribute((const void*)prompt_stats_kernel<HKV, NB>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds);
  static const hipError_t ok2 = hipFuncSetAttribute((const void*)prompt_votes_kernel<HKV, NB>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds);
  if (ok1 != hipSuccess || ok2 != hipSuccess || stats_lds > kMostLds || votes_lds > kMostLds)
    return fail(TS_EHIP, "prompt scores: %zu and %zu bytes of LDS refused", stats_lds, votes_lds);
  const dim3 grid((unsigned)(ceil_div(a.blocks, 8) * 8 * a.sets));
  hipLaunchKernelGGL((prompt_stats_kernel<HKV, NB>), grid, dim3(kPrThreads), stats_lds, stream, a);
  TS_TRY(check_launch("prompt_stats_kernel"));
  hipLaunchKernelGGL((prompt_votes_kernel<HKV, NB>), grid, dim3(kPrThreads), votes_lds, stream, a);
  return check_launch("prompt_votes_kernel");
}

static int launch_prompt_scores(const ts_config* cfg, const PromptScoreArgs& a, hipStream_t stream) {
  const bool wide = cfg->num_heads / cfg->num_kv_heads > 4;
#define TS_PR_CASE(HKV_) \
  case HKV_: return wide ? launch_prompt_scores<HKV_, 2>(a, stream) : launch_prompt_scores<HKV_, 1>(a, stream);
  switch (cfg->num_kv_heads) {
    TS_PR_CASE(1)
    TS_PR_CASE(2)
    TS_PR_CASE(4)
    TS_PR_CASE(8)
    default: return fail(TS_ESHAPE, "unsupported number of KV heads %d", cfg->num_kv_heads);
  }
#undef TS_PR_CASE
}

}  // namespace ts

using namespace ts;

extern "C" {

size_t ts_prefill_prompt_workspace_bytes(const ts_config* cfg, int32_t rows, int32_t chunk_rows, int32_t max_seq_len) {
  if (validate_config(cfg) != TS_OK || rows < 1 || chunk_rows < 1 || max_seq_len < 1) return 0;
  return prompt_workspace(cfg, (int)std::min<int64_t>(ceil_div(rows, chunk_rows), kPrGroup), max_seq_len).total;
}

int ts_prefill_prompt(const ts_config* cfg, const ts_batch* bt, const ts_new_kv* kv, const void* q,
                      int32_t q_row_stride, int32_t kv_row_stride, int32_t rows, int32_t chunk_rows,
                      const float* cos_table, const float* sin_table, int64_t table_rows, void* k_pool, void* v_pool,
                      int64_t pool_rows, void* out, void* workspace, size_t workspace_bytes, ts_stream_t stream) {
  TS_TRY(validate_config(cfg));
  TS_TRY(check_row_stride(q_row_stride, (int64_t)cfg->num_heads * cfg->head_dim, "ts_prefill_prompt"));
  TS_TRY(check_row_stride(kv_row_stride, (int64_t)cfg->num_kv_heads * cfg->head_dim, "ts_prefill_prompt"));
  TS_REQUIRE(bt != nullptr && bt->batch == 1 && bt->k_per_req == nullptr && kv != nullptr, TS_EINVAL,
             "ts_prefill_prompt serves one request at a time (batch must be 1) and needs the prompt's K/V");
  TS_TRY(validate_batch(cfg, bt));
  TS_REQUIRE(rows >= 1 && chunk_rows >= 1 && chunk_rows <= 65535 * 16, TS_EINVAL,
             "ts_prefill_prompt: %d rows in chunks of %d", rows, chunk_rows);
  TS_REQUIRE(kv->pages == nullptr && cfg->page_size == 1, TS_EINVAL,
             "ts_prefill_prompt: slots chosen by the caller and a per-token table only");
  TS_REQUIRE(q && cos_table && sin_table && out, TS_EINVAL, "ts_prefill_prompt: NULL tensor argument");
  int32_t* const table = const_cast<int32_t*>(bt->table);
  int32_t* const seq_len = const_cast<int32_t*>(bt->seq_lens);
  TS_TRY(check_kv_store_chunk(cfg, kv->k, kv->v, kv_row_stride, kv->out_cache_loc, nullptr, rows, k_pool, v_pool,
                              pool_rows, table, seq_len, kv->max_tokens));
  TS_REQUIRE_ALIGNED(q, 16, "q");
  TS_REQUIRE_ALIGNED(out, 16, "out");
  TS_REQUIRE_ALIGNED(workspace, 256, "workspace");
  TS_TRY(check_fingerprint(q, std::min(rows, chunk_rows), cos_table, sin_table, table_rows, workspace, cfg->n_local));
  TS_REQUIRE(bt->max_seq_len - cfg->n_init - cfg->n_local <= (1 << 20), TS_ESHAPE,
             "ts_prefill_prompt: at most 2^20 candidates (max_seq_len %d)", bt->max_seq_len);
  const int chunks = (int)ceil_div(rows, chunk_rows);
  TS_REQUIRE(workspace_bytes >= prompt_workspace(cfg, std::min(chunks, kPrGroup), bt->max_seq_len).total, TS_EWORKSPACE,
             "ts_prefill_prompt: workspace %zu bytes < required %zu", workspace_bytes,
             prompt_workspace(cfg, std::min(chunks, kPrGroup), bt->max_seq_len).total);

  const hipStream_t st = (hipStream_t)stream;
  const int q_stride = q_row_stride ? q_row_stride : cfg->num_heads * cfg->head_dim;
  const int kv_stride = kv_row_stride ? kv_row_stride : cfg->num_kv_heads * cfg->head_dim;
  const int group = (int)ceil_div(chunks, ceil_div(chunks, kPrGroup));  // (rounds of about the same size)
  for (int first = 0; first < chunks; first += group) {
    const int here = std::min(group, chunks - first);
    const int64_t row0 = (int64_t)first * chunk_rows;
    const int32_t n_rows = (int32_t)std::min<int64_t>((int64_t)here * chunk_rows, rows - row0);
    // Bounds every length of the round: what follows it is not there yet (unless the table gets full,
    // and rows are dropped).
    const int64_t later = bt->max_seq_len < kv->max_tokens ? rows - row0 - n_rows : 0;
    const int32_t bound = (int32_t)std::max<int64_t>(bt->max_seq_len - later, 1);
    const PromptWorkspace w = prompt_workspace(cfg, here, bound);
    char* const ws = (char*)workspace;
    int32_t *const lens = (int32_t*)(ws + w.lens), *const sel = (int32_t*)(ws + w.sel),
                   *const sel_len = (int32_t*)(ws + w.sel_len);
    float *const votes = (float*)(ws + w.votes), *const pooled = cfg->pool_kernel > 0 ? (float*)(ws + w.pooled) : nullptr;
    const uint16_t* const q0 = (const uint16_t*)q + row0 * q_stride;

    ts_batch each = *bt;  // the chunks as requests that share the table
    each.batch = here;
    each.max_seq_len = bound;
    each.seq_lens = lens;
    each.table_stride = 0;
    each.host_seq_lens = nullptr;
    TopkArgs topk = make_topk_args(cfg, &each, pooled ? pooled : votes, w.vote_stride, nullptr, nullptr, sel,
                                   (int32_t*)(ws + w.sel_pos), w.max_sel, sel_len, (uint32_t*)(ws + w.topk));
    if (first + here == chunks) topk.hint = bt->threshold_hint;
    const ZeroRegion counters = topk_zero_region(topk, here);
    const PromptChunks pc{n_rows, chunk_rows, here, lens, counters.base, (size_t)counters.stride, counters.words};
    const ChunkStore cs = chunk_store(cfg, (const uint16_t*)kv->k + row0 * kv_stride,
                                      (const uint16_t*)kv->v + row0 * kv_stride, kv_row_stride,
                                      kv->out_cache_loc + row0, n_rows, k_pool, v_pool, pool_rows, table, seq_len,
                                      kv->max_tokens);
    TS_TRY(launch_prompt_fingerprint(cfg, q0, q_stride, cos_table, sin_table, table_rows, ws + w.qf, pc, cs, st));

    PromptScoreArgs a{};
    a.qf = (const uint16_t*)(ws + w.qf);
    a.k_pool = (const uint4*)k_pool;
    a.pool_rows = (uint32_t)pool_rows;
    a.table = table;
    a.page_size = 1;
    a.lens = lens;
    a.chunks = here;
    a.sets = (int)ceil_div(here, kPrChunks);
    a.n_init = cfg->n_init;
    a.n_local = cfg->n_local;
    a.top_k = cfg->top_k;
    a.max_seq_len = bound;
    a.num_heads = cfg->num_heads;
    a.head_map = cfg->head_map;
    a.blocks = w.blocks;
    a.tokens_per_block = w.tokens_per_block;
    a.partials = (float2*)(ws + w.partials);
    a.seq_len = seq_len;
    a.votes = votes;
    a.vote_stride = w.vote_stride;
    a.hist_ws = pooled ? nullptr : topk.ws;  // (the selection sees the pooled votes)
    a.hist_ws_stride = topk.ws_stride;
    TS_TRY(launch_prompt_scores(cfg, a, st));
    if (pooled) TS_TRY(launch_pool(cfg, &each, votes, w.vote_stride, pooled, w.vote_stride, nullptr, st));
    TS_TRY(launch_topk(topk, here, std::max(bound - cfg->n_init - cfg->n_local, 0), st, true, pooled == nullptr));
    TS_TRY(launch_prefill_attn_chunks(cfg, q0, q_stride, n_rows, std::min(chunk_rows, n_rows), k_pool, v_pool, pool_rows,
                                      sel, w.max_sel, sel_len, w.max_sel,
                                      (uint16_t*)out + row0 * cfg->num_heads * cfg->head_dim, ws + w.stage,
                                      w.total - w.stage, st));
  }
  return TS_OK;
}

}  // extern "C"
