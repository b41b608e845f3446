// Several chunks of a prompt at once (patched_radix_attention_extend_forward_flashinfer,
// tr.py:716-773, which takes them one after the other).  The first of them, which attend to all tokens so far,
// are one long chunk; what follows is about the others.
//
// What a chunk selects from is the context before it and its own rows, and what it attends to are
// rows of that: once all rows are stored no chunk needs another one's result.  A chunk on its own
// is four launches that are chains of round trips (fingerprint 7 us, selection 23 to 60 with its
// workgroups waiting for each other, gather 6.5, attention 25); together they are eight launches
// for all of them, nine or ten where some chunks fill no wave of the wide attention or votes are
// pooled (whose first histogram is then a launch too), and only the attention is long:
//
//   fingerprints    of all chunks, the store of all their rows, every chunk's length
//   statistics      per (chunk, head) maximum and sum of exponentials of the scores, by blocks of tokens
//   merge           of the blocks' statistics
//   votes           the scores once more, as votes (tr.py:361), and the first histogram of the top-k
//   [max-pool, histogram]  tr.py:366-369
//   mark, final     the ragged top-k, a chunk as a request
//   gather, attention [, attention of the chunks that are left]
//
// Nobody waits for anybody.  The scores are computed twice instead of kept: for one chunk the keys
// are the cost (the single launch streams them once and holds the scores in LDS), for four chunks
// that a workgroup serves together they are read for all of them, and 16 query rows fill the
// matrix instruction's tile.  A prompt of 31599 tokens with 16 more, 28 heads on 4, its chunks one after
// the other and together: 4183 and 2040 us; three of 700 to 5200 tokens + 8, 32 heads on 8, two layers: 2352 and 1713
// (both of a case in turn on one box).
#include <algorithm>
#include <type_traits>

#include "ts_topk.h"

namespace ts {

typedef __attribute__((ext_vector_type(8))) __bf16 pr_bf16x8;
typedef __attribute__((ext_vector_type(4))) float pr_f32x4;

constexpr int kPrWaves = 4;
constexpr int kPrThreads = 64 * kPrWaves;
constexpr int kPrChunks = 4;    // chunks of a workgroup: lane group l / 16 of a product's result has chunk l / 16
constexpr int kPrTiles = 4;     // tiles of 16 tokens of a wavefront's step

// A workgroup's four wavefronts take KV heads of their own: 64 tokens a step with four of them or more, and
// more tokens where the heads are fewer.  A wavefront then has its query rows in registers for all its tokens,
// and a workgroup of few tokens is a short chain: with all heads one after the other in every wavefront, the
// queries in LDS and each workgroup merging the statistics for itself, a workgroup of 256 tokens took 23 us
// (statistics) and 46 us (votes) whatever the length.  Statistics, merge and votes of 19 chunks up to 31K tokens,
// 28 heads on 4: 43 + 95 -> 26 + 5 + 31 us; of 6 up to 5K, 32 on 8: 23 + 51 -> 9 + 5 + 12.
template <int HKV>
struct PromptSplit {
  static constexpr int kHeadGroups = HKV < kPrWaves ? HKV : kPrWaves;
  static constexpr int kHeads = HKV / kHeadGroups;          // of a wavefront
  static constexpr int kTokenGroups = kPrWaves / kHeadGroups;
  static constexpr int kTokens = kTokenGroups * kPrTiles * 16;  // of a step
};
constexpr int prompt_token_groups(int kv_heads) { return kv_heads < kPrWaves ? kPrWaves / kv_heads : 1; }

struct PromptScoreArgs {
  const uint16_t* qf;  // [chunks, H, 128] bf16 fingerprints
  const uint4* k_pool;
  uint32_t pool_rows;
  const int32_t* table; // per token
  const int32_t* lens;  // [chunks]
  int chunks, sets;     // sets of kPrChunks
  int n_init, n_local, top_k, max_seq_len, num_heads, head_map;
  int blocks, tokens_per_block;
  float2* partials;     // [chunk][head slot][block, token group] (max, sum exp); head slot: KV head x G + g
  float2* stats;        // [chunk][head slot] (max, 1 / sum exp)
  int32_t* seq_len;     // the request's length, advanced by the first of the launches
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

// What a workgroup's set and block are, and a wavefront's share of them.
struct PromptBlock {
  int set, block, base, steps;  // steps that hold candidates of the last chunk
  int most;                     // candidates of that
  int chunk, n;                 // this lane's chunk, and its candidates (0: attends to everything, or no chunk)
  int token0;                   // the lane's first token
  int kvh0, token_group;        // the wavefront's first KV head
};
__device__ __forceinline__ int candidates(const PromptScoreArgs& a, int chunk) {
  if (chunk >= a.chunks) return 0;
  return request_geometry(a.lens, nullptr, chunk, a.n_init, a.n_local, a.top_k, a.max_seq_len).n;
}
// false: nothing to do.
template <int HKV>
__device__ __forceinline__ bool prompt_block(const PromptScoreArgs& a, PromptBlock& pb) {
  using Split = PromptSplit<HKV>;
  prompt_workgroup(a, pb.block, pb.set);
  if (pb.block >= a.blocks) return false;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  pb.base = pb.block * a.tokens_per_block;
  pb.chunk = pb.set * kPrChunks + (lane >> 4);
  // (lengths do not fall from chunk to chunk)
  pb.most = candidates(a, min(pb.set * kPrChunks + kPrChunks, a.chunks) - 1);
  pb.n = candidates(a, pb.chunk);
  if (pb.base >= pb.most) return false;
  pb.steps = (min(a.tokens_per_block, pb.most - pb.base) + Split::kTokens - 1) / Split::kTokens;
  pb.token_group = wave / Split::kHeadGroups;
  pb.kvh0 = wave % Split::kHeadGroups * Split::kHeads;
  pb.token0 = pb.base + pb.token_group * (16 * kPrTiles) + (lane & 15);
  return true;
}

// The query rows of a set for a wavefront's KV heads as A operands: lane l row l % 16, dims
// 32 ks + 8 (l / 16) + [0, 8).  Row 4 c + i is chunk c's head 4 nb + i of the KV head's G (zeros where
// there is none), so that a lane of the result holds heads of one chunk.
template <int HKV, int NB>
struct PromptQueries {
  uint4 q[PromptSplit<HKV>::kHeads][NB][4];
};
template <int HKV, int NB>
__device__ __forceinline__ void load_queries(const PromptScoreArgs& a, const PromptBlock& pb, PromptQueries<HKV, NB>& to) {
  const int lane = threadIdx.x & 63, G = a.num_heads / HKV, chunk = pb.set * kPrChunks + ((lane & 15) >> 2);
#pragma unroll
  for (int x = 0; x < PromptSplit<HKV>::kHeads; ++x)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int g = 4 * nb + (lane & 3), kvh = pb.kvh0 + x;
      const bool there = chunk < a.chunks && g < G;
      const int h = a.head_map == TS_HEADMAP_MOD ? kvh + HKV * g : kvh * G + g;
      const uint16_t* const row = a.qf + ((size_t)chunk * a.num_heads + h) * kHeadDim + 8 * (lane >> 4);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) to.q[x][nb][ks] = there ? *(const uint4*)(row + 32 * ks) : make_uint4(0u, 0u, 0u, 0u);
    }
}

// A wavefront's 64 tokens of a step: lane (token l % 16, l / 16) has dims 32 ks + 8 (l / 16) + [0, 8).
struct KeyTiles {
  uint4 k[kPrTiles][4];
};
// (rows as the table has them: they are checked here, where they are used, and not where they are asked for)
template <int HKV>
__device__ __forceinline__ void load_keys(const PromptScoreArgs& a, const uint32_t (&row)[kPrTiles], int kvh, KeyTiles& t) {
  const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int j = 0; j < kPrTiles; ++j) {
    const uint4* const at = a.k_pool + ((size_t)min(row[j], a.pool_rows - 1) * HKV + kvh) * (kHeadDim / 8) + g4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) t.k[j][ks] = at[4 * ks];
  }
}
template <int HKV>
__device__ __forceinline__ void step_rows(const PromptScoreArgs& a, const PromptBlock& pb, int step, uint32_t (&row)[kPrTiles]) {
#pragma unroll
  for (int j = 0; j < kPrTiles; ++j)
    row[j] = (uint32_t)a.table[a.n_init + min(pb.token0 + step * PromptSplit<HKV>::kTokens + 16 * j, pb.most - 1)];
}
// s[j][r]: the score of token 16 j + l % 16 and head 4 nb + r of chunk l / 16.
__device__ __forceinline__ void score_tiles(const uint4 (&queries)[4], const KeyTiles& t, pr_f32x4 (&s)[kPrTiles]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const pr_bf16x8 q = __builtin_bit_cast(pr_bf16x8, queries[ks]);
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) {
      const pr_f32x4 c = ks == 0 ? pr_f32x4{0.f, 0.f, 0.f, 0.f} : s[j];
      s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q, __builtin_bit_cast(pr_bf16x8, t.k[j][ks]), c, 0, 0, 0);
    }
  }
}

// body(step, x, keys) for every step and every KV head x of the wavefront's, the next turn's keys and
// the table's entries for those of the step after under way.  The entries are asked for before the
// keys: they are waited for first.  No load is behind a branch within the loops, or the compiler would wait
// for all loads where the paths meet.
template <int HKV, typename Body>
__device__ __forceinline__ void walk_keys(const PromptScoreArgs& a, const PromptBlock& pb, Body body) {
  constexpr int kHeads = PromptSplit<HKV>::kHeads;
  static_assert(kHeads == 1 || kHeads == 2, "the turns alternate between two sets of registers");
  constexpr std::integral_constant<int, 0> head0{};
  uint32_t row[kPrTiles], ahead[kPrTiles];
  KeyTiles even, odd;
  step_rows<HKV>(a, pb, 0, row);
  step_rows<HKV>(a, pb, 1, ahead);
  load_keys<HKV>(a, row, pb.kvh0, even);
  auto next_step = [&](int step, KeyTiles& keys) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) row[j] = ahead[j];
    step_rows<HKV>(a, pb, step + 1, ahead);
    load_keys<HKV>(a, row, pb.kvh0, keys);
  };
  int step = 0;
  if constexpr (kHeads == 2) {
    constexpr std::integral_constant<int, 1> head1{};
    for (; step + 1 < pb.steps; ++step) {
      load_keys<HKV>(a, row, pb.kvh0 + 1, odd);
      body(step, head0, even);
      next_step(step + 1, even);
      body(step, head1, odd);
    }
    load_keys<HKV>(a, row, pb.kvh0 + 1, odd);
    body(step, head0, even);
    body(step, head1, odd);
  } else {
    for (; step + 2 < pb.steps; step += 2) {
      next_step(step + 1, odd);
      body(step, head0, even);
      next_step(step + 2, even);
      body(step + 1, head0, odd);
    }
    if (step + 1 < pb.steps) {
      next_step(step + 1, odd);
      body(step, head0, even);
      body(step + 1, head0, odd);
    } else {
      body(step, head0, even);
    }
  }
}

// Per (chunk, head), block of tokens and token group: the largest score and the sum of the exponentials.
template <int HKV, int NB>
__global__ __launch_bounds__(kPrThreads, HKV * NB > 8 ? 1 : 2) void prompt_stats_kernel(PromptScoreArgs a) {
  using Split = PromptSplit<HKV>;
  // (the launch before this one has stored the rows; nobody reads the length from here on)
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.seq_len = a.lens[a.chunks - 1];
  PromptBlock pb;
  if (!prompt_block<HKV>(a, pb)) return;
  PromptQueries<HKV, NB> queries;
  load_queries<HKV, NB>(a, pb, queries);
  float m[Split::kHeads][NB][4], l[Split::kHeads][NB][4];
#pragma unroll
  for (int x = 0; x < Split::kHeads; ++x)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        m[x][nb][r] = kNegBig;
        l[x][nb][r] = 0.f;
      }
  walk_keys<HKV>(a, pb, [&](int step, auto which, const KeyTiles& keys) __attribute__((always_inline)) {
    constexpr int x = decltype(which)::value;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      pr_f32x4 s[kPrTiles];
      score_tiles(queries.q[x][nb], keys, s);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float top = m[x][nb][r];
#pragma unroll
        for (int j = 0; j < kPrTiles; ++j) {
          s[j][r] = pb.token0 + step * Split::kTokens + 16 * j < pb.n ? s[j][r] : -INFINITY;
          top = fmaxf(top, s[j][r]);
        }
        float sum = l[x][nb][r] * __expf(m[x][nb][r] - top);
#pragma unroll
        for (int j = 0; j < kPrTiles; ++j) sum += __expf(s[j][r] - top);
        m[x][nb][r] = top;
        l[x][nb][r] = sum;
      }
    }
  });
  const int lane = threadIdx.x & 63, G = a.num_heads / HKV;
#pragma unroll
  for (int x = 0; x < Split::kHeads; ++x)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        row16_softmax_merge(m[x][nb][r], l[x][nb][r]);
        const int g = 4 * nb + r;
        if ((lane & 15) == 0 && pb.chunk < a.chunks && g < G)
          a.partials[(((size_t)pb.chunk * a.num_heads + (pb.kvh0 + x) * G + g) * a.blocks + pb.block) * Split::kTokenGroups +
                     pb.token_group] = make_float2(m[x][nb][r], l[x][nb][r]);
      }
}

// The blocks' statistics merged, a wavefront a (chunk, head).
__global__ __launch_bounds__(kPrThreads) void prompt_merge_kernel(PromptScoreArgs a, int token_groups) {
  const int i = (int)blockIdx.x * kPrWaves + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= a.chunks * a.num_heads) return;
  const int n = candidates(a, i / a.num_heads);
  const int entries = (n + a.tokens_per_block - 1) / a.tokens_per_block * token_groups;
  const float2* const from = a.partials + (size_t)i * a.blocks * token_groups;
  float m = kNegBig, l = 0.f;
  for (int at = lane; at < entries; at += 4 * 64) {
    float2 p[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) p[x] = at + 64 * x < entries ? from[at + 64 * x] : make_float2(kNegBig, 0.f);
#pragma unroll
    for (int x = 0; x < 4; ++x) softmax_merge(m, l, p[x].x, p[x].y);
  }
  row16_softmax_merge(m, l);
  softmax_merge(m, l, __shfl_xor(m, 16), __shfl_xor(l, 16));
  softmax_merge(m, l, __shfl_xor(m, 32), __shfl_xor(l, 32));
  if (lane == 0) a.stats[i] = n > 0 ? make_float2(m, 1.0f / l) : make_float2(0.f, 0.f);
}

// The votes of a block of tokens for a set of chunks, and their share of the top-k's first histogram.
template <int HKV, int NB>
__global__ __launch_bounds__(kPrThreads, HKV * NB > 8 ? 1 : 2) void prompt_votes_kernel(PromptScoreArgs a) {
  using Split = PromptSplit<HKV>;
  constexpr int kTileWords = 80;  // (64, and 16 more: the readers' tiles start in different banks)
  __shared__ __attribute__((aligned(16))) uint32_t hist[kPrChunks * kTopkBins];
  __shared__ float shares[2][kPrWaves][kPrTiles * kTileWords];  // of a step's votes: [wavefront][tile][lane]
  PromptBlock pb;
  if (!prompt_block<HKV>(a, pb)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = a.num_heads / HKV;
  PromptQueries<HKV, NB> queries;
  load_queries<HKV, NB>(a, pb, queries);
  float2 st[Split::kHeads][NB][4];
#pragma unroll
  for (int x = 0; x < Split::kHeads; ++x)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int g = 4 * nb + r;
        // (a row without a head: its scores are zero, and so is its share of the vote)
        st[x][nb][r] = pb.chunk < a.chunks && g < G
                           ? a.stats[(size_t)pb.chunk * a.num_heads + (pb.kvh0 + x) * G + g] : make_float2(0.f, 0.f);
      }
  if (a.hist_ws)
    for (int i = tid; i < kPrChunks * kTopkBins / 4; i += kPrThreads) ((uint4*)hist)[i] = make_uint4(0u, 0u, 0u, 0u);
  // Of the step's sums this wavefront adds up those of its chunk of the set, a lane a token.
  const int mine = pb.set * kPrChunks + wave, n_mine = candidates(a, mine);
  float vote[kPrTiles];
  walk_keys<HKV>(a, pb, [&](int step, auto which, const KeyTiles& keys) __attribute__((always_inline)) {
    constexpr int x = decltype(which)::value;
    if (x == 0)
#pragma unroll
      for (int j = 0; j < kPrTiles; ++j) vote[j] = 0.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      pr_f32x4 s[kPrTiles];
      score_tiles(queries.q[x][nb], keys, s);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < kPrTiles; ++j) vote[j] += __expf(s[j][r] - st[x][nb][r].x) * st[x][nb][r].y;
    }
    if (x + 1 < Split::kHeads) return;
    float* const to = shares[step & 1][wave];
#pragma unroll
    for (int j = 0; j < kPrTiles; ++j) to[j * kTileWords + lane] = vote[j];
    // One meeting a step: who writes these shares again, two steps on, has met those who read them one step on.
    // (The histogram is cleared before the first.)
    __syncthreads();
#pragma unroll
    for (int tg = 0; tg < Split::kTokenGroups; ++tg) {
      float sum = 0.f;
#pragma unroll
      for (int hg = 0; hg < Split::kHeadGroups; ++hg)
        sum += shares[step & 1][tg * Split::kHeadGroups + hg][(lane >> 4) * kTileWords + 16 * wave + (lane & 15)];
      const int t = pb.base + step * Split::kTokens + 64 * tg + lane;
      if (t < n_mine) {
        a.votes[(size_t)mine * a.vote_stride + t] = sum;
        if (a.hist_ws) atomicAdd(&hist[wave * kTopkBins + key_bin0(vote_key(sum))], 1u);
      }
    }
  });
  if (!a.hist_ws) return;
  // (each wavefront has counted its chunk's on its own)
  uint32_t* const counts = topk_ws(a.hist_ws, a.hist_ws_stride, mine) + kTopkHist0;
  for (int i = 4 * lane; i < kTopkBins; i += 4 * 64) {
    const uint4 c = *(const uint4*)(hist + wave * kTopkBins + i);
    // (of a chunk that is there: others count nothing)
    if (c.x) atomicAdd(&counts[i], c.x);
    if (c.y) atomicAdd(&counts[i + 1], c.y);
    if (c.z) atomicAdd(&counts[i + 2], c.z);
    if (c.w) atomicAdd(&counts[i + 3], c.w);
  }
}

// --------------------------------------------------------------------------------- host
// Chunks that one round of launches takes, at most: the launches' fixed cost is shared by then.
constexpr int kPrGroup = 20;
// And the most workspace of a round of several chunks, so that what a prompt needs beside the KV pool is bounded.
// 20 chunks of 32 heads on 8 and top-k 2048 are 229 MB at 31.6K tokens, 253 at 131K and 476 at 1M; with top-k 4096
// 397, 421 and, of 16 chunks, 515.  (Half of this cost 10240 rows behind 900K tokens 3.59 -> 4.36 ms, two sets of
// chunks more to read the keys for, and 31599 rows with top-k 4096 2.57 -> 2.76.)
constexpr size_t kPrBytes = (size_t)512 << 20;
// Rows that one launch of the attention takes (ts_sparse_prefill_attn's limit too).
constexpr int kPrRows = 65535 * 16;
// Workgroups of the scores' launches: two per CU, as many as run at once.
constexpr int kPrWorkgroups = 512;

// Workspace of a round, carved in this order (256-byte aligned pieces).
struct PromptWorkspace {
  size_t qf, lens, sel, sel_pos, sel_len, votes, pooled, partials, stats, topk, stage, total;
  int64_t vote_stride;
  int max_sel, blocks, tokens_per_block;
};

static PromptWorkspace prompt_workspace(const ts_config* cfg, int chunks, int32_t max_seq_len, bool cut = false) {
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
  const int token_groups = prompt_token_groups(cfg->num_kv_heads), step = token_groups * kPrTiles * 16;
  const int64_t sets = ceil_div(chunks, kPrChunks);
  w.tokens_per_block = (int)ceil_div(max_n, ceil_div(kPrWorkgroups, sets) * step) * step;
  w.blocks = (int)ceil_div(max_n, w.tokens_per_block);
  w.qf = take(C * H * kHeadDim * 2);
  w.lens = take(C * 4);
  w.sel = take(C * w.max_sel * 4);
  w.sel_pos = take(C * w.max_sel * 4);
  w.sel_len = take(C * 4);
  w.votes = take(C * w.vote_stride * 4);
  w.pooled = take(cfg->pool_kernel > 0 ? C * w.vote_stride * 4 : 0);
  // (as much for any round: at most ceil(workgroups / sets) blocks of at most 4 sets chunks)
  w.partials = take((size_t)(kPrWorkgroups + ceil_div(kPrGroup, kPrChunks)) * kPrChunks * H * token_groups * sizeof(float2));
  w.stats = take(C * H * sizeof(float2));
  w.topk = take(ts_topk_workspace_bytes(cfg, chunks, max_seq_len));
  // (what the attention leaves of its jobs that are cut, where nobody reads the selection's any more)
  if (cut) off = std::max(off, w.votes + align_up(prefill_cut_bytes(), 256));
  w.stage = take(C * ts_prefill_attn_workspace_bytes(cfg, w.max_sel));
  w.total = off;
  return w;
}

// The most chunks of a round.
static int prompt_group(const ts_config* cfg, int32_t rows, int32_t chunk_rows, int32_t max_seq_len) {
  int group = (int)std::min<int64_t>({ceil_div(rows, chunk_rows), kPrGroup, kPrRows / chunk_rows});
  while (group > 1 && prompt_workspace(cfg, group, max_seq_len).total > kPrBytes)  // (whole sets, while there are any)
    group = group > kPrChunks ? (group - 1) / kPrChunks * kPrChunks : group - 1;
  return group;
}

// Whether the attention of a call may cut jobs: some launch gains by it, and the bound leaves room for their pieces.
static bool prompt_cuts(const ts_config* cfg, int32_t rows, int32_t chunk_rows, int32_t max_seq_len) {
  const int most = prompt_group(cfg, rows, chunk_rows, max_seq_len);
  const int keys = std::min(cfg->n_init + cfg->top_k + cfg->n_local, max_seq_len);
  // The rows that are one dense chunk, and the keys of its last.
  const int before = std::max(max_seq_len - rows, 0);
  int dense = std::min(rows, std::max(keys - before, 0));
  if (dense < rows) dense = dense / chunk_rows * chunk_rows;
  return ((dense > 0 && prefill_cuts_pay(cfg->num_heads, cfg->num_kv_heads, dense, dense, before + dense)) ||
          prefill_cuts_pay(cfg->num_heads, cfg->num_kv_heads, rows, chunk_rows, keys)) &&
         prompt_workspace(cfg, most, max_seq_len, true).total <= std::max(kPrBytes, prompt_workspace(cfg, most, max_seq_len).total);
}

template <int HKV, int NB>
static int launch_prompt_scores(const PromptScoreArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)(ceil_div(a.blocks, 8) * 8 * a.sets));
  hipLaunchKernelGGL((prompt_stats_kernel<HKV, NB>), grid, dim3(kPrThreads), 0, stream, a);
  TS_TRY(check_launch("prompt_stats_kernel"));
  hipLaunchKernelGGL(prompt_merge_kernel, dim3((unsigned)ceil_div(a.chunks * a.num_heads, kPrWaves)), dim3(kPrThreads), 0,
                     stream, a, PromptSplit<HKV>::kTokenGroups);
  TS_TRY(check_launch("prompt_merge_kernel"));
  hipLaunchKernelGGL((prompt_votes_kernel<HKV, NB>), grid, dim3(kPrThreads), 0, stream, a);
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
  if (validate_config(cfg) != TS_OK || rows < 1 || chunk_rows < 1 || chunk_rows > kPrRows || max_seq_len < 1)
    return 0;
  return prompt_workspace(cfg, prompt_group(cfg, rows, chunk_rows, max_seq_len), max_seq_len,
                          prompt_cuts(cfg, rows, chunk_rows, max_seq_len)).total;
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
  TS_REQUIRE(rows >= 1 && chunk_rows >= 1 && chunk_rows <= kPrRows, TS_EINVAL,
             "ts_prefill_prompt: %d rows in chunks of %d", rows, chunk_rows);
  // (nothing waits here, so that no call gives up and has to be repeated without its append)
  TS_REQUIRE(bt->rerun == 0, TS_EINVAL, "ts_prefill_prompt has no call to repeat (rerun)");
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
  const int chunks = (int)ceil_div(rows, chunk_rows), most = prompt_group(cfg, rows, chunk_rows, bt->max_seq_len);
  const size_t need = prompt_workspace(cfg, most, bt->max_seq_len).total;
  TS_REQUIRE(workspace_bytes >= need, TS_EWORKSPACE, "ts_prefill_prompt: workspace %zu bytes < required %zu",
             workspace_bytes, need);
  const bool cut = prompt_cuts(cfg, rows, chunk_rows, bt->max_seq_len) &&
                   workspace_bytes >= prompt_workspace(cfg, most, bt->max_seq_len, true).total;

  const hipStream_t st = (hipStream_t)stream;
  const int q_stride = q_row_stride ? q_row_stride : cfg->num_heads * cfg->head_dim;
  const int kv_stride = kv_row_stride ? kv_row_stride : cfg->num_kv_heads * cfg->head_dim;
  char* const ws = (char*)workspace;
  const auto rows_at = [&](int64_t row0, int32_t n_rows) {
    return chunk_store(cfg, (const uint16_t*)kv->k + row0 * kv_stride, (const uint16_t*)kv->v + row0 * kv_stride,
                       kv_row_stride, kv->out_cache_loc + row0, n_rows, k_pool, v_pool, pool_rows, table, seq_len,
                       kv->max_tokens);
  };
  // Bounds the length after the first `done` rows: what follows them is not there yet (unless the table
  // gets full, and rows are dropped).
  const auto bound_after = [&](int64_t done) {
    const int64_t later = bt->max_seq_len < kv->max_tokens ? rows - done : 0;
    return (int32_t)std::max<int64_t>(bt->max_seq_len - later, 1);
  };

  // The first chunks, which attend to everything before them, are one: a row's keys are the same wherever its
  // chunk ends.  Five chunks of 512, 32 heads on 8: five times a gather (5 to 8 us) and an attention (12 to 23),
  // each with the device half idle at its end, and together 9 and 79 us.  Three prompts of 700 to 5200
  // tokens + 8, two layers, 32 heads on 8: 1915 -> 1729 us.
  int dense = 0;
  while (dense < chunks && bound_after(std::min<int64_t>((dense + 1LL) * chunk_rows, rows)) <=
                               (int64_t)cfg->n_init + cfg->top_k + cfg->n_local)
    ++dense;
  // (A table that may get full: where a chunk's rows lie follows from the length after the chunk, which stops at
  // the table's end, so that they are taken one by one.)
  const int merged = bt->max_seq_len < kv->max_tokens ? std::min(dense, kPrRows / chunk_rows) : 1;
  for (int first = 0; first < dense; first += merged) {
    const int64_t row0 = (int64_t)first * chunk_rows;
    const int32_t n_rows = (int32_t)std::min<int64_t>((int64_t)std::min(merged, dense - first) * chunk_rows, rows - row0);
    const int32_t bound = bound_after(row0 + n_rows);
    const bool cut_here = cut && prefill_cuts_pay(cfg->num_heads, cfg->num_kv_heads, n_rows, n_rows, bound);
    const PromptWorkspace w = prompt_workspace(cfg, 1, bound, cut_here);
    PrefillDense all{};
    all.table = table;
    all.seq_len = seq_len;
    all.sel = (int32_t*)(ws + w.sel);
    all.sel_pos = (int32_t*)(ws + w.sel_pos);
    all.sel_len = (int32_t*)(ws + w.sel_len);
    all.list_bound = std::min(bound, kv->max_tokens);
    all.store = rows_at(row0, n_rows);
    TS_TRY(launch_prefill_attn(cfg, (const uint16_t*)q + row0 * q_stride, q_stride, n_rows, k_pool, v_pool, pool_rows,
                               all.sel, all.sel_len, bound, (uint16_t*)out + row0 * cfg->num_heads * cfg->head_dim,
                               ws + w.stage, w.total - w.stage, st, &all, cut_here ? ws + w.votes : nullptr));
  }

  if (dense == chunks) return TS_OK;
  const int rest = chunks - dense, group = (int)ceil_div(rest, ceil_div(rest, most));  // (rounds of about the same size)
  for (int first = dense; first < chunks; first += group) {
    const int here = std::min(group, chunks - first);
    const int64_t row0 = (int64_t)first * chunk_rows;
    const int32_t n_rows = (int32_t)std::min<int64_t>((int64_t)here * chunk_rows, rows - row0);
    const int32_t bound = bound_after(row0 + n_rows);
    const int max_sel = cfg->n_init + cfg->top_k + cfg->n_local;
    const bool cut_here =
        cut && prefill_cuts_pay(cfg->num_heads, cfg->num_kv_heads, n_rows, std::min(chunk_rows, n_rows), max_sel);
    const PromptWorkspace w = prompt_workspace(cfg, here, bound, cut_here);
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
    const PromptChunks pc{n_rows, std::min(chunk_rows, n_rows), here, lens, counters.base, (size_t)counters.stride,
                          counters.words};
    TS_TRY(launch_prompt_fingerprint(cfg, q0, q_stride, cos_table, sin_table, table_rows, ws + w.qf, pc,
                                     rows_at(row0, n_rows), st));

    PromptScoreArgs a{};
    a.qf = (const uint16_t*)(ws + w.qf);
    a.k_pool = (const uint4*)k_pool;
    a.pool_rows = (uint32_t)pool_rows;
    a.table = table;
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
    a.stats = (float2*)(ws + w.stats);
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
                                      w.total - w.stage, st, nullptr, cut_here ? ws + w.votes : nullptr));
  }
  return TS_OK;
}

}  // extern "C"
