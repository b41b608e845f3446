// Criticality scoring: scores[h,t] = q[h,:] . K[slot(t), kv(h), :] streamed over the
// paged KV cache (the reference's paged_matmul_kernel, tr.py:166-231), plus the
// per-head softmax statistics the soft vote needs (tr.py:361).
//
// The pass is bound by HBM: every candidate row (Hkv*256 bytes) is read exactly
// once for all H query heads.  The dot products go through the matrix cores, not
// because the shape is a dense GEMM (it is 1 to 8 query rows per KV head) but
// because one v_mfma_f32_16x16x32_bf16 replaces some 64 dot / reduce / select
// vector instructions, which is what lets a wavefront keep 32 KB of loads in
// flight instead of computing.
//
// Operand layout (lane l: rg = l/16, t4 = (l%16)/4, p = l%4).  One load
// instruction covers four tokens of a tile and one KV head: lane l reads the 16
// bytes at offset 64*rg + 16*p of token 4m + t4, so each token's 256-byte head
// row is fetched as one contiguous piece and every 128-byte line is consumed by
// a single instruction.  Seen as the B operand (column l%16, k-group rg), column
// (t4, p) holds the dims {8(4rg + p) + e} of token t4: a quarter of the head
// dimension per column.  The A operand uses the same mapping with the query head
// in place of the token, so that D[(g, p'), (t4, p)] is the partial dot product
// of query g and token t4 over quarter p when p' == p.  Each lane keeps the
// diagonal element (register p of its 4 results) and the four quarters are added
// across the 4 lanes of a quad with two DPP quad_perm adds.  After the four
// instructions of a tile (m = 0..3) lane (rg, t4, p) keeps the result of m == p:
// the score of query rg for token 4p + t4, one token per lane, 16 tokens per
// 16-lane row, stored as one 64-byte segment per head.
//
// Products of bf16 pairs are exact in fp32 and the accumulation is fp32.
// Loads are double-buffered in half iterations (16 x 128-bit loads per lane
// each) and the table entries of the next iteration are fetched one iteration
// ahead.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <type_traits>
#include <vector>

#include "ts_score.h"
#include "ts_topk.h"

namespace ts {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int HKV, int G>
__device__ __forceinline__ int head_of(int kvh, int g, int head_map) {
  return head_map == TS_HEADMAP_MOD ? kvh + HKV * g : kvh * G + g;
}

// 128-bit load with the non-temporal hint: the keys are read once, and keeping
// them out of the caches' replacement order is worth about 10 % of streaming
// bandwidth on this part.
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
__device__ __forceinline__ uint4 load_streaming(const char* p) {
  const u32x4_t v = __builtin_nontemporal_load((const u32x4_t*)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}

constexpr int kQuadSwap1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kQuadSwap2 = 0x4E;  // quad_perm [2,3,0,1]

// One iteration of a wave covers TG tiles of 16 tokens and all HKV heads: always
// 8 (tile, KV head) units = 32 loads of 1 KB.  Units 0-3 and 4-7 alternate
// between two register buffers.
//
// Output forms:
//   kScoreDirect (paged_matmul): scores[h][t] row-major in the caller's dtype,
//     stored directly.
//   kScoreTiled (the selection path, separate kernels): fp32 scores leave the
//     kernel tile-major, scores[b][tile][head slot][16 tokens] with head slot =
//     kvh*G + g.  They are staged in LDS and written once per workgroup as one
//     contiguous burst: trickling 64-byte pieces into 32 separate head rows while
//     the keys stream in costs a quarter of the read bandwidth (DRAM read/write
//     turnarounds).
//   kScoreFused (the whole selection in one launch whose workgroups are all
//     resident at once and wait for each other): the scores never leave LDS.
//     Every workgroup publishes its per-head (max, sum exp); the (request, head)
//     pairs are dealt out over the grid, merged and written to replicas that the
//     workgroups poll; every workgroup turns its own
//     scores into votes (tr.py:361); histogram rounds (11 + 11 + 10 key bits) narrow
//     the k-th largest vote down until at most 256 candidates are left, which are
//     listed and ranked by every workgroup together with the counts that tell it
//     where its selected positions, in ascending order, belong (tr.py:371-373,
//     433-449); masses of exact ties go through all three levels and a count round.
//     That is two to four rendezvous, and one more for the max-pool's neighbours; none
//     where a hint says near which bin the threshold lies and it does.
constexpr int kScoreDirect = 0, kScoreTiled = 1, kScoreFused = 2;
// The fused kernel's votes-only form (phases of requests in one launch): a kernel of its
// own, so that the single-launch selection does not carry the bookkeeping.
constexpr int kScorePacked = 3;
// kScoreFused that meets wherever the band does not do: an instantiation of its own for ts_select by itself and for votes
// pooled over wide windows, where what is sent late does not pay (kLatePool).  With that code in it, never taken, a
// chunk of 250 rows on 24K tokens with a window of 124 took 64.2 us a layer, and 63.7 so (63.4 before there was such code).
constexpr int kScoreMeeting = 4;
constexpr int kMaxHeads = 128;

// What a workgroup of the fused kernel serves: the whole launch, or one phase of a
// launch of the votes-only form.
struct LaunchPart {
  int tokens_per_block;
  int batch_offset;       // first request
  int packed;             // requests of the phase (0: the grid is [chunks, requests])
  const int* pack_first;  // first workgroup of each of them
  int x;                  // this workgroup along x
  uint32_t* sync;         // rendezvous area
};

// Chunks of request r of a phase that hold candidates: those of its n candidates, but no
// more than the phase has workgroups for it (a length above the bound the phase was sized
// by is the caller's error: the tokens beyond are not scored, and the launch reports it).
__device__ __forceinline__ int packed_chunks(const LaunchPart& lp, int r, int n) {
  const int chunks = (n + lp.tokens_per_block - 1) / lp.tokens_per_block;
  return min(chunks, lp.pack_first[r + 1] - lp.pack_first[r]);
}

// A request's length, the new token counted where this launch appends it, and that token's slot
// (kNoSlot: none).  With one request every thread knows them (`own`), else they are in LDS.
constexpr uint32_t kNoSlot = 0xffffffffu;
struct Appended {
  int len;
  uint32_t slot;
};
// (Chosen word by word: a choice between two structs puts both in memory.)
__device__ __forceinline__ Appended append_at(bool ok, int len, uint32_t slot) {
  return Appended{ok ? len + 1 : len, ok ? slot : kNoSlot};
}
struct Lengths {
  int own_len;
  uint32_t own_slot;
  int taken;  // pages that the launch takes from the pool
};
__device__ __forceinline__ Appended appended(const ScoreArgs& a, const Lengths lens, const Appended* plans, int b) {
  if (!a.appends) return Appended{a.seq_lens[b], kNoSlot};
  if (a.batch == 1) return Appended{lens.own_len, lens.own_slot};
  Appended noted = plans[b];
  // (loaded here: one load for this and the case above it would be from either of two memories)
  asm("" : "+v"(noted.len), "+v"(noted.slot));
  return noted;
}
// The kernel's arguments, read again from here on.  What the compiler can see at the start of a
// kernel it loads there and holds to the end: the scalar registers did not suffice, the first load
// waited behind 50 moves of them to vector lanes and a second round of arguments, and the phases
// after the stream began by fetching them back.
__device__ __forceinline__ const ScoreArgs& late_args() {
  auto args = (const __attribute__((address_space(4))) ScoreArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return *(const ScoreArgs*)args;
}

// The softmax statistics of the fused kernel, without a rendezvous: every workgroup
// publishes its per-head (max, sum exp) into a table that was zero at launch; the
// (request, head) pairs are dealt out over all wavefronts of the team; a wavefront polls
// the entries of its pair, a lane per chunk, until none is zero any more (a sum of
// exponentials never is: the data is its own flag), merges them in a fixed order and
// writes the result into 64 replicas, lane r into replica r.  The workgroups poll the
// words of the replica of their index in the same way.  The wait is bounded like those
// of the rendezvous: on giving up it sets the fault word and merges what is there.
template <bool PACKED>
__device__ __forceinline__ void merge_request_stats(const ScoreArgs& a, const LaunchPart& lp,
                                                    const GridTeam& team, const Lengths lens, const Appended* plans,
                                                    int lane, int wave) {
  const int H = a.num_heads;
  const int items = (PACKED ? lp.packed : a.batch) * H;
  const int first = (int)team.index * 4 + wave;
  const int step = (int)team.size * 4;
  for (int item = first; item < items; item += step) {
    const int b = lp.batch_offset + item / H, h = item % H;
    if (a.skip && a.skip[b]) continue;
    const ReqGeom geo = geometry_of_length(PACKED ? a.seq_lens[b] : appended(a, lens, plans, b).len, a.k_per_req, b, a.n_init,
                                           a.n_local, a.top_k, a.max_seq_len);
    if (geo.n <= 0) continue;
    const int chunks = PACKED ? packed_chunks(lp, item / H, geo.n)
                              : (geo.n + lp.tokens_per_block - 1) / lp.tokens_per_block;
    const float2* part = (const float2*)a.partials + ((size_t)b * H + h) * a.nchunks;
    float m = kNegBig, l = 0.f;
    const uint64_t t0 = wall_clock64();
    bool lost = false;
    for (int base = 0; base < chunks; base += 8 * 64) {  // 8 loads in flight per lane
      float2 v[8];
      for (uint32_t polls = 1;; ++polls) {
        bool there = true;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int c = base + 64 * i + lane;
          v[i] = c < chunks ? load_coherent(part + c) : make_float2(kNegBig, 0.f);
          there = there && (c >= chunks || __float_as_uint(v[i].y) != 0u);
        }
        if (__all(there) || lost) break;
        if ((polls & 7u) == 0) {
          if (load_coherent(&lp.sync[0]) != 0u) {
            lost = true;
          } else if (wall_clock64() - t0 > a.spin_ticks) {
            raise_fault(lp.sync);
            lost = true;
          }
        }
        __builtin_amdgcn_s_sleep(2);  // (a few dozen wavefronts poll)
      }
      // The maximum first, then every sum scaled to it: one exponential per entry, none of
      // them waiting for another.  (An entry past the last chunk has the weight zero.)
      float top = m;
#pragma unroll
      for (int i = 0; i < 8; ++i) top = fmaxf(top, v[i].x);
      top = fmaxf(top, dpp_move<kRowRor8>(top));
      top = fmaxf(top, dpp_move<kRowRor4>(top));
      top = fmaxf(top, dpp_move<kRowRor2>(top));
      top = fmaxf(top, dpp_move<kRowRor1>(top));
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      float add = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (base + 64 * i < chunks) add += v[i].y * __expf(v[i].x - top);
      add = row16_sum(add);
      add += __shfl_xor(add, 16);
      add += __shfl_xor(add, 32);
      l = l * __expf(m - top) + add;
      m = top;
    }
    store_coherent((float2*)(a.stats + (size_t)lane * a.stats_stride) + (size_t)b * H + h, m, l);
  }
}

constexpr int kStatsPollSleep = 4;     // x 64 clocks between a workgroup's polls for the merged statistics
constexpr uint32_t kSelectRounds = 5;  // rendezvous of the fused kernel at most (without the max-pool's)

#ifdef TS_TRACE  // development builds only: per-workgroup phase timestamps of the fused kernel
#include "ts_trace.h"
#else
#define TS_MARK(i) \
  do {             \
  } while (0)
#endif

// The workgroups that take part in the rendezvous of the fused kernel: all those of
// the requests that select (neither dense nor served by the selection cache).  The
// others write their fixed output and leave, so that a step in which every request
// hits the cache costs a few microseconds instead of empty rounds.
// (req, chunk: this workgroup's request within the launch and its chunk of that request.)
template <bool PACKED>
__device__ __forceinline__ GridTeam selecting_team(const ScoreArgs& a, const LaunchPart& lp,
                                                   uint32_t* lds, int req, int chunk) {
  GridTeam team{0u, 0u};
  if (PACKED) {
    // A phase holds a handful of requests and its members are the workgroups
    // that hold candidates: every thread adds them up for itself.
    uint32_t before = 0, total = 0;
    for (int r = 0; r < lp.packed; ++r) {
      const int b = lp.batch_offset + r;
      if (a.skip && a.skip[b]) continue;
      const int n = request_geometry(a.seq_lens, a.k_per_req, b, a.n_init, a.n_local, a.top_k,
                                     a.max_seq_len).n;
      const uint32_t members = n > 0 ? (uint32_t)packed_chunks(lp, r, n) : 0u;
      total += members;
      if (r < req) before += members;
    }
    team.size = total + a.absent;
    team.index = before + (uint32_t)chunk;
    return team;
  }
  (void)lds;
  return team;  // (the single launch deals its workgroups itself: deal_workgroups)
}

// The single-launch selection deals its workgroups on the device, from the lengths and the
// hit flags as they are at launch: only the requests that select (neither dense nor served
// by the selection cache) get workgroups, all of them the same number of tokens, the
// smallest multiple of 64 with which the requests' chunks fit the grid; consecutive
// workgroups serve consecutive chunks, request after request.  A step in which one request
// of four misses the cache thus streams that request's keys through the whole device
// instead of through the quarter a fixed [chunks, requests] grid would give it, and a
// ragged batch is spread by what the requests hold, not by the longest.  Workgroups past
// the last chunk have nothing to do.  The workgroups with tokens are the team of the
// rendezvous, in grid order.
struct Deal {
  int tokens_per_block;  // of every selecting request of this launch
  int req;               // this workgroup's request (within the launch), -1: none
  int chunk, chunks;     // its chunk of that request, and the request's chunks
  int n;                 // the request's candidates
  uint32_t team_size, team_index;
  int own_len;           // of the only request, with the new token that this launch appends,
  uint32_t own_slot;     // and that token's slot (kNoSlot: none)
  int taken;             // pages that the launch takes from the pool
};
constexpr int kDealRequests = 512;  // of a launch at most: every request has a workgroup of the grid

// Where the new tokens go, as the store kernels place them (store_step): with one request by every
// thread for itself, else by the dealing wavefront for all, a lane each (at most kCommitBatch of them).
// Pages: the rank of the only request that may need one is zero.
__device__ __forceinline__ void plan_append_one(const ScoreArgs& a, int len, Deal& d) {
  const StepStore& st = late_args().append;
  if (st.free_pages == nullptr) {
    const int slot = st.loc[0];
    const bool ok = append_fits(slot, len, st.pool_rows, st.max_tokens);
    d.own_len = ok ? len + 1 : len;
    d.own_slot = ok ? (uint32_t)slot : kNoSlot;
    return;
  }
  const int page_mask = (1 << st.page_shift) - 1, count = max(*st.free_count, 0);
  const bool room = len >= 0 && len < st.max_tokens, need = room && (len & page_mask) == 0;
  const AppendPlan p = make_append_plan(st.table, len, room, need, 0u, count, st.free_pages, st.page_shift, page_mask,
                                        (uint32_t)st.pool_rows);
  d.taken = need ? min(1, count) : 0;
  d.own_len = p.ok ? len + 1 : len;
  d.own_slot = p.ok ? p.slot : kNoSlot;
}
__device__ __forceinline__ int plan_appends(const ScoreArgs& a, int lane, Appended* plans) {
  const StepStore& st = late_args().append;
  if (st.free_pages == nullptr) {
    if (lane < a.batch) {
      const int len = st.seq_lens[lane], slot = st.loc[lane];
      const bool ok = append_fits(slot, len, st.pool_rows, st.max_tokens);
      plans[lane] = append_at(ok, len, (uint32_t)slot);
    }
    return 0;
  }
  const PagePool pool{st.free_pages, st.free_count, st.ticket};
  return for_each_append(st.seq_lens, st.table, st.table_stride, a.batch, pool, st.page_shift, st.max_tokens,
                         (uint32_t)st.pool_rows, lane, [&](int b, const AppendPlan& p) {
                           plans[b] = append_at(p.ok, p.len, p.slot);
                         });
}

__device__ __forceinline__ int wave_sum(int x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// (cand: LDS of kDealRequests words, free again when this returns.  The loops over the requests are
// rolled up and hold them there: unrolled over registers they were 2000 instructions at the head of
// the kernel that one request skips, and a selection's start is bound by what it fetches of them.)
__device__ __forceinline__ Deal deal_workgroups(const ScoreArgs& a, int* lds, int* cand, Appended* plans) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int B = a.batch, T = (int)gridDim.x, w = (int)blockIdx.x;
  if (__builtin_expect(B == 1, 1)) {  // one request: every thread works it out for itself, no exchange
    Deal d{a.tokens_per_block, -1, 0, 0, 0, a.absent, (uint32_t)w, 0, kNoSlot, 0};
    int n = 0;
    d.own_len = a.seq_lens[a.batch_offset];
    if (__builtin_expect(a.appends != 0, 0)) plan_append_one(a, d.own_len, d);
    if (!(a.skip && a.skip[a.batch_offset]))
      n = geometry_of_length(d.own_len, a.k_per_req, a.batch_offset, a.n_init, a.n_local, a.top_k,
                             a.max_seq_len).n;
    if (n <= 0) return d;
    d.n = n;
    int tpb = max((n + T * 64 - 1) / (T * 64) * 64, 64);
    while ((n + tpb - 1) / tpb > T && tpb < a.tokens_per_block) tpb += 64;
    d.tokens_per_block = tpb;
    d.chunks = (n + tpb - 1) / tpb;
    d.team_size = (uint32_t)d.chunks + a.absent;
    if (w < d.chunks) {
      d.req = 0;
      d.chunk = w;
    }
    return d;
  }
  if (tid < 64) {
    const int taken = a.appends ? plan_appends(a, lane, plans) : 0;
    // Every request's candidates if it selects, else 0.
    int all = 0;  // (what one launch holds fits the LDS of the device: far below 2^31)
#pragma unroll 1
    for (int b = lane; b < B; b += 64) {
      int len = 0, n = 0;
      if (a.appends) len = plans[b].len;
      asm("" : "+v"(len));  // (or the two loads become one, from either of two memories)
      if (!a.appends) len = a.seq_lens[a.batch_offset + b];
      if (!(a.skip && a.skip[a.batch_offset + b]))
        n = geometry_of_length(len, a.k_per_req, a.batch_offset + b, a.n_init, a.n_local, a.top_k, a.max_seq_len).n;
      cand[b] = n;
      all += n;
    }
    const long long total_n = wave_sum(all);
    // Fewest tokens per workgroup that could do, then upwards until the chunks fit (a step
    // or two: the rounding of every request's last chunk).  The launch's own figure always
    // fits: the host sized the grid for every request at the longest length.
    int tpb = (int)((total_n + (long long)T * 64 - 1) / ((long long)T * 64)) * 64;
    tpb = max(tpb, 64);
    for (;; tpb += 64) {
      int mine = 0;
#pragma unroll 1
      for (int b = lane; b < B; b += 64) mine += (cand[b] + tpb - 1) / tpb;
      if (wave_sum(mine) <= T || tpb >= a.tokens_per_block) break;
    }
    // First workgroup of every request, in request order, 64 of them at a time.
    int base = 0, req = -1, chunk = 0, req_chunks = 0, req_n = 0;
#pragma unroll 1
    for (int b0 = 0; b0 < B; b0 += 64) {
      const int n = b0 + lane < B ? cand[b0 + lane] : 0;
      const int chunks = (n + tpb - 1) / tpb;
      int incl = chunks;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
      }
      const int first = base + incl - chunks;
      const uint64_t who = __ballot(w >= first && w < first + chunks);
      if (who) {
        const int src = __ffsll((unsigned long long)who) - 1;
        req = b0 + src;
        chunk = w - __shfl(first, src);
        req_chunks = __shfl(chunks, src);
        req_n = __shfl(n, src);
      }
      base += __shfl(incl, 63);
    }
    if (lane == 0) {
      lds[0] = tpb;
      lds[1] = req;
      lds[2] = chunk;
      lds[3] = req_chunks;
      lds[4] = base;  // workgroups with tokens: the team
      lds[5] = req_n;
      lds[6] = taken;
    }
  }
  __syncthreads();
  Deal d;
  d.tokens_per_block = lds[0];
  d.req = lds[1];
  d.chunk = lds[2];
  d.chunks = lds[3];
  d.n = lds[5];
  d.own_len = 0;
  d.own_slot = kNoSlot;
  d.taken = lds[6];
  d.team_size = (uint32_t)lds[4] + a.absent;
  d.team_index = (uint32_t)w;
  __syncthreads();
  return d;
}

// The new token of request b, by one workgroup: its rows to the pool, and the note of what the
// attention kernel is to write.
__device__ __forceinline__ void append_token(const ScoreArgs& a, int b, const Appended& now, int taken) {
  const StepStore& st = late_args().append;
  const bool ok = now.slot != kNoSlot;
  if (ok)
    for (int i = threadIdx.x; i < st.row_vec; i += 256) {
      const uint4 k = st.k[(size_t)b * st.kv_stride + i], v = st.v[(size_t)b * st.kv_stride + i];
      st.k_pool[(size_t)now.slot * st.row_vec + i] = k;
      st.v_pool[(size_t)now.slot * st.row_vec + i] = v;
    }
  if (threadIdx.x == 0) {
    const int at = now.len - 1;
    const bool entry = ok && (at & ((1 << st.page_shift) - 1)) == 0;
    a.notes[b] = make_int4(ok ? now.len : -1, at >> st.page_shift, entry ? (int)(now.slot >> st.page_shift) : -1, taken);
  }
}

// The parts of the output that need no votes, written while the statistics are on their way: a
// dense request gets all its positions and a selection-cache hit its cached ones
// (both spread over the request's workgroups); workgroup 0 of a request writes the
// length, the sink and the local window, and clears the words the next kernel of
// the stream wants cleared.
// (x of nx: this workgroup among those that write the request's fixed parts.)
__device__ __forceinline__ void fixed_segments(const ScoreArgs& a, const Lengths lens, const Appended* plans, int b, int x,
                                               int nx) {
  const Appended now = appended(a, lens, plans, b);
  const ReqGeom geo =
      geometry_of_length(now.len, a.k_per_req, b, a.n_init, a.n_local, a.top_k, a.max_seq_len);
  if (x == 0 && a.appends) append_token(a, b, now, b == 0 ? lens.taken : 0);
  const int new_pos = now.slot == kNoSlot ? -1 : now.len - 1;  // (the table does not know its slot yet)
  const int32_t* tab = a.table + (int64_t)b * a.table_stride;
  int32_t* sel = a.sel + (int64_t)b * a.sel_stride;
  int32_t* sel_pos = a.sel_pos + (int64_t)b * a.sel_stride;
  const int L = geo.seq_len;
  const int first = x * 256 + threadIdx.x, step = nx * 256;
  auto emit = [&](int out_idx, int pos) {
    sel_pos[out_idx] = pos;
    sel[out_idx] = (int32_t)(pos == new_pos ? now.slot : lookup_slot(tab, pos, a.page_size, a.page_shift, a.pool_rows));
  };
  if (x == 0 && a.clear)
    for (int i = threadIdx.x; i < a.clear_per_req; i += 256)
      a.clear[(size_t)b * a.clear_per_req + i] = 0u;
  if (geo.dense) {  // tr.py:377-378, 741-744: attend over every token
    for (int i = first; i < L; i += step) emit(i, i);
    if (first == 0) a.sel_len[b] = L;
    return;
  }
  const bool is_hit = a.skip && a.skip[b];
  const int k = is_hit ? min(a.cache_len[b], a.top_k) : geo.k;
  if (is_hit) {  // tr.py:419: reuse the cached positions
    const int32_t* cached = a.topk_cache + (int64_t)b * a.top_k;
    for (int i = first; i < k; i += step) emit(a.n_init + i, cached[i]);
  }
  if (x != 0) return;
  if (threadIdx.x == 0) {
    // (The length of a request that selects is written when its selection is through, by
    // the workgroup that also reports a wait that gave up: one writer, one order.)
    if (is_hit) a.sel_len[b] = a.n_init + k + a.n_local;
    if (!is_hit && a.cache_len) a.cache_len[b] = k;
  }
  for (int i = threadIdx.x; i < a.n_init; i += 256) emit(i, i);
  for (int i = threadIdx.x; i < a.n_local; i += 256) emit(a.n_init + k + i, L - a.n_local + i);
}

// Sum over the 16 lanes of a DPP row, in every lane of it.
__device__ __forceinline__ uint32_t row16_total(uint32_t x) {
  auto ror = [](uint32_t v, auto ctrl) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false);
  };
  x += ror(x, std::integral_constant<int, kRowRor8>{});
  x += ror(x, std::integral_constant<int, kRowRor4>{});
  x += ror(x, std::integral_constant<int, kRowRor2>{});
  x += ror(x, std::integral_constant<int, kRowRor1>{});
  return x;
}
// Sum over the wavefront, in every lane.
__device__ __forceinline__ uint32_t wave_total(uint32_t x) {
  x = row16_total(x);
  return (uint32_t)(__builtin_amdgcn_readlane((int)x, 0) + __builtin_amdgcn_readlane((int)x, 16) +
                    __builtin_amdgcn_readlane((int)x, 32) + __builtin_amdgcn_readlane((int)x, 48));
}

// Bits set in any lane of the wavefront, in every lane.
__device__ __forceinline__ uint32_t wave_or(uint32_t x) {
  auto ror = [](uint32_t v, auto ctrl) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false);
  };
  x |= ror(x, std::integral_constant<int, kRowRor8>{});
  x |= ror(x, std::integral_constant<int, kRowRor4>{});
  x |= ror(x, std::integral_constant<int, kRowRor2>{});
  x |= ror(x, std::integral_constant<int, kRowRor1>{});
  return (uint32_t)(__builtin_amdgcn_readlane((int)x, 0) | __builtin_amdgcn_readlane((int)x, 16) |
                    __builtin_amdgcn_readlane((int)x, 32) | __builtin_amdgcn_readlane((int)x, 48));
}

// This workgroup's share of the launch's parts that need no votes: counted from the last
// workgroup down, those of request w % B, as one of the workgroups w % B, w % B + B, ...
// (The first workgroups of the team merge the statistics, and everybody waits for those; the
// last ones often have no candidates.)
__device__ __forceinline__ void fixed_parts(const ScoreArgs& a, const Lengths lens, const Appended* plans) {
  const int B = a.batch, T = (int)gridDim.x, w = T - 1 - (int)blockIdx.x;
  fixed_segments(a, lens, plans, a.batch_offset + w % B, w / B, (T - w % B + B - 1) / B);
}

// Adds the wavefront's candidates to a histogram in memory with one fetch-add per
// distinct bin: normally a wavefront has a few candidates in different bins, but
// nearly uniform votes (a query of small norm) put all 64 lanes, of every wavefront,
// into the same bin, and that many single increments of one address take
// milliseconds.  Returns the old values (to be awaited).  Every lane of the wavefront
// must call it.
__device__ __forceinline__ uint32_t wave_histogram_add(uint32_t* hist, bool have, uint32_t bin,
                                                      int lane) {
  uint32_t done = 0;
  uint64_t todo = __ballot(have);
  while (todo) {
    const int leader = __ffsll((unsigned long long)todo) - 1;
    const uint32_t leader_bin = (uint32_t)__shfl((int)bin, leader);
    const uint64_t same = __ballot(have && bin == leader_bin) & todo;
    // Little sharing: the remaining lanes add on their own, in one instruction (a
    // wavefront whose 64 candidates sit in 64 bins must not issue 64 of them).
    if (__popcll(same) < 4) break;
    if (lane == leader) done += fetch_add_coherent(&hist[leader_bin], (uint32_t)__popcll(same));
    todo &= ~same;
  }
  if ((todo >> lane) & 1ull) done += fetch_add_coherent(&hist[bin], 1u);
  return done;
}

// 256 threads, thread 0 holding the highest bin: finds the thread at which the
// running count (from thread 0 on) reaches `need`.  Returns that thread's index
// (or -1 if the total stays below `need`), the count before it, the total, and
// that thread's own count.  `scratch` is LDS of 8 words.
__device__ __forceinline__ int block_threshold_scan(uint32_t mine, uint32_t need, uint32_t* scratch,
                                                    uint32_t& before_out, uint32_t& total_out,
                                                    uint32_t& count_out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
  if (lane == 63) scratch[wave] = incl;
  if (tid == 0) scratch[4] = 0xffffffffu;
  __syncthreads();
  uint32_t wave_base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) wave_base += scratch[w];
    total += scratch[w];
  }
  const uint32_t before = wave_base + incl - mine;
  if (before < need && need <= before + mine) {
    scratch[4] = (uint32_t)tid;
    scratch[5] = before;
    scratch[6] = mine;
  }
  __syncthreads();
  const uint32_t who = scratch[4];
  before_out = scratch[5];
  count_out = scratch[6];
  total_out = total;
  __syncthreads();
  return who == 0xffffffffu ? -1 : (int)who;
}

// Votes-only launches: a phase ends with the memory idle while its statistics are on
// their way, and when a request takes the whole device no other phase streams meanwhile.
// The wavefronts that do not poll for the statistics touch the first keys of the
// workgroup that is going to take this one's place: `resident` workgroups further on in
// the grid, hence on the same XCD, whose L2 then holds what each of that workgroup's
// wavefronts asks for first.  One 4-byte load per 128-byte line; the values are only
// kept so that the loads are (the caller hands them to an empty asm at its end).
// Eight tokens per wavefront of the successor (64 KB per workgroup at eight KV heads, 2 MB
// per XCD): C5 layer 425 -> 420 us, C3 442 -> 438 us; 16 tokens bring less, 24 are slower
// than none (the L2 of an XCD holds 4 MB).
constexpr int kAheadTokens = 8;
constexpr int kAheadLoads = (4 * kAheadTokens * 16 + 191) / 192;  // per lane, at 16 lines per row
template <int HKV>
__device__ __forceinline__ void touch_successor_keys(const ScoreArgs& a, int wave, int lane,
                                                     uint32_t (&got)[kAheadLoads]) {
  constexpr uint32_t ROW_BYTES = HKV * kHeadDim * 2;
  constexpr int kLines = (int)ROW_BYTES / 128;
  constexpr int kItems = 4 * kAheadTokens * kLines;
  static_assert(kItems <= kAheadLoads * 192, "three wavefronts cover the lines");
#pragma unroll
  for (int i = 0; i < kAheadLoads; ++i) got[i] = 0u;
  const int g = (int)blockIdx.x + a.resident;
  if (a.resident <= 0 || g >= (int)gridDim.x) return;
  int phase = 0;
  while (phase + 1 < a.nphases && g >= a.phases[phase + 1].first_workgroup) ++phase;
  const VotePhase& ph = a.phases[phase];
  const int x = g - ph.first_workgroup;
  int req = 0;
  while (req + 1 < ph.requests && x >= ph.pack_first[req + 1]) ++req;
  const int b = ph.first + req;
  if (a.skip && a.skip[b]) return;
  const ReqGeom geo =
      request_geometry(a.seq_lens, a.k_per_req, b, a.n_init, a.n_local, a.top_k, a.max_seq_len);
  const int block_lo = (x - ph.pack_first[req]) * ph.tokens_per_block;
  if (block_lo >= geo.n) return;
  const int per_wave = ph.tokens_per_block >> 2;
  const int32_t* tab = a.table + (int64_t)b * a.table_stride;
#pragma unroll
  for (int i = 0; i < kAheadLoads; ++i) {
    const int item = (wave - 1) * 64 + lane + 192 * i;
    if (item < kItems) {
      const int t = item / kLines, line = item % kLines;
      const int tok = min(block_lo + (t / kAheadTokens) * per_wave + t % kAheadTokens, geo.n - 1);
      const int pos = a.n_init + tok;
      uint32_t slot = ((uint32_t)tab[pos >> a.page_shift] << a.page_shift) + (uint32_t)(pos & (a.page_size - 1));
      slot = slot < a.pool_rows ? slot : a.pool_rows - 1;
      got[i] = *(const uint32_t*)((const char*)a.k_pool + (size_t)slot * ROW_BYTES + line * 128);
    }
  }
}

template <int HKV, int G, bool OUT_BF16, int MODE>
__global__ __launch_bounds__(256, (G > 4 ? 1 : 2)) void score_kernel(ScoreArgs a) {
  extern __shared__ float stage[];  // tiled / fused: [tiles of the workgroup][tile_stride]
  constexpr bool TILED = MODE != kScoreDirect;
  constexpr bool LATE = MODE == kScoreFused;
  constexpr bool FUSED = LATE || MODE == kScoreMeeting || MODE == kScorePacked;
  constexpr bool PACKED = MODE == kScorePacked;
  constexpr int TG = 8 / HKV;
  constexpr int UNITS = 8;
  constexpr int HALF = UNITS / 2;
  constexpr int NA = (G + 3) / 4;  // A operands (4 query heads each) per KV head
  constexpr int ITER = 16 * TG;    // tokens per iteration
  constexpr uint32_t ROW_BYTES = HKV * kHeadDim * 2;

  constexpr bool SHARED_QUERY = FUSED && !PACKED;  // the query operands are shared in LDS (below)
  constexpr bool RAW = SHARED_QUERY;               // and the query may be un-rotated (a.q_raw)
  constexpr int OPS = HKV * NA, MINE = (OPS + 3) / 4;
  // One after the other: the requests while they are dealt, the query operands, the histogram.
  constexpr int LH = SHARED_QUERY && OPS * 256 > kTopkBins ? OPS * 256 : kTopkBins;
  static_assert(LH >= kDealRequests, "a word per request");
  __shared__ __attribute__((aligned(16))) uint32_t lh[FUSED ? LH : 4];

  // This workgroup's request within the launch, and its chunk of that request.
  LaunchPart lp{a.tokens_per_block, a.batch_offset, 0, nullptr, (int)blockIdx.x, a.sync};
  int req = blockIdx.y, chunk = blockIdx.x;
  int req_chunks = (int)gridDim.x;  // chunks of this workgroup's request (the single launch: dealt)
  int dealt_n = 0;
  int own_len = 0, taken = 0;
  uint32_t own_slot = kNoSlot;
  __shared__ Appended plans[FUSED && !PACKED ? kCommitBatch : 1];
  GridTeam team{0u, 0u};
  if (PACKED) {
    TS_MARK(0);
    // This workgroup's phase, and its request and chunk within the phase.
    int phase = 0;
    while (phase + 1 < a.nphases && (int)blockIdx.x >= a.phases[phase + 1].first_workgroup) ++phase;
    const VotePhase& ph = a.phases[phase];
    lp = LaunchPart{ph.tokens_per_block, ph.first, ph.requests, ph.pack_first,
                      (int)blockIdx.x - ph.first_workgroup, a.sync + (size_t)phase * kSyncWords};
    req = 0;
    while (req + 1 < lp.packed && lp.x >= lp.pack_first[req + 1]) ++req;
    chunk = lp.x - lp.pack_first[req];
  }
  if constexpr (FUSED && !PACKED) {
    __shared__ int deal_lds[8];
    TS_MARK(0);
    const Deal deal = deal_workgroups(a, deal_lds, (int*)lh, plans);
    own_len = deal.own_len;
    own_slot = deal.own_slot;
    taken = deal.taken;
    if (__builtin_expect(deal.req < 0, 0)) {  // no chunk left for this workgroup
      fixed_parts(late_args(), Lengths{own_len, own_slot, taken}, plans);
      return;
    }
    lp.tokens_per_block = deal.tokens_per_block;
    req = deal.req;
    chunk = deal.chunk;
    req_chunks = deal.chunks;
    dealt_n = deal.n;
    team = GridTeam{deal.team_size, deal.team_index};
  }
  const int b = req + lp.batch_offset;
  int n, first_pos;
  if (FUSED && !PACKED) {
    n = dealt_n;
    first_pos = a.n_init;
  } else if (a.direct_n >= 0) {
    n = (int)a.direct_n;
    first_pos = 0;
  } else {
    ReqGeom geo = request_geometry(a.seq_lens, a.k_per_req, b, a.n_init, a.n_local, a.top_k,
                                   a.max_seq_len);
    n = (a.skip && a.skip[b]) ? 0 : geo.n;
    first_pos = a.n_init;
  }
  const int block_lo = chunk * lp.tokens_per_block;
  // (asked for here, long before it is used: the bin of the request's last selection)
  const int hint_word = (FUSED && !PACKED && a.hint) ? a.hint[b] : 0;
  if constexpr (PACKED) {
    __shared__ uint32_t team_lds[8];
    if (n <= 0) return;  // dense or served by the cache: nothing to select, not on the team
    if (block_lo >= n) return;  // no candidates here, and the team is made without it
    if (chunk == 0 && threadIdx.x == 0 &&
        (n + lp.tokens_per_block - 1) / lp.tokens_per_block > lp.pack_first[req + 1] - lp.pack_first[req])
      __hip_atomic_store(&lp.sync[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // length above its bound
    team = selecting_team<PACKED>(a, lp, team_lds, req, chunk);
  }
  if (block_lo >= n) return;  // (a dealt workgroup always has tokens)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rg = lane >> 4;        // k-group of the operands, row group of the result
  const int t4 = (lane & 15) >> 2;  // token of a 4-token group / query of a 4-query group
  const int p = lane & 3;           // quarter of the head dimension
  const uint32_t lane_off = (uint32_t)(rg * 64 + p * 16);
  const int H = a.num_heads;
  // Fused: one spare row per tile keeps the four tiles a wavefront reads in the
  // vote phase on different LDS banks.
  const int tile_stride = FUSED ? 16 * H + 16 : 16 * H;
  const int32_t* tab = a.table + (int64_t)b * a.table_stride;

  // A operands: query 4*na + t4 of each KV head, same byte offsets as the keys.  In the single
  // launch the four wavefronts share the work of preparing them: wavefront w loads the operands w,
  // w + 4, ... (one of which is also rotated where the kernel does that itself: the 8 dims 64
  // further on and the rotation's rows are loaded too) and hands them over in LDS.  Only the table
  // entries stand before the first keys; the queries arrive and are rotated while the keys
  // travel (every wavefront preparing all operands first, the first key was asked for 3.3 us
  // into a selection from 32K tokens that takes 27).
  // The other forms have rotated queries, and workgroups that follow each other on a CU: a
  // wavefront loads its own, and one without tokens asks for no keys.  Shared in LDS they cost
  // a barrier between every workgroup's first keys and its first product, and keys asked for
  // by wavefronts without tokens are bytes.  Votes of 9 x 60K tokens, seven heads per KV head:
  // 159.4 us shared, 155.4 without the barrier, 149.1 without those keys either; 18 x 20K 97.3,
  // 95.8 and 93.4; scores alone of 8 x 20K 54.0, 52.9 and 50.5; with four heads per KV head (16 x
  // 68K, 4 x 256K) all within the spread.
  const bool raw = RAW && a.q_raw != nullptr;
  const bool lower = rg < 2;
  uint4 q_own[MINE], q_other[MINE];
  float4 q_cs[2], q_sn[2];
  auto load_queries = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int op = min(wave + 4 * i, OPS - 1), kvh = op / NA, g = 4 * (op % NA) + t4;
      const int h = head_of<HKV, G>(kvh, g < G ? g : 0, a.head_map);
      const char* qrow = raw ? (const char*)(a.q_raw + (size_t)b * a.q_stride + h * kHeadDim)
                             : (const char*)(a.qf + ((size_t)b * H + h) * kHeadDim);
      q_own[i] = *(const uint4*)(qrow + lane_off);
      if (RAW) q_other[i] = *(const uint4*)(qrow + (lower ? lane_off + 128u : lane_off - 128u));
    }
    if (RAW) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {  // (q_cos and q_sin are readable whether or not they are used)
        q_cs[i] = *(const float4*)((const char*)a.q_cos + 2 * lane_off + 16 * i);
        q_sn[i] = *(const float4*)((const char*)a.q_sin + 2 * lane_off + 16 * i);
      }
    }
  };
  auto share_queries = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int op = wave + 4 * i, g = 4 * (op % NA) + t4;
      uint4 v = q_own[i];
      if (RAW && raw) {
        // The caller's un-rotated query: this lane's 8 dims and the 8 dims 64 further on (or
        // back), rotated as the rotation kernel does it.
        const uint32_t ow[4] = {v.x, v.y, v.z, v.w};
        const uint32_t th[4] = {q_other[i].x, q_other[i].y, q_other[i].z, q_other[i].w};
        const float cs[8] = {q_cs[0].x, q_cs[0].y, q_cs[0].z, q_cs[0].w, q_cs[1].x, q_cs[1].y, q_cs[1].z, q_cs[1].w};
        const float sn[8] = {q_sn[0].x, q_sn[0].y, q_sn[0].z, q_sn[0].w, q_sn[1].x, q_sn[1].y, q_sn[1].z, q_sn[1].w};
        uint32_t r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = rotate_element(bf16_lo(ow[e]), bf16_lo(th[e]), cs[2 * e], sn[2 * e], lower);
          const float hi = rotate_element(bf16_hi(ow[e]), bf16_hi(th[e]), cs[2 * e + 1], sn[2 * e + 1], lower);
          r[e] = (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16);
        }
        v = make_uint4(r[0], r[1], r[2], r[3]);
      }
      if (g >= G) v = make_uint4(0u, 0u, 0u, 0u);
      if (op < OPS) *(uint4*)&lh[op * 256 + lane * 4] = v;
    }
  };

  bf16x8_t qa[HKV][NA];
  float run_m[HKV][NA], run_l[HKV][NA];
#pragma unroll
  for (int kvh = 0; kvh < HKV; ++kvh)
#pragma unroll
    for (int na = 0; na < NA; ++na) {
      run_m[kvh][na] = kNegBig;
      run_l[kvh][na] = 0.f;
    }

  const int per_wave = lp.tokens_per_block >> 2;
  const int wave_lo = block_lo + wave * per_wave;
  const int wave_hi = min(wave_lo + per_wave, n);

  // Lane (rg, t4, p) addresses tokens tile + 4m + t4, m = 0..3, of every tile.
  // The table loads and the slot arithmetic are split so that the entries of the
  // next iteration are requested a whole iteration before they are needed.
  // Positions past the wave's range are clamped to its last token: every load
  // stays in bounds and no branch splits the load pipeline.
  const int last_pos = first_pos + max(wave_hi - 1, 0);
  const int page_mask = a.page_size - 1;
  auto table_entry = [&](int tok) -> int32_t {
    const int pos = min(first_pos + tok, last_pos);
    return tab[pos >> a.page_shift];
  };
  // Byte offset of this lane's 16 bytes inside the pool.  Offsets, not pointers,
  // are carried across iterations: a pointer rebuilt from the kernel argument at
  // the load is known to be global memory, whereas a loop-carried pointer decays
  // to a flat access, whose completion the wave must wait for in full.
  auto row_off = [&](int32_t entry, int tok) -> size_t {
    const int pos = min(first_pos + tok, last_pos);
    uint32_t slot = ((uint32_t)entry << a.page_shift) + (uint32_t)(pos & page_mask);
    slot = slot < a.pool_rows ? slot : a.pool_rows - 1;
    return (size_t)slot * ROW_BYTES + lane_off;
  };
  const char* const pool = (const char*)a.k_pool;

  // Lane-constant bit masks: all ones where p == i.  Selecting with and/or keeps
  // the loop free of branches (a ternary chain on p is lowered to a switch).
  uint32_t pmask[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    pmask[i] = p == i ? 0xffffffffu : 0u;
    asm volatile("" : "+v"(pmask[i]));
  }

  uint4 buf0[HALF][4], buf1[HALF][4];
  auto issue = [&](uint4 (&buf)[HALF][4], auto& rows, int first_unit) {
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
      const int u = first_unit + i;
#pragma unroll
      for (int m = 0; m < 4; ++m)
        buf[i][m] = load_streaming(pool + rows[u / HKV][m] + (u % HKV) * (kHeadDim * 2));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // res[u][na]: score of query 4*na + rg (of the unit's KV head) for token
  // tile + 4p + t4.
  auto multiply = [&](const uint4 (&buf)[HALF][4], float (&res)[UNITS][NA], int first_unit) {
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
      const int u = first_unit + i;
#pragma unroll
      for (int na = 0; na < NA; ++na) {
        uint32_t keep = 0u;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
          const f32x4_t d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              qa[u % HKV][na], __builtin_bit_cast(bf16x8_t, buf[i][m]), zero, 0, 0, 0);
          float v = __uint_as_float((__float_as_uint(d[0]) & pmask[0]) | (__float_as_uint(d[1]) & pmask[1]) |
                                    (__float_as_uint(d[2]) & pmask[2]) | (__float_as_uint(d[3]) & pmask[3]));
          v += dpp_move<kQuadSwap1>(v);
          v += dpp_move<kQuadSwap2>(v);
          keep |= __float_as_uint(v) & pmask[m];
        }
        res[u][na] = __uint_as_float(keep);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  size_t rows_cur[TG][4];
  size_t rows_next[TG][4];
  if constexpr (!SHARED_QUERY) {
#pragma unroll
    for (int kvh = 0; kvh < HKV; ++kvh)
#pragma unroll
      for (int na = 0; na < NA; ++na) {
        const int g = 4 * na + t4;
        const int h = head_of<HKV, G>(kvh, g < G ? g : 0, a.head_map);
        uint4 v = *(const uint4*)((const char*)(a.qf + ((size_t)b * H + h) * kHeadDim) + lane_off);
        if (g >= G) v = make_uint4(0u, 0u, 0u, 0u);
        qa[kvh][na] = __builtin_bit_cast(bf16x8_t, v);
      }
  }
  if (SHARED_QUERY || wave_lo < wave_hi) {
    // (in the single launch a wavefront without tokens asks too, for its request's last ones:
    // behind a branch the compiler would wait for the queries' loads where it joins)
    int32_t entry_first[TG][4];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m) entry_first[t][m] = table_entry(wave_lo + 16 * t + 4 * m + t4);
    if constexpr (SHARED_QUERY) {
      load_queries();  // (in flight together with the table entries)
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m) rows_cur[t][m] = row_off(entry_first[t][m], wave_lo + 16 * t + 4 * m + t4);
    issue(buf0, rows_cur, 0);
  }
  if constexpr (SHARED_QUERY) {
    share_queries();
    __syncthreads();
#pragma unroll
    for (int kvh = 0; kvh < HKV; ++kvh)
#pragma unroll
      for (int na = 0; na < NA; ++na)
        qa[kvh][na] = __builtin_bit_cast(bf16x8_t, *(const uint4*)&lh[(kvh * NA + na) * 256 + lane * 4]);
  }

  for (int base = wave_lo; base < wave_hi; base += ITER) {
    int32_t entry_next[TG][4];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m) entry_next[t][m] = table_entry(base + ITER + 16 * t + 4 * m + t4);
    __builtin_amdgcn_sched_barrier(0);

    float res[UNITS][NA];
    issue(buf1, rows_cur, HALF);
    multiply(buf0, res, 0);
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m)
        rows_next[t][m] = row_off(entry_next[t][m], base + ITER + 16 * t + 4 * m + t4);
    issue(buf0, rows_next, 0);
    multiply(buf1, res, HALF);
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m) rows_cur[t][m] = rows_next[t][m];

#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int t = u / HKV, kvh = u % HKV;
      const int tok = base + 16 * t + 4 * p + t4;
#pragma unroll
      for (int na = 0; na < NA; ++na) {
        const int g = 4 * na + rg;
        if (g < G && tok < wave_hi) {
          const int h = head_of<HKV, G>(kvh, g, a.head_map);
          const float x = res[u][na];
          if (TILED) {
            stage[((tok - block_lo) >> 4) * tile_stride + (kvh * G + g) * 16 + (tok & 15)] = x;
          } else {
            const size_t at = ((size_t)b * H + h) * (size_t)a.score_stride + (size_t)tok;
            if (OUT_BF16)
              ((uint16_t*)a.scores)[at] = f32_to_bf16(x);
            else
              ((float*)a.scores)[at] = x;
          }
          // Online (max, sum exp) with a single exponential per element.
          const float d = x - run_m[kvh][na];
          const float e = __expf(-fabsf(d));
          if (d > 0.f) {
            run_l[kvh][na] = run_l[kvh][na] * e + 1.f;
            run_m[kvh][na] = x;
          } else {
            run_l[kvh][na] += e;
          }
        }
      }
    }
  }

  if (MODE == kScoreTiled) {  // one contiguous burst per workgroup
    __syncthreads();
    const int tiles = (min(lp.tokens_per_block, n - block_lo) + 15) >> 4;
    float4* dst = (float4*)((float*)a.scores + ((size_t)b * a.score_stride + block_lo) * H);
    const float4* src = (const float4*)stage;
    for (int i = threadIdx.x; i < tiles * H * 4; i += 256) dst[i] = src[i];
  }
  if (a.partials == nullptr) return;

  // Per-workgroup (max, sum exp) of every head: 16 lanes of a row, then 4 waves, each time the
  // maximum first and then one exponential per sum, none waiting for another.  (Pairs merged step by
  // step, two exponentials each, were 1 us of the 2.1 between the last product and the published
  // statistics.)
  __shared__ float local_max[FUSED ? kMaxHeads : 1];  // by head slot
  __shared__ float sm_m[4][4][HKV][NA];
  __shared__ float sm_l[4][4][HKV][NA];
#pragma unroll
  for (int kvh = 0; kvh < HKV; ++kvh)
#pragma unroll
    for (int na = 0; na < NA; ++na) {
      float m = run_m[kvh][na];
      m = fmaxf(m, dpp_move<kRowRor8>(m));
      m = fmaxf(m, dpp_move<kRowRor4>(m));
      m = fmaxf(m, dpp_move<kRowRor2>(m));
      m = fmaxf(m, dpp_move<kRowRor1>(m));
      const float l = row16_sum(run_l[kvh][na] * __expf(run_m[kvh][na] - m));
      if ((lane & 15) == 0) {
        sm_m[wave][rg][kvh][na] = m;
        sm_l[wave][rg][kvh][na] = l;
      }
    }
  __syncthreads();
  if ((int)threadIdx.x < 4 * HKV * NA) {
    const int na = threadIdx.x % NA;
    const int kvh = (threadIdx.x / NA) % HKV;
    const int g4 = threadIdx.x / (NA * HKV);
    const int g = 4 * na + g4;
    if (g < G) {
      float m = sm_m[0][g4][kvh][na], l = 0.f;
#pragma unroll
      for (int w = 1; w < 4; ++w) m = fmaxf(m, sm_m[w][g4][kvh][na]);
#pragma unroll
      for (int w = 0; w < 4; ++w) l += sm_l[w][g4][kvh][na] * __expf(sm_m[w][g4][kvh][na] - m);
      const int h = head_of<HKV, G>(kvh, g, a.head_map);
      float2* out = (float2*)a.partials + ((size_t)b * H + h) * a.nchunks + chunk;
      if (FUSED) {
        store_coherent(out, m, l);
        local_max[kvh * G + g] = m;
      } else {
        *out = make_float2(m, l);
      }
    }
  }

  if constexpr (FUSED) {
    const ScoreArgs& a = late_args();
    const int32_t* tab = a.table + (int64_t)b * a.table_stride;
    __shared__ float s_rz[kMaxHeads];
    __shared__ uint32_t scratch[16];
    const int tid = threadIdx.x;
    static_assert(kBandSlots == 4, "a workgroup's candidates of a bin are two words");
    __shared__ uint32_t band_lds[kBandBins][kBandSlots];
    __shared__ uint32_t band_count[kBandBins + 1];  // per bin; [kBandBins]: tokens above the band
    // Over all workgroups: [0..3] the counts of two bins each, [4] the tokens above the band, [8] how many
    // bins from the lowest on hold one without room for its count, [9] a bin's candidates do not fit.
    __shared__ uint32_t band_sum[kBandBins + 2];
    // Per bin of the wide band, and above them all; over all workgroups two bins each, the tokens above, and how many
    // bins from the lowest on hold one without room for its count.  (Of 40 to 64 heads on 8 behind the histogram, where their query
    // operands have left room: with 208 bytes more, and the stage that a workgroup with a CU to itself may ask for, their kernels
    // were past the 160 KB of a CU, and those shapes had no fused selection.  In the place of the histogram's first bins for all shapes: one request of
    // 32K 501 -> 505 us, a chunk at 128K 199.0 -> 200.)
    constexpr bool kWideInRoom = LATE && LH >= kTopkBins + kWideBins + 1 + 4 * kWideWords + 2;
    __shared__ uint32_t wide_count_own[LATE && !kWideInRoom ? kWideBins + 1 : 1], wide_sum_own[LATE && !kWideInRoom ? 4 * kWideWords + 2 : 1];
    uint32_t *const wide_count = kWideInRoom ? lh + kTopkBins : wide_count_own,
             *const wide_sum = kWideInRoom ? lh + kTopkBins + kWideBins + 1 : wide_sum_own;
    static_assert(kLateSlots <= kBandBins * kBandSlots, "the late candidates take the place of the band's");
    for (int i = tid; i < kTopkBins; i += 256) lh[i] = 0u;
    if (tid < 16) scratch[tid] = 0u;
    if (tid < kBandBins * kBandSlots) band_lds[tid / kBandSlots][tid % kBandSlots] = 0u;
    if (tid <= kBandBins) band_count[tid] = 0u;
    if (tid < kBandBins + 2) band_sum[tid] = 0u;
    if (LATE && tid <= kWideBins) wide_count[tid] = 0u;
    if (LATE && tid < 4 * kWideWords + 2) wide_sum[tid] = 0u;
    TS_MARK(1);
    __syncthreads();  // scores, own maxima and the cleared histogram are in LDS for all
    TS_MARK(2);
    // The votes-only form merges first: its workgroups hold up to twice the tokens, all of them
    // stream to the phase's end, and the next phase waits for them (4 x 256K: 420 us, 425 with
    // the exponentials first).
    if constexpr (PACKED) {
      merge_request_stats<PACKED>(a, lp, team, Lengths{own_len, own_slot, taken}, plans, lane, wave);
      TS_MARK(3);
    } else {
      fixed_parts(a, Lengths{own_len, own_slot, taken}, plans);
    }
    uint32_t ahead[kAheadLoads];
#pragma unroll
    for (int i = 0; i < kAheadLoads; ++i) ahead[i] = 0u;
    if constexpr (PACKED) {
      if (wave != 0) touch_successor_keys<HKV>(a, wave, lane, ahead);  // (wavefront 0 polls)
    }
    // While the statistics are on their way: the exponentials, relative to this
    // workgroup's own maxima; exp(s - max) / sum = exp(s - own max) * exp(own max - max) / sum.
    // (only k: whatever the length)
    const uint32_t k = (uint32_t)geometry_of_length(0, a.k_per_req, b, a.n_init, a.n_local, a.top_k, a.max_seq_len).k;
    const int count = min(lp.tokens_per_block, n - block_lo);
    uint32_t* ctr = a.counters + (size_t)b * kSelCounterWords;
    auto column = [&](int i) -> float* { return stage + (i >> 4) * tile_stride + (i & 15); };
    auto key_of = [&](int i) -> uint32_t { return vote_key(*column(i)); };
    for (int i = tid; i < count; i += 256) {
      float* sc = column(i);
#pragma unroll
      for (int s0 = 0; s0 < HKV * G; s0 += 8) {  // H = HKV * G head slots, 8 LDS reads in flight
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = s0 + j < HKV * G ? sc[(s0 + j) * 16] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (s0 + j < HKV * G) sc[(s0 + j) * 16] = __expf(x[j] - local_max[s0 + j]);
      }
    }
    // (after the exponentials: the workgroups that merge are among those that wait for the last one's)
    if constexpr (!PACKED) {
      merge_request_stats<PACKED>(a, lp, team, Lengths{own_len, own_slot, taken}, plans, lane, wave);
      TS_MARK(3);
    }
    if (tid < H) {  // H <= kMaxHeads < 256
      const int h = head_of<HKV, G>(tid / G, tid % G, a.head_map);
      const uint64_t* rep = (const uint64_t*)(a.stats + (size_t)(team.index % kSyncSlots) * a.stats_stride) +
                            (size_t)b * H + h;
      const uint64_t st = poll_nonzero<kStatsPollSleep>(rep, lp.sync, a.spin_ticks);
      const float mx = __uint_as_float((uint32_t)st), sum = __uint_as_float((uint32_t)(st >> 32));
      s_rz[tid] = st ? __expf(local_max[tid] - mx) / sum : 0.f;  // 0: the wait gave up
    }
    __syncthreads();
    TS_MARK(4);

    // Votes of this workgroup's tokens: fp32 sum over the head slots in slot order.
    // The vote replaces the first score of its token in LDS (only the thread that
    // owns a token reads its column).
    for (int i = tid; i < count; i += 256) {
      float* sc = column(i);
      float c = 0.f;
#pragma unroll
      for (int s0 = 0; s0 < HKV * G; s0 += 8) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = s0 + j < HKV * G ? sc[(s0 + j) * 16] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (s0 + j < HKV * G) c += x[j] * s_rz[s0 + j];
      }
      if (a.votes && a.pool_kernel <= 0) a.votes[(size_t)b * a.vote_stride + block_lo + i] = c;
      sc[0] = c;
    }
    TS_MARK(5);
    uint32_t round = 0;  // rendezvous passed so far
    if (a.pool_kernel > 0) {
      // Max-pool smoothing of the votes (tr.py:366-369): stride 1, padding (kernel-1)/2
      // with -inf, an even kernel makes the result one shorter.  The workgroups
      // exchange their votes through memory (one more rendezvous), gather the
      // kernel-1 neighbours on either side of their range into LDS (the histogram
      // array is still unused) and replace each vote by the maximum of its window.
      float* pv = a.pool_votes + (size_t)b * a.pool_stride;
      float* window = (float*)lh;  // [pad | own votes | kernel-1-pad]
      const int pad = (a.pool_kernel - 1) / 2;
      const int halo = a.pool_kernel - 1;
      for (int i = tid; i < count; i += 256) {
        const float c = *column(i);
        __hip_atomic_store((uint32_t*)&pv[block_lo + i], __float_as_uint(c), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        window[pad + i] = c;
      }
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
      for (int hx = tid; hx < halo; hx += 256) {
        const int t = hx < pad ? block_lo - pad + hx : block_lo + count + (hx - pad);
        const int at = hx < pad ? hx : count + hx;
        window[at] = (t >= 0 && t < n) ? __uint_as_float(load_coherent((const uint32_t*)&pv[t]))
                                       : -INFINITY;
      }
      __syncthreads();
      const int n_pooled = n + 2 * pad - a.pool_kernel + 1;
      for (int i = tid; i < count; i += 256) {
        float m = -INFINITY;  // past the pooled length: never selected (k < n)
        if (block_lo + i < n_pooled) {
          for (int w = 0; w < a.pool_kernel; ++w) m = fmaxf(m, window[i + w]);
          if (a.votes) a.votes[(size_t)b * a.vote_stride + block_lo + i] = m;
        }
        *column(i) = m;
      }
      __syncthreads();
      for (int i = tid; i < count + halo; i += 256) lh[i] = 0u;
      __syncthreads();
    }
    if (PACKED) {
      // The launch ends here: the votes are in memory, and their first histogram level
      // goes to the top-k workspace, where the kernels after this one pick it up.
      if (a.hist_ws) {
        for (int i = tid; i < count; i += 256) atomicAdd(&lh[key_bin0(key_of(i))], 1u);
        __syncthreads();
        uint32_t* hist0 = topk_ws(a.hist_ws, a.hist_ws_stride, b) + kTopkHist0;
        for (int i = tid; i < kTopkBins; i += 256)
          if (lh[i]) atomicAdd(&hist0[i], lh[i]);
      }
      if (chunk == 0 && tid == 0 && load_coherent(&lp.sync[0]) != 0u) {
        __hip_atomic_store(a.fault_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.fault_out)
          __hip_atomic_store(a.fault_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
#pragma unroll
      for (int i = 0; i < kAheadLoads; ++i) asm volatile("" ::"v"(ahead[i]));
      return;
    }
    // The physical slots of this thread's tokens, for the emission at the very end: the
    // table entries are asked for here, several rendezvous ahead, instead of in the
    // kernel's last microsecond with the stores waiting behind them.
    constexpr int kEmitAhead = 5;  // x 256 tokens: the largest workgroup (1056 tokens)
    uint32_t slot_ahead[kEmitAhead];
#pragma unroll
    for (int it = 0; it < kEmitAhead; ++it) {
      slot_ahead[it] = 0u;
      if (it * 256 >= count) continue;
      const int i = min(it * 256 + tid, count - 1);
      slot_ahead[it] = lookup_slot(tab, a.n_init + block_lo + i, a.page_size, a.page_shift, a.pool_rows);
    }
    // With a hint, what the band around it needs: the candidates of each band bin go to slots
    // in LDS (published below), and the tokens above the band are counted.  Without one, the
    // local histogram: one LDS atomic per candidate (lanes that hit the same bin are
    // performed one after the other, which for 256 candidates is a few hundred cycles).
    const int hint_bin = hint_word - 1;
    const bool banded = hint_bin >= 0 && hint_bin < kTopkBins && lp.tokens_per_block <= kBandMaxTokens &&
                        req_chunks <= kSelMaxChunks / 2;
    const int band_lo = hint_bin - kBandBelow;  // (bins outside [0, kTopkBins) hold nothing)
    if (banded) {
      uint32_t over_band = 0;  // this thread's tokens above the band
      for (int i = tid; i < count; i += 256) {
        const uint32_t key = key_of(i);
        const int d = (int)key_bin0(key) - band_lo;
        if (d >= 0 && d < kBandBins) {
          const uint32_t at = atomicAdd(&band_count[d], 1u);
          if (at < (uint32_t)kBandSlots) band_lds[d][at] = 0x80000000u | ((key & 0x1fffffu) << 10) | (uint32_t)i;
        }
        over_band += d >= kBandBins ? 1u : 0u;
      }
      over_band = wave_total(over_band);
      if (lane == 0 && over_band) atomicAdd(&band_count[kBandBins], over_band);
    }
    uint32_t top = 0;  // this thread's highest bin
    auto count_bins = [&]() {
      for (int i = tid; i < count; i += 256) {
        const uint32_t bin = key_bin0(key_of(i));
        atomicAdd(&lh[bin], 1u);
        top = max(top, bin);
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, off));
      if (lane == 0) atomicMax(&scratch[8], top);
      __syncthreads();
    };
    if (!banded) count_bins();
    else __syncthreads();

    TS_MARK(6);
    // First level: top 11 key bits.  The workgroups add their local histograms to one
    // of the copies and note the highest occupied bin; afterwards each searches
    // downwards from that bin, 256 bins at a time (one is enough unless the votes
    // span more than 64 binades).  With a hint the band's counts go out instead, and the
    // histogram only follows when the threshold turns out to lie outside the band.
    uint32_t* hist0 = ctr + kSelHist0 + (chunk % kSelHistCopies) * kTopkBins;
    auto publish_histogram = [&]() {
      // Two adjacent bins per 64-bit add (their counts cannot carry into each other):
      // half as many read-modify-writes on the few hot lines.
      uint64_t done = 0;  // old values: waited for once, after all are on their way
#pragma unroll
      for (int j = 0; j < kTopkBins / 512; ++j) {
        const int i = 2 * (tid + 256 * j);
        const uint64_t pair = (uint64_t)lh[i] | ((uint64_t)lh[i + 1] << 32);
        if (pair)
          done += __hip_atomic_fetch_add((uint64_t*)&hist0[i], pair, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
      }
      if (tid == 0)
        done += fetch_max_coherent(&ctr[kSelMaxBin + (chunk % kSelHistCopies) * 32], scratch[8]);
      await(done);
    };
    uint64_t* const band = a.band + (size_t)b * kBandRows * kSelMaxChunks;  // [kBandRows][workgroup]
    if (!banded) {
      publish_histogram();
    } else if (wave == 0) {
      // The candidates of bin l by lane l (none when they do not fit, since the bin is then not
      // ranked from the band), then the counts.  Nothing waits for these stores: no word of them
      // is zero, and whoever needs one asks until it has come.
      const uint32_t here = lane < kBandBins ? band_count[lane] : 0u;
      if (here >= 1 && here <= (uint32_t)kBandSlots) {
        store_coherent(&band[(size_t)band_piece_row(lane, 0) * kSelMaxChunks + chunk],
                       (uint64_t)band_lds[lane][0] | ((uint64_t)band_lds[lane][1] << 32));
        if (here >= 3)
          store_coherent(&band[(size_t)band_piece_row(lane, 1) * kSelMaxChunks + chunk],
                         (uint64_t)band_lds[lane][2] | ((uint64_t)band_lds[lane][3] << 32));
      }
      const bool full = __any(here >= kBandCountMost);
      uint32_t low = 0, high = 0;  // four counts each
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        low |= min(band_count[d], kBandCountMost) << (d * kBandCountBits);
        high |= min(band_count[4 + d], kBandCountMost) << (d * kBandCountBits);
      }
      if (lane < kBandReplicas)
        store_coherent(&band[(size_t)lane * kSelMaxChunks + chunk],
                       (uint64_t)low | ((uint64_t)high << (4 * kBandCountBits)) |
                           ((uint64_t)band_count[kBandBins] << kBandOverAt) |
                           (full ? kBandFull : 0ull) | kBandSent);
    }
    // (Ahead of the waits that follow: in memory before this workgroup decides that it stands.)
    if (chunk == 0 && tid == 0) store_coherent((uint32_t*)&a.sel_len[b], (uint32_t)(a.n_init + (int)k + a.n_local));
    TS_MARK(7);
    if (!banded) grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
    TS_MARK(8);
    uint32_t t0 = 0, above0 = 0, in_bin0 = 0;
    // With a hint: every workgroup's counts and its candidates of the bin the hint names, a thread
    // per workgroup, asked for until they have come (the bin is a guess: the threshold bin is
    // known after the search, and another bin of the band costs one more round of loads).
    constexpr int kBandLoads = kSelMaxChunks / 2 / 256;  // (512 chunks at most)
    uint64_t band_counts[kBandLoads];
    uint64_t band_piece[kBandLoads][2];
    auto band_here = [&](int r, int d) {  // candidates in bin d
      return (uint32_t)(band_counts[r] >> (d * kBandCountBits)) & kBandCountMask;
    };
    // Asks with `ask` until that says that all has come; bounded, as every wait is.  On giving up
    // (or when another wait did) the request is lost: what this workgroup is going to write is
    // wrong, and if the length stands already it is taken back here.
    auto until_come = [&](auto&& ask) {
      const uint64_t t_start = wall_clock64();
      for (uint32_t polls = 1; !__all(ask()); ++polls) {
        if ((polls & 15u) == 0 &&
            (load_coherent(&lp.sync[0]) != 0u || wall_clock64() - t_start > a.spin_ticks)) {
          raise_fault(lp.sync);
          if (lane == 0 && (fetch_or_coherent(&ctr[kSelVerdict], kSelLost) & kSelDecided) != 0u) {
            store_coherent((uint32_t*)&a.sel_len[b], 0xffffffffu);
            if (a.fault_out)
              __hip_atomic_store(a.fault_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          }
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    };
    auto load_counts = [&]() {
      const uint64_t* from = &band[(size_t)(team.index % kBandReplicas) * kSelMaxChunks];
      until_come([&]() {
        // (An absent member, in tests, is missed by all but the request's first workgroup: the harder
        // order, in which the length stands before a wait gives up.)
        bool come = a.absent == 0u || chunk == 0;
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) {
          const int at = tid + 256 * r;
          band_counts[r] = at < req_chunks ? load_coherent(&from[at]) : 0ull;
          come = come && (at >= req_chunks || band_counts[r] != 0ull);
        }
        return come;
      });
    };
    auto load_pieces = [&](int d) {
      until_come([&]() {
        bool come = true;
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) {
          const int at = tid + 256 * r;
          const uint32_t here = band_here(r, d);
          const bool fits = here >= 1 && here <= (uint32_t)kBandSlots;
          band_piece[r][0] = fits ? load_coherent(&band[(size_t)band_piece_row(d, 0) * kSelMaxChunks + at]) : 0ull;
          band_piece[r][1] = fits && here >= 3 ? load_coherent(&band[(size_t)band_piece_row(d, 1) * kSelMaxChunks + at]) : 0ull;
          come = come && (!fits || (band_piece[r][0] != 0ull && (here < 3 || band_piece[r][1] != 0ull)));
        }
        return come;
      });
    };
    bool found = false;     // the threshold bin is known
    bool from_band = false; // and its candidates are in `entries`
    // Where it is known and they are not: what each workgroup holds in it, and above it.
    uint32_t late_few[kBandLoads], late_above[kBandLoads];
    int late_from = 0, late_skip0 = kBandBins, late_skip1 = kBandBins;  // the bins whose words are free: from the first, less two
    // The candidates that the last step ranks, in any order (in the place of the histogram's
    // last bins: with a hint it has not been counted yet, else it has been searched by then).
    uint2* const entries = (uint2*)(lh + kTopkBins - 2 * kSelListCap);
    // Appends the band's candidates of the loaded bin and counts the tokens above it in the
    // workgroups before this one; a workgroup with more candidates than slots is noted.
    auto gather_band = [&](uint32_t bin) {
      const int bin_at = (int)bin - band_lo;
      // What the workgroups before this one hold above the bin: their fields of six bits, added
      // in pairs, then the pairs.
      uint64_t lower = 0;
#pragma unroll
      for (int r = 0; r < kBandLoads; ++r) lower += tid + 256 * r < chunk ? band_counts[r] : 0ull;
      uint32_t before = (uint32_t)(lower >> kBandOverAt) & kBandOverMask;
      lower = (lower & kBandFields) >> (kBandCountBits * bin_at);
      lower = ((lower >> 6) & kBandEven) + ((lower >> 12) & kBandEven);
      lower += lower >> 24;
      before += ((uint32_t)lower & 0xfffu) + ((uint32_t)(lower >> 12) & 0xfffu);
#pragma unroll
      for (int r = 0; r < kBandLoads; ++r) {
        const uint32_t packed[4] = {(uint32_t)band_piece[r][0], (uint32_t)(band_piece[r][0] >> 32),
                                    (uint32_t)band_piece[r][1], (uint32_t)(band_piece[r][1] >> 32)};
        const uint32_t from = (uint32_t)(tid + 256 * r) * (uint32_t)lp.tokens_per_block;  // that workgroup's first token
        uint32_t have = band_here(r, bin_at);  // (zero where the load was skipped)
        if (have > (uint32_t)kBandSlots) {
          band_sum[kBandBins + 1] = 1u;
          have = 0u;
        }
        // Places for the wavefront's candidates with one addition (each lane adding its own
        // count to the one word would be performed lane after lane).
        const uint64_t b0 = __ballot(have & 1u), b1 = __ballot(have & 2u), b2 = __ballot(have & 4u);
        if ((b0 | b1 | b2) == 0ull) continue;
        const uint64_t low = (1ull << lane) - 1ull;
        uint32_t at = 0;
        if (lane == 0)
          at = atomicAdd(&scratch[15], (uint32_t)(__popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2)));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) +
             (uint32_t)(__popcll(b0 & low) + 2 * __popcll(b1 & low) + 4 * __popcll(b2 & low));
#pragma unroll
        for (uint32_t h2 = 0; h2 < 4; ++h2)
          if (h2 < have && at + h2 < (uint32_t)kSelListCap)
            entries[at + h2] = make_uint2((bin << 21) | ((packed[h2] >> 10) & 0x1fffffu), from + (packed[h2] & 1023u));
      }
      before = wave_total(before);
      if (lane == 0 && before) atomicAdd(&scratch[10], before);
    };
    if (banded) {
      load_counts();
      TS_MARK(16);
      load_pieces(kBandBelow);
      if (chunk == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the length's store among others
      TS_MARK(17);
      // The counts of all workgroups: two fields to a register, 16 lanes each, then in LDS; and the
      // highest bin that some workgroup's field has no room for.
      {
        uint64_t both = 0;
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) {
          both += band_counts[r];
          if (__builtin_expect((band_counts[r] & kBandFull) != 0ull, 0)) {
            uint64_t ones = band_counts[r] & kBandFields;  // becomes: the lowest bit of a field of ones
            ones &= ones >> 1;
            ones &= (ones >> 2) & (ones >> 3);
            ones &= kBandLowest;
            if (ones) atomicMax(&band_sum[kBandBins], (63u - (uint32_t)__builtin_clzll(ones)) / kBandCountBits + 1u);
          }
        }
        uint32_t sums[kBandBins / 2 + 1];
#pragma unroll
        for (int j = 0; j < kBandBins / 2; ++j) {
          const uint32_t two = (uint32_t)(both >> (2 * j * kBandCountBits));
          sums[j] = (two & kBandCountMask) | ((two >> kBandCountBits & kBandCountMask) << 16);
        }
        sums[kBandBins / 2] = (uint32_t)(both >> kBandOverAt) & kBandOverMask;
#pragma unroll
        for (int j = 0; j <= kBandBins / 2; ++j) sums[j] = row16_total(sums[j]);
        if ((lane & 15) == 0) {
#pragma unroll
          for (int j = 0; j <= kBandBins / 2; ++j) atomicAdd(&band_sum[j], sums[j]);
        }
      }
      gather_band((uint32_t)hint_bin);
      __syncthreads();
      // Downwards from the bins above the band: the bin in which the count reaches k.
      uint32_t sums[kBandBins];
#pragma unroll
      for (int d = 0; d < kBandBins; ++d) sums[d] = band_sum[d / 2] >> (16 * (d & 1)) & 0xffffu;
      uint32_t run = band_sum[kBandBins / 2];
      int d0 = -1;
#pragma unroll
      for (int d = kBandBins - 1; d >= 0; --d) {
        const bool here = d0 < 0 && run < k && run + sums[d] >= k;
        if (here) {
          d0 = d;
          in_bin0 = sums[d];
        }
        if (d0 < 0) run += sums[d];
      }
      // (the sums above the highest bin without room are exact, and the threshold has to lie there)
      if (d0 >= (int)band_sum[kBandBins] && band_lo + d0 >= 0) {
        found = true;
        t0 = (uint32_t)(band_lo + d0);
        above0 = run;
        if (in_bin0 <= (uint32_t)kSelListCap) {
          if (d0 != kBandBelow) {  // another bin of the band: once more, with its words
            __syncthreads();
            if (tid == 0) scratch[10] = scratch[15] = band_sum[kBandBins + 1] = 0u;
            load_pieces(d0);
            __syncthreads();
            gather_band(t0);
            __syncthreads();
          }
          from_band = band_sum[kBandBins + 1] == 0u;
          // (every candidate of the bin is in a slot: the count is that of the histogram)
          if (from_band && scratch[15] != in_bin0 && tid == 0) raise_fault(lp.sync);
        }
        if (LATE && __builtin_expect(!from_band, 0)) {
          late_skip0 = min(d0, kBandBelow);
          late_skip1 = d0 == kBandBelow ? kBandBins : max(d0, kBandBelow);
#pragma unroll
          for (int r = 0; r < kBandLoads; ++r) {
            late_few[r] = band_here(r, d0);
            late_above[r] = (uint32_t)(band_counts[r] >> kBandOverAt) & kBandOverMask;
            for (int d = d0 + 1; d < kBandBins; ++d) late_above[r] += band_here(r, d);
          }
        }
      }
    }
    if (LATE && __builtin_expect(banded && !found && (band_sum[kBandBins / 2] >= k || band_sum[kBandBins] == 0u), 0)) {
      // Not in the band: the counts of the bins around it, of every workgroup, on the side where it is.  (The tokens of
      // the band are known where it has room for them all.)
      const bool higher = band_sum[kBandBins / 2] >= k;
      for (int i = tid; i < count; i += 256) {
        const int e = (int)key_bin0(key_of(i)) - (hint_bin - kWideBelow);
        if (e >= 0 && (higher ? e >= kWideBand + kBandBins : e < kWideBand)) atomicAdd(&wide_count[min(e, kWideBins)], 1u);
      }
      __syncthreads();
      if (wave == 0 && lane < kWideWords * kWideReplicas) {
        const int word = lane / kWideReplicas;
        uint64_t fields = kLateMark | (word == 2 ? (uint64_t)wide_count[kWideBins] << kWideOverAt : 0ull);
#pragma unroll
        for (int d = 0; d < 8; ++d) {
          const uint32_t n = wide_count[wide_bin(word, d)];
          fields |= (uint64_t)min(n, kBandCountMost) << wide_field_at(d);
          fields |= n >= kBandCountMost ? kWideFull : 0ull;
        }
        store_coherent(&band[(size_t)(kWideFirst + lane) * kSelMaxChunks + chunk], fields);
      }
      uint64_t sent[kBandLoads][kWideWords];
      const uint64_t* from = &band[(size_t)(kWideFirst + team.index % kWideReplicas) * kSelMaxChunks];
      until_come([&]() {
        bool come = true;
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r)
#pragma unroll
          for (int w = 0; w < kWideWords; ++w) {
            const int at = tid + 256 * r;
            sent[r][w] = at < req_chunks ? load_coherent(&from[(size_t)w * kWideReplicas * kSelMaxChunks + at]) : 0ull;
            come = come && (at >= req_chunks || late_come(sent[r][w]));
          }
        return come;
      });
      auto field = [&](int r, int w, int d) { return (uint32_t)(sent[r][w] >> wide_field_at(d)) & kBandCountMask; };
#pragma unroll
      for (int w = 0; w < kWideWords; ++w) {
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r)
          if (__builtin_expect((sent[r][w] & kWideFull) != 0ull, 0))
            for (int d = 0; d < 8; ++d)
              if (field(r, w, d) == kBandCountMost) atomicMax(&wide_sum[4 * kWideWords + 1], (uint32_t)wide_bin(w, d) + 1u);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t two = 0;
#pragma unroll
          for (int r = 0; r < kBandLoads; ++r) two += field(r, w, 2 * j) | field(r, w, 2 * j + 1) << 16;
          two = row16_total(two);
          if ((lane & 15) == 0) atomicAdd(&wide_sum[4 * w + j], two);
        }
      }
      {
        uint32_t over = 0;
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) over += (uint32_t)(sent[r][2] >> kWideOverAt) & kBandOverMask;
        over = row16_total(over);
        if ((lane & 15) == 0) atomicAdd(&wide_sum[4 * kWideWords], over);
      }
      __syncthreads();
      int e0 = -1;
      uint32_t run = higher ? wide_sum[4 * kWideWords] : band_sum[kBandBins / 2];
      uint32_t above[kBandLoads];
#pragma unroll
      for (int r = 0; r < kBandLoads; ++r) {
        above[r] = higher ? (uint32_t)(sent[r][2] >> kWideOverAt) & kBandOverMask
                          : (uint32_t)(band_counts[r] >> kBandOverAt) & kBandOverMask;
        late_few[r] = late_above[r] = 0u;
      }
      auto search = [&](int w, int d) {
        const uint32_t here = wide_sum[4 * w + d / 2] >> (16 * (d & 1)) & 0xffffu;
        if (e0 >= 0) return;
        const bool in = run < k && run + here >= k;
        if (in) {
          e0 = wide_bin(w, d);
          in_bin0 = here;
        } else {
          run += here;
        }
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) {
          const uint32_t own = field(r, w, d);
          if (in) {
            late_few[r] = own;
            late_above[r] = above[r];
          }
          above[r] += own;
        }
      };
      if (higher) {
#pragma unroll
        for (int d = 7; d >= 0; --d) search(2, d);
#pragma unroll
        for (int d = 7; d >= 4; --d) search(1, d);
      } else {
#pragma unroll
        for (int j = 0; j < kBandBins / 2; ++j) run += (band_sum[j] & 0xffffu) + (band_sum[j] >> 16);
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r)
#pragma unroll
          for (int d = 0; d < kBandBins; ++d) above[r] += band_here(r, d);
#pragma unroll
        for (int d = 3; d >= 0; --d) search(1, d);
#pragma unroll
        for (int d = 7; d >= 0; --d) search(0, d);
      }
      // (as in the band: above every bin without room)
      if (e0 >= (int)wide_sum[4 * kWideWords + 1] && hint_bin - kWideBelow + e0 >= 0) {
        found = true;
        t0 = (uint32_t)(hint_bin - kWideBelow + e0);
        above0 = run;
        late_from = kWideWords * kWideReplicas / 2;  // (the others are the words just read)
        late_skip0 = kBandBelow;
      }
    }
    if (banded && !found) {  // the hint was of no use: the histogram is needed after all
      __syncthreads();
      for (int i = tid; i < 2 * kSelListCap; i += 256) lh[kTopkBins - 2 * kSelListCap + i] = 0u;  // (the entries)
      __syncthreads();
      count_bins();
      publish_histogram();
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
    }
    if (!found) {
    // The search starts at the highest occupied bin of the request.  Together with the
    // words that hold it, the 128 bins below a guess (a little above this workgroup's
    // own highest bin) are fetched; the guess serves if no bin above it is occupied.
    constexpr int kWindow = 128;  // bins per step: two threads per bin, half the copies each
    const int guess = min((int)scratch[8] + 32, kTopkBins - 1);
    auto bins_below = [&](int top) {
      const int bin = top - (tid >> 1);
      const int first = (tid & 1) * (kSelHistCopies / 2);
      uint32_t part[kSelHistCopies / 2];
#pragma unroll
      for (int c = 0; c < kSelHistCopies / 2; ++c)
        part[c] = bin >= 0 ? load_coherent(&ctr[kSelHist0 + (first + c) * kTopkBins + bin]) : 0u;
      uint32_t sum = 0;
#pragma unroll
      for (int c = 0; c < kSelHistCopies / 2; ++c) sum += part[c];
      sum += (uint32_t)__shfl_xor((int)sum, 1);
      return (tid & 1) ? 0u : sum;  // the even thread of a pair stands for the bin
    };
    uint32_t mine = bins_below(guess);
    int top = guess;
    {
      uint32_t m = tid < kSelHistCopies ? load_coherent(&ctr[kSelMaxBin + tid * 32]) : 0u;
#pragma unroll
      for (int off = kSelHistCopies / 2; off >= 1; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off));
      __syncthreads();  // every thread has read this workgroup's own highest bin
      if (tid == 0) scratch[8] = m;
      __syncthreads();
      if ((int)scratch[8] > guess) {
        top = (int)scratch[8];
        mine = bins_below(top);
      }
    }
    for (;;) {
      uint32_t before, total, in_bin;
      const int who = block_threshold_scan(mine, k - above0, scratch, before, total, in_bin);
      if (who >= 0) {
        t0 = (uint32_t)(top - (who >> 1));
        above0 += before;
        in_bin0 = in_bin;
        break;
      }
      above0 += total;
      top -= kWindow;
      if (top < 0) break;
      mine = bins_below(top);
    }
    }

    TS_MARK(9);
    // What is left: `need` of the `in_bin` candidates whose key >> shift equals `prefix`.
    // As soon as they are few enough, they go to a short list that every workgroup
    // ranks on its own (the usual case: heavy-tailed votes leave a hundred candidates
    // in the threshold bin of the first level); otherwise the next histogram level.
    uint32_t need = k - above0, in_bin = in_bin0, prefix = t0;
    int shift = 21;
    if (in_bin > (uint32_t)kSelListCap) {
      // Second level: next 11 bits of the candidates inside bin t0.
      uint32_t done = 0;
      for (int base = 0; base < count; base += 256) {
        const uint32_t key = base + tid < count ? key_of(base + tid) : 0u;
        done += wave_histogram_add(ctr + kSelHist1 + (chunk % kSelHist1Copies) * kTopkBins,
                                   base + tid < count && key_bin0(key) == t0, key_bin1(key), lane);
      }
      await(done);
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
      {
        uint32_t h[kTopkBins / 256];
#pragma unroll
        for (int j = 0; j < kTopkBins / 256; ++j) {
          uint32_t part[kSelHist1Copies];
#pragma unroll
          for (int c = 0; c < kSelHist1Copies; ++c)
            part[c] = load_coherent(&ctr[kSelHist1 + c * kTopkBins + tid + 256 * j]);
          h[j] = 0u;
#pragma unroll
          for (int c = 0; c < kSelHist1Copies; ++c) h[j] += part[c];
        }
#pragma unroll
        for (int j = 0; j < kTopkBins / 256; ++j) lh[tid + 256 * j] = h[j];
      }
      __syncthreads();
      uint32_t t1, above1;
      find_threshold_bin<kTopkBins>(lh, need, scratch, t1, above1);
      need -= above1;
      in_bin = lh[t1];
      prefix = (t0 << 11) | t1;
      shift = 10;
      __syncthreads();
    }

    uint2* counts = a.block_counts + (size_t)b * kSelMaxChunks;
    const bool listed = in_bin <= (uint32_t)kSelListCap;
    uint32_t kth, need_eq = 0, pos_thr = 0, lower_taken = 0;
    // With a hint whose band holds the threshold bin and its candidates, everything the ranking
    // needs has come in the words of the band: no list round.  The test was the same for every
    // workgroup of the request (the same words, whole unless a wait gave up), so all take the same way.
    if (!from_band) {
      __syncthreads();
      if (tid < 8) scratch[8 + tid] = 0u;
      __syncthreads();
    }
    // The candidates of the threshold bin, wherever it was found, from word to word as those of the band: nobody meets.
    // (A hint that failed altogether leaves no words free, a bin that was cut further no counts, and more candidates than
    // kLateSlots of some workgroup no room.  Of pooled votes, whose peaks are as many equal keys as the window, a workgroup
    // has more than one look brings: window 15, one request of 100K tokens 64.1 us a layer met, 64.6 so.)  us a layer,
    // with two rounds, or one, met for in place of the wide band and this: eight requests of 3-16K 92.4 -> 88.0 (their
    // bins are crowded, and whoever fails keeps all waiting), one of 32K 32.6 -> 32.2 in the mean over hints that hold and
    // some that do not; four of 64K with a selection cache and a chunk at 128K, of which hardly one comes here, the same within
    // their runs' spread (612 and 606 us for eight steps, 198.1 and 198.2 for two layers).
    // (Both behind __builtin_expect: in line with the path of a hint that holds they cost that 0.3 us.)
    bool late = LATE && listed && !from_band && (banded ? found && shift == 21 : true) && lp.tokens_per_block <= kBandMaxTokens &&
                req_chunks <= kSelMaxChunks / 2;
    if (LATE && __builtin_expect(late, 0)) {
      const uint32_t slots = late_from ? (uint32_t)kLateSlotsWide : (uint32_t)kLateSlots;
      auto piece_row = [&](int p) {  // of a workgroup's p-th word of candidates
        int bin = late_from + (p >> 1);
        bin += bin >= late_skip0 ? 1 : 0;
        bin += bin >= late_skip1 ? 1 : 0;
        return (size_t)band_piece_row(bin, p & 1) * kSelMaxChunks;
      };
      uint32_t* const own = &band_lds[0][0];
      uint32_t above = 0;
      for (int base = 0; base < count; base += 256) {
        const int i = base + tid;
        const uint32_t key = i < count ? key_of(i) : 0u;
        const uint32_t top = key >> shift;
        above += (i < count && top > prefix) ? 1u : 0u;
        if (i < count && top == prefix) {
          const uint32_t at = atomicAdd(&scratch[9], 1u);
          if (at < slots) own[at] = ((key & 0x1fffffu) << 10) | (uint32_t)i;
        }
      }
      if (!banded) {
        above = wave_total(above);
        if (lane == 0 && above) atomicAdd(&scratch[8], above);
      }
      if (tid == 0) band_sum[kBandBins + 1] = 0u;
      __syncthreads();
      TS_MARK(10);
      if (wave == 0) {
        const uint32_t n = scratch[9];
        if (2u * (uint32_t)lane < n && n <= slots)
          store_coherent(&band[piece_row(lane) + chunk],
                         kLateMark | (uint64_t)own[2 * lane] | ((uint64_t)(2u * (uint32_t)lane + 1u < n ? own[2 * lane + 1] : 0u) << 32));
        if (!banded && lane < kBandReplicas)
          store_coherent(&band[(size_t)lane * kSelMaxChunks + chunk], kBandSent | ((uint64_t)n << kLateFewAt) | (uint64_t)scratch[8]);
      }
      if (!banded) {
        uint64_t sent[kBandLoads];
        const uint64_t* const words = &band[(size_t)(team.index % kBandReplicas) * kSelMaxChunks];
        until_come([&]() {
          bool come = true;
#pragma unroll
          for (int r = 0; r < kBandLoads; ++r) {
            const int at = tid + 256 * r;
            sent[r] = at < req_chunks ? load_coherent(&words[at]) : 0ull;
            come = come && (at >= req_chunks || sent[r] != 0ull);
          }
          return come;
        });
#pragma unroll
        for (int r = 0; r < kBandLoads; ++r) {
          late_few[r] = (uint32_t)(sent[r] >> kLateFewAt) & 0xffffu;
          late_above[r] = (uint32_t)sent[r] & 0xffffu;
        }
      }
      uint32_t before = 0;
#pragma unroll
      for (int r = 0; r < kBandLoads; ++r) {
        const uint32_t fits = late_few[r] <= slots ? late_few[r] : 0u;
        before += tid + 256 * r < chunk ? late_above[r] : 0u;
        if (late_few[r] != fits) band_sum[kBandBins + 1] = 1u;
        const uint32_t from = (uint32_t)(tid + 256 * r) * (uint32_t)lp.tokens_per_block;
        const uint64_t low = (1ull << lane) - 1ull;
        constexpr int kBatch = 4;  // words asked for together: eight candidates
        static_assert(kLateSlots % (2 * kBatch) == 0 && kLateSlotsWide % (2 * kBatch) == 0, "whole batches");
        for (uint32_t p0 = 0; 2 * p0 < slots && __any(fits > 2 * p0); p0 += kBatch) {
          uint64_t piece[kBatch];
          until_come([&]() {
            bool come = true;
#pragma unroll
            for (int p = 0; p < kBatch; ++p)
              piece[p] = fits > 2 * (p0 + p) ? load_coherent(&band[piece_row((int)p0 + p) + tid + 256 * r]) : kLateMark;
#pragma unroll
            for (int p = 0; p < kBatch; ++p) come = come && late_come(piece[p]);
            return come;
          });
          const uint32_t have = fits > 2 * p0 ? min(fits - 2 * p0, 2u * kBatch) : 0u;
          // (places for the wavefront's candidates with one addition)
          uint32_t total = 0, mine = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint64_t bits = __ballot(have >> i & 1u);
            total += (uint32_t)__popcll(bits) << i;
            mine += (uint32_t)__popcll(bits & low) << i;
          }
          uint32_t at = 0;
          if (lane == 0) at = atomicAdd(&scratch[15], total);
          at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + mine;
#pragma unroll
          for (uint32_t h = 0; h < 2 * kBatch; ++h) {
            const uint32_t packed = (uint32_t)(piece[h >> 1] >> (32 * (h & 1)));
            if (h < have && at + h < (uint32_t)kSelListCap)
              entries[at + h] = make_uint2((t0 << 21) | ((packed >> 10) & 0x1fffffu), from + (packed & 1023u));
          }
        }
      }
      before = wave_total(before);
      if (lane == 0 && before) atomicAdd(&scratch[10], before);
      __syncthreads();
      TS_MARK(11);
      late = band_sum[kBandBins + 1] == 0u;
      // (every candidate is there: the count is the one that was found)
      if (late && scratch[15] != in_bin && tid == 0) raise_fault(lp.sync);
      if (!late) {  // (everybody has seen the same words)
        __syncthreads();
        if (tid < 8) scratch[8 + tid] = 0u;
        __syncthreads();
      }
    }
    if (listed && !from_band && !late) {
      // Last round, short form: the candidates of the threshold bin are appended to
      // the list (in kSelListParts parts with a counter each, a wavefront reserving
      // its entries with one add), and every workgroup publishes how many of its
      // tokens lie above the bin.
      uint2* list = a.short_list + (size_t)b * kSelListParts * kSelListCap;
      const int part = chunk % kSelListParts;
      const uint64_t below_mask = (1ull << lane) - 1ull;
      uint32_t above = 0;
      for (int base = 0; base < count; base += 256) {
        const int i = base + tid;
        const uint32_t key = i < count ? key_of(i) : 0u;
        const uint32_t top = key >> shift;
        above += (i < count && top > prefix) ? 1u : 0u;
        const bool match = i < count && top == prefix;
        const uint64_t mm = __ballot(match);
        if (mm) {
          const int leader = __ffsll((unsigned long long)mm) - 1;
          uint32_t slot = 0;
          if (lane == leader)
            slot = fetch_add_coherent(&ctr[kSelListCount + part * 32], (uint32_t)__popcll(mm));
          slot = (uint32_t)__shfl((int)slot, leader) + (uint32_t)__popcll(mm & below_mask);
          if (match && slot < (uint32_t)kSelListCap)
            store_coherent(&list[part * kSelListCap + slot], key, (uint32_t)(block_lo + i));
        }
      }
      above = wave_total(above);
      if (lane == 0) atomicAdd(&scratch[8], above);
      __syncthreads();
      if (tid == 0) store_coherent(&counts[chunk], scratch[8], 0u);
      TS_MARK(10);
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
      TS_MARK(11);
      // The fill counters, the entries (a thread asks for two of a part, which covers all
      // unless a part holds more than a quarter of the list) and the counts of the
      // workgroups before this one are fetched together.
      constexpr uint32_t kPerPart = 2 * 256 / kSelListParts;
      const int my_part = tid % kSelListParts;
      const uint32_t first = (uint32_t)(tid / kSelListParts), second = first + 256u / kSelListParts;
      const uint32_t fill = load_coherent(&ctr[kSelListCount + my_part * 32]);
      const uint2 e0 = load_coherent(&list[my_part * kSelListCap + first]);
      const uint2 e1 = load_coherent(&list[my_part * kSelListCap + second]);
      uint32_t sure = 0;
      for (int j = tid; j < chunk; j += 256) sure += load_coherent(&counts[j]).x;
      auto append = [&](const uint2& e) {
        const uint32_t at = atomicAdd(&scratch[15], 1u);
        if (at < (uint32_t)kSelListCap) entries[at] = e;
      };
      if (first < fill) append(e0);
      if (second < fill) append(e1);
      for (uint32_t at = kPerPart + first; at < min(fill, (uint32_t)kSelListCap); at += 256u / kSelListParts)
        append(load_coherent(&list[my_part * kSelListCap + at]));
      sure = wave_total(sure);
      if (lane == 0 && sure) atomicAdd(&scratch[10], sure);
      __syncthreads();
    } else {
      TS_MARK(10);
    }
    if (listed) {
      // Every wavefront finds the last candidate taken on its own, in the order (key
      // descending, position ascending): it holds all of them, four to a lane, and the
      // need-th largest key is built bit by bit from how many keys reach it, until as many do
      // as are needed: some ten steps, and no barrier (narrowing the entries down by one
      // more digit in LDS took seven of them, and counting the larger keys for every entry
      // 2-6 us).  Equal keys, which a max-pool makes of every peak, are never told apart that
      // way: after twelve steps it is looked whether the keys that are left are all one (128K
      // tokens, windows of 15: 5.9 us with a step for every bit of key and position, 3.2 so; one
      // request of 100K tokens 71.5 -> 69.3 us a layer.  Votes without ties are through before).
      constexpr int kHeld = kSelListCap / 64;
      const uint32_t total = min(scratch[15], (uint32_t)kSelListCap);
      uint2 e[kHeld];
#pragma unroll
      for (int i = 0; i < kHeld; ++i)
        e[i] = (uint32_t)(64 * i + lane) < total ? entries[64 * i + lane] : make_uint2(0u, 0xffffffffu);
      auto count = [&](auto&& pred) {
        uint64_t lanes[kHeld];
#pragma unroll
        for (int i = 0; i < kHeld; ++i) lanes[i] = __ballot(pred(e[i]));
        // (all compared before the first is counted: in turn, through the one VCC, a step takes
        // half as long again)
        __builtin_amdgcn_sched_barrier(0);
        uint32_t sum = 0;
#pragma unroll
        for (int i = 0; i < kHeld; ++i) sum += (uint32_t)__popcll(lanes[i]);
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)sum);
      };
      // The first entry (of the lowest lane that has one) for which `pred` holds.
      auto first = [&](auto&& pred) {
        uint2 got = make_uint2(0u, 0u);
#pragma unroll
        for (int i = kHeld - 1; i >= 0; --i) {
          const uint64_t lanes = __ballot(pred(e[i]));
          if (lanes != 0ull) {
            const int at = __builtin_ctzll(lanes);
            got = make_uint2((uint32_t)__builtin_amdgcn_readlane((int)e[i].x, at),
                             (uint32_t)__builtin_amdgcn_readlane((int)e[i].y, at));
          }
        }
        return got;
      };
      // `reach` keys are at least `floor`, and fewer than are wanted are past its next 2 << bit.
      uint32_t floor = (uint32_t)__builtin_amdgcn_readfirstlane((int)(prefix << shift)), reach = total;
      const uint32_t wanted = (uint32_t)__builtin_amdgcn_readfirstlane((int)need);
      const int bits = __builtin_amdgcn_readfirstlane(shift);
      int bit = bits - 1;
      auto narrow = [&](int last) {
        for (; bit >= last && reach != wanted; --bit) {
          const uint32_t trial = floor | (1u << bit);
          const uint32_t with = count([&](const uint2& x) { return x.x >= trial; });
          if (with >= wanted) {
            floor = trial;
            reach = with;
          }
        }
      };
      narrow(max(bits - 12, 0));
      // (both ways for ties out of line: in the path of the calls without any, their instructions
      // cost 0.5 us, which is 1 % of three requests' prompts and 8 tokens)
      if (__builtin_expect(bit >= 0 && reach != wanted, 0)) {
        const uint32_t one = first([&](const uint2& x) { return x.x - floor < (2u << bit); }).x;
        if (count([&](const uint2& x) { return x.x == one; }) ==
            count([&](const uint2& x) { return x.x - floor < (2u << bit); })) {
          floor = one;
          bit = -1;
        }
        narrow(0);
      }
      kth = floor;
      pos_thr = 0xffffffffu;
      if (__builtin_expect(reach > wanted, 0)) {
        // More ties at the k-th key than places: those at the lowest positions are taken.  The
        // largest position with which the ties up to it still fit, from the highest bit in which
        // the ties' positions differ (there are two at least) down.
        const uint32_t places = wanted - count([&](const uint2& x) { return x.x > kth; });
        const uint32_t any = first([&](const uint2& x) { return x.x == kth; }).y;
        uint32_t differ = 0u;
#pragma unroll
        for (int i = 0; i < kHeld; ++i) differ |= e[i].x == kth ? e[i].y ^ any : 0u;
        int bit = 31 - __builtin_clz(wave_or(differ) | 1u);
        pos_thr = any & ~((2u << bit) - 1u);
        for (; bit >= 0; --bit) {
          const uint32_t trial = pos_thr | (1u << bit);
          if (count([&](const uint2& x) { return x.x == kth && x.y < trial; }) < places) pos_thr = trial;
        }
      }
      lower_taken = count([&](const uint2& x) {
        return (x.x > kth || (x.x == kth && x.y <= pos_thr)) && x.y < (uint32_t)block_lo;
      });
      TS_MARK(12);
    } else {
      // Third level: last 10 bits of the candidates inside (t0, t1).
      const uint32_t t1 = prefix & 2047u;
      {
        uint32_t done = 0;
        for (int base = 0; base < count; base += 256) {
          const uint32_t key = base + tid < count ? key_of(base + tid) : 0u;
          done += wave_histogram_add(
              ctr + kSelHist2, base + tid < count && key_bin0(key) == t0 && key_bin1(key) == t1,
              key_bin2(key), lane);
        }
        await(done);
      }
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
      {
        uint32_t h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = load_coherent(&ctr[kSelHist2 + tid + 256 * j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) lh[tid + 256 * j] = h[j];
      }
      __syncthreads();
      uint32_t t2, above2;
      find_threshold_bin<1024>(lh, need, scratch, t2, above2);
      need_eq = need - above2;  // ties at the k-th key still to take
      kth = (t0 << 21) | (t1 << 10) | t2;

      // Count step: every workgroup publishes how many of its tokens lie above the k-th
      // key and how many tie with it; ties are taken lowest position first, so the
      // counts of the workgroups before this one fix where its output starts and
      // how many of its ties still fit.
      uint32_t sure = 0, tie = 0;
      for (int i = tid; i < count; i += 256) {
        const uint32_t key = key_of(i);
        sure += key > kth ? 1u : 0u;
        tie += key == kth ? 1u : 0u;
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        sure += __shfl_xor(sure, off);
        tie += __shfl_xor(tie, off);
      }
      if (lane == 0) {
        atomicAdd(&scratch[8], sure);
        atomicAdd(&scratch[9], tie);
      }
      __syncthreads();
      if (tid == 0) store_coherent(&counts[chunk], scratch[8], scratch[9]);
      grid_arrive(lp.sync, ++round, a.spin_ticks, team.size, team.index);
    }
    // The requests of a batch may need different numbers of rounds, and the rendezvous
    // spans them all: whoever is through counts itself in for the rounds it skipped.
    if (team.size != (uint32_t)req_chunks) {  // other requests select in this launch as well
      const uint32_t rounds = kSelectRounds + (a.pool_kernel > 0 ? 1u : 0u);
      grid_arrive_rest(lp.sync, round + 1, rounds, team.size, team.index);
      round = rounds;
    }
    if (!listed) {
      // Counts of the workgroups before this one.
      uint32_t sure = 0, tie = 0;
      for (int j = tid; j < chunk; j += 256) {
        const uint2 v = load_coherent(&counts[j]);
        sure += v.x;
        tie += v.y;
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        sure += __shfl_xor(sure, off);
        tie += __shfl_xor(tie, off);
      }
      if (lane == 0) {
        atomicAdd(&scratch[10], sure);
        atomicAdd(&scratch[11], tie);
      }
    }
    __syncthreads();
    TS_MARK(13);
    uint32_t tie_run = scratch[11];  // ties at lower positions
    // selected at lower positions
    uint32_t out_run = scratch[10] + (listed ? lower_taken : min(tie_run, need_eq));
    __syncthreads();

    // Emission in position order.
    const int32_t* tab_b = a.table + (int64_t)b * a.table_stride;
    int32_t* sel = a.sel + (int64_t)b * a.sel_stride;
    int32_t* sel_pos = a.sel_pos + (int64_t)b * a.sel_stride;
    int32_t* cache_out = a.topk_cache ? a.topk_cache + (int64_t)b * a.top_k : nullptr;
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll 1
    for (int base = 0, it = 0; base < count; base += 256, ++it) {
      const int i = base + tid;
      const uint32_t key = i < count ? key_of(i) : 0u;
      const bool tie = i < count && key == kth;
      // The per-wavefront counts of an iteration go to one of two sets of words in turn: a
      // set is written again two iterations later, after a barrier that every wavefront
      // reaches only once it has read the set, so no barrier closes an iteration.
      uint32_t* counts_lds = scratch + (it & 1) * 8;
      uint32_t tie_rank = 0, tie_total = 0;
      if (!listed) {  // (with the short list a tie is taken by its position: no ranks needed)
        const uint64_t tie_mask = __ballot(tie);
        if (lane == 0) counts_lds[wave] = (uint32_t)__popcll(tie_mask);
        __syncthreads();
        tie_rank = tie_run + (uint32_t)__popcll(tie_mask & below);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (w < wave) tie_rank += counts_lds[w];
          tie_total += counts_lds[w];
        }
      }
      // A tie is taken if it is among the first need_eq in position order; with the
      // short list that is: not beyond the position of the k-th entry.
      const bool tie_taken = listed ? (uint32_t)(block_lo + i) <= pos_thr : tie_rank < need_eq;
      const bool chosen = i < count && (key > kth || (tie && tie_taken));
      const uint64_t chosen_mask = __ballot(chosen);
      if (lane == 0) counts_lds[4 + wave] = (uint32_t)__popcll(chosen_mask);
      __syncthreads();
      uint32_t rank = out_run + (uint32_t)__popcll(chosen_mask & below);
      uint32_t chosen_total = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (w < wave) rank += counts_lds[4 + w];
        chosen_total += counts_lds[4 + w];
      }
      if (chosen && rank < k) {
        const int pos = a.n_init + block_lo + i;
        sel_pos[a.n_init + rank] = pos;
        uint32_t slot = slot_ahead[0];
#pragma unroll
        for (int x = 1; x < kEmitAhead; ++x) slot = it == x ? slot_ahead[x] : slot;
        if (it >= kEmitAhead) slot = lookup_slot(tab_b, pos, a.page_size, a.page_shift, a.pool_rows);
        sel[a.n_init + rank] = (int32_t)slot;
        if (cache_out) cache_out[rank] = pos;
      }
      tie_run += tie_total;
      out_run += chosen_total;
    }
    TS_MARK(14);
    // A grid-wide wait of this launch gave up (the workgroups were not all resident
    // within the bound): what was selected is not valid.  The first workgroup of every
    // selecting request says so in place of the length, and in the caller's word.  A wait before a
    // rendezvous, or before this workgroup's words of the band were sent, raised the fault word
    // ahead of those; one for the band itself answers for itself (kSelVerdict).
    if (chunk == 0 && tid == 0) {
      const uint32_t verdict = fetch_or_coherent(&ctr[kSelVerdict], kSelDecided);
      const bool gave_up = load_coherent(&lp.sync[0]) != 0u || (verdict & kSelLost) != 0u;
      if (gave_up) {
        store_coherent((uint32_t*)&a.sel_len[b], 0xffffffffu);
        if (a.fault_out)
          __hip_atomic_store(a.fault_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      } else if (a.hint) {
        a.hint[b] = (int)t0 + 1;  // where the next step's band is going to lie
      }
    }
  }
}

static_assert(std::is_same<decltype(&score_kernel<8, 4, false, kScoreFused>), void (*)(ScoreArgs)>::value,
              "late_args() reads ScoreArgs from the start of the arguments");

template <bool OUT_BF16, int MODE>
static int launch_score(int hkv, int group, const ScoreArgs& a, dim3 grid, hipStream_t stream) {
  const size_t lds =
      MODE == kScoreTiled ? (size_t)a.tokens_per_block * a.num_heads * sizeof(float) : 0;
#define TS_SCORE_CASE(HKV_, G_)                                                                  \
  if (hkv == HKV_ && group == G_) {                                                              \
    hipLaunchKernelGGL((score_kernel<HKV_, G_, OUT_BF16, MODE>), grid, dim3(256), lds, stream, a); \
    return check_launch("score_kernel");                                                         \
  }
#define TS_SCORE_ROW(HKV_) \
  TS_SCORE_CASE(HKV_, 1) TS_SCORE_CASE(HKV_, 2) TS_SCORE_CASE(HKV_, 3) TS_SCORE_CASE(HKV_, 4) \
      TS_SCORE_CASE(HKV_, 5) TS_SCORE_CASE(HKV_, 6) TS_SCORE_CASE(HKV_, 7) TS_SCORE_CASE(HKV_, 8)
  TS_SCORE_ROW(1)
  TS_SCORE_ROW(2)
  TS_SCORE_ROW(4)
  TS_SCORE_ROW(8)
#undef TS_SCORE_ROW
#undef TS_SCORE_CASE
  return fail(TS_ESHAPE, "unsupported head shape: num_kv_heads=%d group=%d", hkv, group);
}

// The fused kernel of a head shape (its packed votes-only form), or NULL.
static const void* fused_kernel_of(int hkv, int group, int mode) {
#define TS_SCORE_CASE(HKV_, G_)                                                        \
  if (hkv == HKV_ && group == G_)                                                      \
    return mode == kScorePacked  ? (const void*)&score_kernel<HKV_, G_, false, kScorePacked>  \
         : mode == kScoreMeeting ? (const void*)&score_kernel<HKV_, G_, false, kScoreMeeting> \
                                 : (const void*)&score_kernel<HKV_, G_, false, kScoreFused>;
#define TS_SCORE_ROW(HKV_) \
  TS_SCORE_CASE(HKV_, 1) TS_SCORE_CASE(HKV_, 2) TS_SCORE_CASE(HKV_, 3) TS_SCORE_CASE(HKV_, 4) \
      TS_SCORE_CASE(HKV_, 5) TS_SCORE_CASE(HKV_, 6) TS_SCORE_CASE(HKV_, 7) TS_SCORE_CASE(HKV_, 8)
  TS_SCORE_ROW(1)
  TS_SCORE_ROW(2)
  TS_SCORE_ROW(4)
  TS_SCORE_ROW(8)
#undef TS_SCORE_ROW
#undef TS_SCORE_CASE
  return nullptr;
}

static size_t fused_lds_bytes(int tokens_per_block, int num_heads) {
  return (size_t)(tokens_per_block / 16) * (16 * num_heads + 16) * sizeof(float);
}

// Dynamic LDS the fused form may use.  With the 10 KB of static arrays two workgroups
// of 68 KB fit the 160 KB of a CU; a workgroup that asks for more than half of a CU's LDS
// (up to 140 KB) has the CU to itself.  Which of the two a launch gets is decided by its
// planner (fused_tokens_per_block, plan_vote_launches).
constexpr size_t kFusedStageBytes = 68 * 1024;
constexpr size_t kFusedLargeStageBytes = 140 * 1024;
constexpr size_t kFusedLargeFloorBytes = 76 * 1024;  // more than half a CU's LDS: one workgroup per CU
static size_t fused_stage_bytes(bool large) { return large ? kFusedLargeStageBytes : kFusedStageBytes; }

// The one process-wide switch of the library (ts_set_fused_select).
static std::atomic<int> g_fused_select{1};

int set_fused_select(int enable) { return g_fused_select.exchange(enable ? 1 : 0); }

static thread_local bool g_separate_call = false;
bool fused_kernels_enabled() { return g_fused_select.load() != 0 && !g_separate_call; }
SeparateKernelsScope::SeparateKernelsScope(bool on) : was(g_separate_call) {
  if (on) g_separate_call = true;
}
SeparateKernelsScope::~SeparateKernelsScope() { g_separate_call = was; }

// Workgroups of a fused kernel that the current device keeps resident at once (0: the
// shape has no fused kernel, or the runtime refused); depends on the kernel only.
static int kernel_capacity(const void* fn, bool large) {
  if (!fn) return 0;
  struct Entry { const void* fn; int device; bool large; int capacity; };
  constexpr int kMemo = 24;  // four shapes
  static thread_local Entry memo[kMemo] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  int capacity = 0;
  for (const Entry& e : memo)
    if (e.fn == fn && e.device == device && e.large == large) capacity = e.capacity;
  if (capacity == 0) {
    int per_cu = 0, cus = 0;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)kFusedLargeStageBytes) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, fused_stage_bytes(large)) !=
            hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    capacity = per_cu * cus;
    if (capacity <= 0) return 0;
    static thread_local int next = 0;
    memo[next++ % kMemo] = Entry{fn, device, large, capacity};
  }
  return capacity;
}
// ... of the kernel that a call may turn out to launch: of a selection's two forms the one that fewer fit of.
static int fused_capacity(const ts_config* cfg, bool packed, bool large) {
  const int hkv = cfg->num_kv_heads, group = cfg->num_heads / cfg->num_kv_heads;
  if (packed) return kernel_capacity(fused_kernel_of(hkv, group, kScorePacked), large);
  return std::min(kernel_capacity(fused_kernel_of(hkv, group, kScoreFused), large),
                  kernel_capacity(fused_kernel_of(hkv, group, kScoreMeeting), large));
}

// With max-pooling a workgroup gathers its votes and kernel - 1 neighbours into the LDS
// array of the histogram (kTopkBins words): the most tokens a workgroup may take then.
static int pooling_tokens_cap(const ts_config* cfg) {
  if (cfg->pool_kernel <= 0) return 1 << 30;
  return (kTopkBins - (cfg->pool_kernel - 1)) / 64 * 64;
}

// Tokens per workgroup of ts_select for a batch, 0 when the shape is not served; *large:
// whether the workgroups have a CU to themselves; *most_blocks: the most workgroups per
// request of any plan this shape may get (what has to be cleared for it).
// One workgroup per CU wherever the batch fits that way with no more LDS than a small
// workgroup has (C2 64.2 -> 61.9 us; 1.7-2.9 us at every length from 8K on for one request,
// 1-2 us for 2 x 64K and 4 x 32K): below 256 workgroups the dispatcher otherwise doubles
// them up on some CUs while others idle, above that half as many workgroups stream as
// fast and hand over less.  Batches that need more LDS per CU than that run as well or
// better on two workgroups per CU (2 x 128K the same, 4 x 64K and 8 x 32K 1-2 us better),
// unless requests may be skipped (selection cache): the workgroups are dealt over the
// requests that select, a step rarely has all of them, and the large workgroups then
// hold fewer tokens than they could (C4: 89.0 -> 87.4 us per step).
int fused_tokens_per_block(const ts_config* cfg, int batch, int max_seq_len, bool ignore_switch,
                           bool* large_out, bool may_skip, int* most_blocks_out) {
  if (large_out) *large_out = false;
  if (most_blocks_out) *most_blocks_out = 0;
  // Max-pool windows beyond 256 would not fit the LDS the neighbours are gathered into.
  if ((!ignore_switch && !fused_kernels_enabled()) || cfg->num_heads > kMaxHeads || cfg->pool_kernel > 256)
    return 0;
  const int max_n = max_seq_len - cfg->n_init - cfg->n_local;
  if (max_n <= 0) return 0;
  auto plan = [&](bool large) {
    const int capacity = fused_capacity(cfg, false, large);
    if (capacity <= 0) return 0;
    int tpb = score_tokens_per_block((int64_t)batch * max_n, cfg->num_heads);
    while ((int64_t)ceil_div(max_n, tpb) * batch > capacity) tpb += 64;
    if (fused_lds_bytes(tpb, cfg->num_heads) > fused_stage_bytes(large) || tpb > pooling_tokens_cap(cfg))
      return 0;
    if (ceil_div(max_seq_len, tpb) > kSelMaxChunks) return 0;  // what the workspace is laid out for
    return tpb;
  };
  const int tpb_small = plan(false), tpb_large = plan(true);
  // (the workgroups of a launch are dealt over the requests that select: one request may
  // get them all)
  if (most_blocks_out)
    *most_blocks_out = std::min<int>(
        kSelMaxChunks, batch * std::max(tpb_small > 0 ? (int)ceil_div(max_n, tpb_small) : 0,
                                        tpb_large > 0 ? (int)ceil_div(max_n, tpb_large) : 0));
  const bool roomy = tpb_large > 0 && fused_lds_bytes(tpb_large, cfg->num_heads) <= kFusedStageBytes;
  if (roomy || tpb_small == 0 || (may_skip && batch >= 2 && tpb_large > 0)) {
    if (large_out) *large_out = tpb_large > 0;
    return tpb_large;
  }
  return tpb_small;
}

static SelectWorkspace plan_select_workspace(const ts_config* cfg, int batch, int max_seq_len, bool ignore_switch,
                                             bool may_skip) {
  SelectWorkspace w{};
  // The layout depends on the batch, the head count and (for the pooled votes) the
  // length, not on how the candidates are dealt out, and is the same whether or not
  // this shape is served: a workspace sized for the longest context serves every
  // shorter one.
  bool large = false;
  w.tokens_per_block =
      fused_tokens_per_block(cfg, batch, max_seq_len, ignore_switch, &large, may_skip, &w.clear_chunks);
  w.lds_bytes = w.tokens_per_block > 0
                    ? std::max(fused_lds_bytes(w.tokens_per_block, cfg->num_heads),
                               large ? kFusedLargeFloorBytes : (size_t)0)
                    : 0;
  const int max_n = std::max(max_seq_len - cfg->n_init - cfg->n_local, 0);
  w.blocks_per_req = w.tokens_per_block > 0 ? (int)ceil_div(max_n, w.tokens_per_block) : 0;
  const size_t B = (size_t)batch, H = (size_t)cfg->num_heads;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align_up(bytes, 256);
    return at;
  };
  w.partials = take(B * H * (size_t)kSelMaxChunks * 2 * sizeof(float) +
                    B * kBandRows * (size_t)kSelMaxChunks * sizeof(uint64_t));  // (rows of the same size)
  // The counters and, right behind them, the replicas of the statistics are cleared
  // together before every launch.
  w.counters = take(B * kSelCounterWords * 4);
  w.stats_stride = (int64_t)align_up(B * H * 2, 1024);
  w.stats = take((size_t)kSyncSlots * w.stats_stride * sizeof(float));
  w.block_counts = take(B * (size_t)kSelMaxChunks * sizeof(uint2));
  w.short_list = take(B * kSelListParts * kSelListCap * sizeof(uint2));
  w.pool_stride = (int64_t)align_up((size_t)std::max(max_n, 1), 64);
  w.pool_votes = take(cfg->pool_kernel > 0 ? B * (size_t)w.pool_stride * sizeof(float) : 0);
  w.sync = take(B * kSyncWords * 4);  // one rendezvous area per launch of a batch served in groups
  w.total = off;
  return w;
}

// A step asks for the same plan half a dozen times (the layer object for the layout, the driver for
// the pieces, the form and the launch), 0.25 us each, and so does every layer of a forward: a thread
// keeps the last few, by everything that they follow from.  Lengths without a candidate are
// planned anew: that costs less than the look (a decode call of 2003 tokens 26.4 -> 25.4 us; one of
// 300 tokens 0.3 us slower where it looked too).
SelectWorkspace select_workspace(const ts_config* cfg, int batch, int max_seq_len, bool ignore_switch,
                                 bool may_skip) {
  struct Key {
    int device, num_heads, num_kv_heads, n_init, n_local, pool_kernel, batch, max_seq_len, options;
    bool operator==(const Key& o) const { return memcmp(this, &o, sizeof(Key)) == 0; }
  };
  int device = 0;
  if (max_seq_len <= cfg->n_init + cfg->n_local || hipGetDevice(&device) != hipSuccess)
    return plan_select_workspace(cfg, batch, max_seq_len, ignore_switch, may_skip);
  const Key key{device, cfg->num_heads, cfg->num_kv_heads, cfg->n_init, cfg->n_local, cfg->pool_kernel, batch,
                max_seq_len, (ignore_switch ? 1 : 0) | (may_skip ? 2 : 0) | (fused_kernels_enabled() ? 4 : 0)};
  struct Entry {
    Key key;
    SelectWorkspace w;
  };
  constexpr int kKept = 4;
  static thread_local Entry memo[kKept] = {};
  static thread_local int kept = 0, next = 0;
  for (int i = 0; i < kept; ++i)
    if (memo[i].key == key) return memo[i].w;
  const SelectWorkspace w = plan_select_workspace(cfg, batch, max_seq_len, ignore_switch, may_skip);
  if (fused_capacity(cfg, false, false) > 0) {  // (a device that did not answer is asked again)
    memo[next] = Entry{key, w};
    next = (next + 1) % kKept;
    kept = std::min(kept + 1, kKept);
  }
  return w;
}

// One phase of the votes-only form: requests [first, first + requests), `workgroups` in
// all, `table_chunks` an upper bound of the chunks of any of its requests.
struct VoteLaunch {
  int first, requests, tokens_per_block, workgroups, table_chunks;
};
// The phases of a batch, up to kMaxPhases of them to a launch.
struct VotePlan {
  std::vector<VoteLaunch> parts;
  int resident = 0;  // workgroups of the kernel that the device holds at once
};
bool plan_vote_launches(const ts_config* cfg, const ts_batch* bt, VotePlan* plan);

// The per-workgroup statistics are their own flags (a sum of exponentials is never
// zero): the chunks a launch may fill have to be zero before it, `chunks` of every
// (request, head) row, and of every row of the bands behind them.
static ZeroRegion partials_zero_region(const SelectWorkspace& w, void* workspace, int batch, int rows,
                                       int chunks) {
  ZeroRegion z;
  z.base = (uint32_t*)((char*)workspace + w.partials);
  z.stride = (int64_t)kSelMaxChunks * 2;
  z.words = std::min(chunks, kSelMaxChunks) * 2;
  z.count = batch * rows;
  return z;
}
static ZeroRegion stats_zero_region(const SelectWorkspace& w, void* workspace, int batch, int heads) {
  ZeroRegion z;  // the live words of the 64 replicas
  z.base = (uint32_t*)((char*)workspace + w.stats);
  z.stride = w.stats_stride;
  z.words = batch * heads * 2;
  z.count = kSyncSlots;
  return z;
}
static ZeroRegion sync_zero_region(const SelectWorkspace& w, void* workspace, int areas) {
  ZeroRegion z;
  z.base = (uint32_t*)((char*)workspace + w.sync);
  z.stride = kSyncSlotWords;
  z.words = kSyncLiveWords;
  z.count = (kSyncSlots + 1) * areas;
  return z;
}

void select_zero_regions(const ts_config* cfg, const SelectWorkspace& w, void* workspace, int batch,
                         ZeroSet* zero) {
  ZeroRegion counters;
  counters.base = (uint32_t*)((char*)workspace + w.counters);
  counters.words = batch * kSelCounterWords;
  counters.stride = counters.words;
  counters.count = 1;
  zero->add(counters);
  zero->add(stats_zero_region(w, workspace, batch, cfg->num_heads));
  zero->add(sync_zero_region(w, workspace, 1));
  zero->add(partials_zero_region(w, workspace, batch, cfg->num_heads + kBandRows, w.clear_chunks));
}

void score_votes_zero_regions(const ts_config* cfg, const ts_batch* bt, const SelectWorkspace& w,
                              void* workspace, ZeroSet* zero) {
  VotePlan plan;
  int chunks = 0;
  if (plan_vote_launches(cfg, bt, &plan))
    for (const VoteLaunch& v : plan.parts) chunks = std::max(chunks, v.table_chunks);
  zero->add(stats_zero_region(w, workspace, bt->batch, cfg->num_heads));
  zero->add(sync_zero_region(w, workspace, bt->batch));
  zero->add(partials_zero_region(w, workspace, bt->batch, cfg->num_heads, chunks));
}

bool vote_launches_planned(const ts_config* cfg, const ts_batch* bt) {
  if (bt->max_seq_len - cfg->n_init - cfg->n_local <= 0) return false;
  VotePlan plan;
  return plan_vote_launches(cfg, bt, &plan);
}
bool vote_launches_planned(const ts_config* cfg, int batch, int max_seq_len) {
  ts_batch bt{};
  bt.batch = batch;
  bt.max_seq_len = max_seq_len;
  return vote_launches_planned(cfg, &bt);
}

const uint32_t* score_votes_fault_word(const ts_config* cfg, int batch, int max_seq_len,
                                       const void* workspace) {
  return (const uint32_t*)((const char*)workspace + select_workspace(cfg, batch, max_seq_len, true).sync);
}

__global__ __launch_bounds__(256) void select_zero_kernel(ZeroSet zero) {
  clear_regions(zero, blockIdx.x * 4 + (threadIdx.x >> 6), gridDim.x * 4);
}
int launch_select_zero(const ZeroSet& zero, hipStream_t stream) {
  TS_REQUIRE(!zero.overflow, TS_EINVAL, "internal: more than %d regions to clear in one launch", kZeroRegions);
  const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(1024, ceil_div(zero.total(), 1024)));
  hipLaunchKernelGGL(select_zero_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, zero);
  return check_launch("select_zero_kernel");
}

static ScoreArgs selection_args(const ts_config* cfg, const ts_batch* bt, const void* qf,
                                const void* k_pool, int64_t pool_rows, const int32_t* skip,
                                float* partials, int tokens_per_block) {
  ScoreArgs a{};
  a.qf = (const uint16_t*)qf;
  a.k_pool = (const uint16_t*)k_pool;
  a.pool_rows = (uint32_t)pool_rows;
  a.seq_lens = bt->seq_lens;
  a.table = bt->table;
  a.table_stride = bt->table_stride;
  a.k_per_req = bt->k_per_req;
  a.skip = skip;
  a.n_init = cfg->n_init;
  a.n_local = cfg->n_local;
  a.top_k = cfg->top_k;
  a.max_seq_len = bt->max_seq_len;
  a.page_size = cfg->page_size;
  a.page_shift = page_shift_of(cfg->page_size);
  a.direct_n = -1;
  a.partials = partials;
  a.tokens_per_block = tokens_per_block;
  a.nchunks = (int)ceil_div(bt->max_seq_len, tokens_per_block);
  a.num_heads = cfg->num_heads;
  a.head_map = cfg->head_map;
  return a;
}

int launch_select(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
                  int64_t pool_rows, const int32_t* hit, const ts_selcache* cache, int32_t* sel,
                  int32_t* sel_pos, int64_t sel_stride, int32_t* sel_len, float* votes,
                  int64_t vote_stride, void* workspace, uint32_t* clear, int clear_per_req,
                  hipStream_t stream, uint64_t wait_ticks, uint32_t absent,
                  const UnrotatedQuery* unrotated, const StepStore* append, int4* notes, bool late) {
  // (requests may be skipped when the caller brings hit flags: the selection cache)
  const SelectWorkspace w = select_workspace(cfg, bt->batch, bt->max_seq_len, false, hit != nullptr);
  TS_REQUIRE(w.tokens_per_block > 0, TS_ESHAPE, "fused selection: unsupported shape");
  char* ws = (char*)workspace;
  ScoreArgs a = selection_args(cfg, bt, qf, k_pool, pool_rows, hit, (float*)(ws + w.partials),
                               w.tokens_per_block);
  a.nchunks = kSelMaxChunks;  // the row of a (request, head) pair in the statistics' table
  a.q_cos = a.q_sin = (const float*)(ws + w.counters);  // (readable, not used)
  if (unrotated) {
    a.q_raw = (const uint16_t*)unrotated->q;
    a.q_stride = unrotated->stride;
    a.q_cos = unrotated->cos;
    a.q_sin = unrotated->sin;
  }
  if (append) {
    TS_REQUIRE(bt->batch <= kCommitBatch && cfg->n_local >= 1 && notes, TS_EINVAL,
               "internal: this step's store does not ride in the selection");
    a.appends = 1;
    a.append = *append;
    a.notes = notes;
  }
  a.sync = (uint32_t*)(ws + w.sync);
  a.stats = (float*)(ws + w.stats);
  a.stats_stride = w.stats_stride;
  a.votes = votes;
  a.vote_stride = vote_stride;
  a.counters = (uint32_t*)(ws + w.counters);
  a.block_counts = (uint2*)(ws + w.block_counts);
  a.short_list = (uint2*)(ws + w.short_list);
  a.hint = bt->threshold_hint;
  a.band = (uint64_t*)(ws + w.partials) + (size_t)bt->batch * cfg->num_heads * kSelMaxChunks;
  a.sel = sel;
  a.sel_pos = sel_pos;
  a.sel_stride = sel_stride;
  a.sel_len = sel_len;
  a.topk_cache = cache ? cache->topk_cache : nullptr;
  a.cache_len = cache ? cache->cache_len : nullptr;
  a.clear = clear;
  a.clear_per_req = clear_per_req;
  a.spin_ticks = wait_ticks;
  a.absent = absent;
  a.fault_out = bt->fault;
  a.pool_kernel = cfg->pool_kernel;
  a.pool_votes = (float*)(ws + w.pool_votes);
  a.pool_stride = w.pool_stride;
  constexpr int kLatePool = 8;  // (wider windows fill fields and words too often: 9 of 0.9-7.5K, 58, 51.4 us a layer, and 49.1 met)
  const void* fn = fused_kernel_of(cfg->num_kv_heads, cfg->num_heads / cfg->num_kv_heads,
                                   late && cfg->pool_kernel <= kLatePool ? kScoreFused : kScoreMeeting);
  // One-dimensional: the kernel deals these workgroups over the requests that select.
  a.batch = bt->batch;
  const dim3 grid((unsigned)(w.blocks_per_req * bt->batch), 1u);
  void* params[] = {(void*)&a};
  // An ordinary launch: the grid was sized to be resident all at once, which holds
  // as long as the device runs nothing else beside this stream.  (The cooperative
  // launch API would guarantee it, at some 25 us of extra launch latency.)
  const hipError_t e =
      hipLaunchKernel(fn, grid, dim3(256), params, w.lds_bytes, stream);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(TS_EHIP, "fused selection launch: %s", hipGetErrorString(e));
  }
  return TS_OK;
}

// The votes-only form: consecutive requests are packed into phases by what they can
// hold -- the host's upper bounds of the lengths (ts_batch.host_seq_lens) where it has
// them, max_seq_len else -- as many as fit half the device (all of it, when a request
// needs more) with the most tokens per workgroup that the LDS takes.  One launch holds
// the workgroups of many phases, one after the other in a one-dimensional grid.  The
// device starts the workgroups of a grid in the order of their numbers as room becomes
// free (of those that go to one XCD, every eighth): with phases of half the device two
// of them are resident side by side, and when the workgroups of the earlier one leave,
// those of the next but one take their places.  A phase ends with the memory idle (the
// statistics on their way, scores turned into votes); the other phase streams
// meanwhile.  Two phases that start together would also wait together, so the second
// phase is given about half the candidates of a full one.  A workgroup without
// candidates (the bound was above the length) leaves at once and is not on the phase's
// team.  Nothing can wait forever: the workgroups of the earliest unfinished phase wait
// for each other only, and all of them have been started, since every workgroup started
// before them has left and fewer than fit are left to start.
// (A grid [chunks of the longest, requests] of a group of requests that must all be
// resident at once is not an alternative: its members have gaps between them and do not
// spread evenly over the XCDs; such launches were seen to wait for room that never came.)
bool plan_vote_launches(const ts_config* cfg, const ts_batch* bt, VotePlan* plan) {
  plan->parts.clear();
  if (!fused_kernels_enabled()) return false;
  if (cfg->num_heads > kMaxHeads || cfg->pool_kernel > 256) return false;
  const int fixed = cfg->n_init + cfg->n_local;
  auto bound = [&](int b) { return bt->host_seq_lens ? std::min(bt->host_seq_lens[b], bt->max_seq_len) : bt->max_seq_len; };
  auto candidates = [&](int b) { return std::max(bound(b) - fixed, 0); };
  int longest_n = 0;
  for (int b = 0; b < bt->batch; ++b) longest_n = std::max(longest_n, candidates(b));
  // The most tokens a workgroup of either size takes, and what is resident of them.
  auto size_up = [&](bool large, int* capacity_out) {
    *capacity_out = fused_capacity(cfg, /*packed=*/true, large);
    int most = 64;
    while (fused_lds_bytes(most + 64, cfg->num_heads) <= fused_stage_bytes(large) &&
           most + 64 <= pooling_tokens_cap(cfg))
      most += 64;
    return (*capacity_out > 0 && fused_lds_bytes(most, cfg->num_heads) <= fused_stage_bytes(large)) ? most : 0;
  };
  int capacity = 0;
  int tpb_max = size_up(false, &capacity);
  // The large workgroups when the longest request takes more than half of the device.
  if (tpb_max == 0 || ceil_div(longest_n, tpb_max) > capacity / 2) {
    int capacity_large = 0;
    const int most = size_up(true, &capacity_large);
    if (most > tpb_max) {
      tpb_max = most;
      capacity = capacity_large;
    }
  }
  if (tpb_max == 0) return false;
  plan->resident = capacity;
  // Phases of half the device when every request fits that.
  bool halves = bt->batch >= 2;
  for (int b = 0; b < bt->batch && halves; ++b)
    if (ceil_div(candidates(b), tpb_max) > capacity / 2) halves = false;
  const int room_full = halves ? capacity / 2 : capacity;
  for (int first = 0; first < bt->batch;) {
    // (the second phase: half a phase, see above)
    const bool shorter = halves && plan->parts.size() == 1;
    int64_t wgs = 0;
    int last = first, longest = 0;
    for (int pass = shorter ? 0 : 1; pass < 2 && last == first; ++pass) {
      const int64_t room = pass == 0 ? room_full / 2 : room_full;
      for (; last < bt->batch && last - first < kMaxPacked; ++last) {
        const int64_t more = ceil_div(candidates(last), tpb_max);
        if (wgs + more > room) break;
        wgs += more;
        longest = std::max(longest, bound(last));
      }
    }
    if (last == first) return false;  // a single request does not fit the device
    // Every workgroup takes as many tokens as the LDS holds (the statistics' table of a
    // request has room for kSelMaxChunks chunks): the fewer workgroups a phase has, the
    // sooner those of the next one find room, and the less each token carries of what a
    // workgroup does once (queries, statistics, the wait for them).
    const int tpb = tpb_max;
    if (ceil_div(longest, tpb) > kSelMaxChunks) return false;
    if (wgs > 0)  // (nothing to do for requests that are all sink and local window)
      plan->parts.push_back(VoteLaunch{first, last - first, tpb, (int)wgs, (int)ceil_div(longest, tpb)});
    first = last;
  }
  return true;
}

int launch_score_votes(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
                       int64_t pool_rows, const int32_t* skip, float* votes, int64_t vote_stride,
                       uint32_t* hist_ws, size_t hist_ws_stride, void* workspace, hipStream_t stream) {
  VotePlan plan;
  TS_REQUIRE(plan_vote_launches(cfg, bt, &plan), TS_ESHAPE,
             "fused scoring + vote: not even one request of %d tokens fits", bt->max_seq_len);
  // Offsets of the pieces: those of the whole batch's workspace, whatever the launches.
  const SelectWorkspace all = select_workspace(cfg, bt->batch, bt->max_seq_len, true);
  char* ws = (char*)workspace;
  const void* fn = fused_kernel_of(cfg->num_kv_heads, cfg->num_heads / cfg->num_kv_heads, kScorePacked);
  const int per_launch = kMaxPhases;
  for (size_t at = 0; at < plan.parts.size(); at += per_launch) {
    const VoteLaunch& v = plan.parts[at];
    ScoreArgs a = selection_args(cfg, bt, qf, k_pool, pool_rows, skip, (float*)(ws + all.partials),
                                 v.tokens_per_block);
    a.nchunks = kSelMaxChunks;
    a.sync = (uint32_t*)(ws + all.sync) + at * kSyncWords;  // one rendezvous area per part
    a.fault_word = (uint32_t*)(ws + all.sync);
    a.stats = (float*)(ws + all.stats);
    a.stats_stride = all.stats_stride;
    a.votes = votes;
    a.vote_stride = vote_stride;
    a.counters = (uint32_t*)(ws + all.counters);
    a.spin_ticks = select_wait_ticks(bt);
    a.absent = (uint32_t)std::max(bt->absent_workgroups, 0);
    a.fault_out = bt->fault;
    a.pool_kernel = cfg->pool_kernel;
    a.pool_votes = (float*)(ws + all.pool_votes);
    a.pool_stride = all.pool_stride;
    a.batch_offset = v.first;
    a.hist_ws = hist_ws;
    a.hist_ws_stride = hist_ws_stride;
    a.resident = plan.resident;
    int tpb_lds = v.tokens_per_block;
    dim3 grid;
    {
      const int phases = (int)std::min<size_t>(per_launch, plan.parts.size() - at);
      const int fixed = cfg->n_init + cfg->n_local;
      a.nphases = phases;
      int workgroups = 0;
      for (int p = 0; p < phases; ++p) {
        const VoteLaunch& part = plan.parts[at + p];
        VotePhase& ph = a.phases[p];
        ph.tokens_per_block = part.tokens_per_block;
        ph.first = part.first;
        ph.requests = part.requests;
        ph.first_workgroup = workgroups;
        ph.pack_first[0] = 0;
        for (int r = 0; r < part.requests; ++r) {
          const int len = bt->host_seq_lens ? std::min(bt->host_seq_lens[part.first + r], bt->max_seq_len)
                                            : bt->max_seq_len;
          const int cand = std::max(len - fixed, 0);
          ph.pack_first[r + 1] = ph.pack_first[r] + (int)ceil_div(cand, part.tokens_per_block);
        }
        workgroups += part.workgroups;
        tpb_lds = std::max(tpb_lds, part.tokens_per_block);
      }
      grid = dim3((unsigned)workgroups, 1u);
    }
    void* params[] = {(void*)&a};
    const hipError_t e = hipLaunchKernel(fn, grid, dim3(256), params,
                                         fused_lds_bytes(tpb_lds, cfg->num_heads), stream);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return fail(TS_EHIP, "fused scoring + vote launch: %s", hipGetErrorString(e));
    }
  }
  return TS_OK;
}

}  // namespace ts

using namespace ts;

extern "C" {

int ts_set_fused_select(int enable) { return set_fused_select(enable); }

size_t ts_score_partials_bytes(const ts_config* cfg, int32_t batch, int32_t max_seq_len) {
  if (validate_config(cfg) != TS_OK || batch < 1 || max_seq_len < 1) return 0;
  // A bound that never shrinks when max_seq_len grows, unlike the number of workgroups
  // itself (the candidates per workgroup move in steps of 64), so that a buffer sized
  // for the longest context serves every shorter one: 256 workgroups are aimed at (the
  // bound leaves room for twice that), more only once a workgroup holds as many candidates
  // as its LDS takes.
  const int64_t cap = std::max<int64_t>((16384 / cfg->num_heads) / 64 * 64, 64);
  const size_t nchunks = (size_t)std::max<int64_t>(520, ceil_div(max_seq_len, cap) + 8);
  return align_up((size_t)batch * cfg->num_heads * nchunks * 2 * sizeof(float), 256);
}

int ts_score(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
             int64_t pool_rows, const int32_t* skip, float* scores, int64_t score_stride,
             float* partials, size_t partials_bytes, ts_stream_t stream) {
  TS_TRY(validate_config(cfg));
  TS_TRY(validate_batch(cfg, bt));
  TS_REQUIRE(qf && k_pool && scores && partials, TS_EINVAL, "ts_score: NULL tensor argument");
  TS_REQUIRE_ALIGNED(qf, 16, "qf");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(scores, 16, "scores");
  TS_REQUIRE_ALIGNED(partials, 16, "partials");
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  const int max_n = bt->max_seq_len - cfg->n_init - cfg->n_local;
  TS_REQUIRE(score_stride >= max_n && score_stride >= 16 && score_stride % 16 == 0, TS_EWORKSPACE,
             "score_stride %lld must be a multiple of 16 and >= max candidates %d",
             (long long)score_stride, max_n);
  const size_t need = ts_score_partials_bytes(cfg, bt->batch, bt->max_seq_len);
  TS_REQUIRE(partials_bytes >= need, TS_EWORKSPACE, "ts_score: partials %zu bytes < required %zu",
             partials_bytes, need);
  if (max_n <= 0) return TS_OK;  // every request is dense

  ScoreArgs a = selection_args(
      cfg, bt, qf, k_pool, pool_rows, skip, partials,
      score_tokens_per_block((int64_t)bt->batch * bt->max_seq_len, cfg->num_heads));
  a.scores = scores;
  a.score_stride = score_stride;
  const dim3 grid((unsigned)ceil_div(max_n, a.tokens_per_block), (unsigned)bt->batch);
  return launch_score<false, kScoreTiled>(cfg->num_kv_heads, cfg->num_heads / cfg->num_kv_heads, a, grid,
                                   (hipStream_t)stream);
}

int ts_score_vote_supported(const ts_config* cfg, int32_t batch, int32_t max_seq_len) {
  if (validate_config(cfg) != TS_OK || batch < 1 || max_seq_len < 1) return 0;
  return vote_launches_planned(cfg, batch, max_seq_len) ? 1 : 0;
}

int ts_score_vote(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
                  int64_t pool_rows, const int32_t* skip, float* votes, int64_t vote_stride,
                  void* workspace, size_t workspace_bytes, ts_stream_t stream) {
  TS_TRY(validate_config(cfg));
  TS_TRY(validate_batch(cfg, bt));
  TS_REQUIRE(qf && k_pool && votes && workspace, TS_EINVAL, "ts_score_vote: NULL argument");
  TS_REQUIRE_ALIGNED(workspace, 256, "workspace");
  TS_REQUIRE_ALIGNED(qf, 16, "qf");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  TS_REQUIRE(ts_score_vote_supported(cfg, bt->batch, bt->max_seq_len), TS_ESHAPE,
             "ts_score_vote: not even one request of %d tokens fits the LDS of the device (or "
             "pool_kernel is above 256, or the fused kernels are switched off); use ts_score + ts_vote",
             bt->max_seq_len);
  const SelectWorkspace w = select_workspace(cfg, bt->batch, bt->max_seq_len, true);
  TS_REQUIRE(workspace_bytes >= w.total, TS_EWORKSPACE, "ts_score_vote: workspace %zu bytes < required %zu",
             workspace_bytes, w.total);
  const int max_n = bt->max_seq_len - cfg->n_init - cfg->n_local;
  TS_REQUIRE(vote_stride >= max_n, TS_EWORKSPACE, "vote_stride %lld < max candidates %d",
             (long long)vote_stride, max_n);
  if (max_n <= 0) return TS_OK;
  ZeroSet zero;
  score_votes_zero_regions(cfg, bt, w, workspace, &zero);
  TS_TRY(launch_select_zero(zero, (hipStream_t)stream));
  return launch_score_votes(cfg, bt, qf, k_pool, pool_rows, skip, votes, vote_stride, nullptr, 0,
                            workspace, (hipStream_t)stream);
}

int ts_select_supported(const ts_config* cfg, int32_t batch, int32_t max_seq_len) {
  if (validate_config(cfg) != TS_OK || batch < 1 || max_seq_len < 1) return 0;
  return fused_tokens_per_block(cfg, batch, max_seq_len, false, nullptr, false, nullptr) > 0 ? 1 : 0;
}

size_t ts_select_workspace_bytes(const ts_config* cfg, int32_t batch, int32_t max_seq_len) {
  if (validate_config(cfg) != TS_OK || batch < 1 || max_seq_len < 1) return 0;
  return select_workspace(cfg, batch, max_seq_len).total;
}

// Argument checks shared by the three forms of the call.
static int check_select(const ts_config* cfg, const ts_batch* bt, const void* workspace,
                        size_t workspace_bytes, SelectWorkspace* w_out) {
  TS_TRY(validate_config(cfg));
  TS_TRY(validate_batch(cfg, bt));
  TS_REQUIRE(workspace != nullptr, TS_EINVAL, "ts_select: NULL workspace");
  TS_REQUIRE_ALIGNED(workspace, 256, "workspace");
  const SelectWorkspace w = select_workspace(cfg, bt->batch, bt->max_seq_len);
  TS_REQUIRE(w.tokens_per_block > 0, TS_ESHAPE,
             "ts_select: batch %d x %d tokens does not fit one co-resident grid (or pool_kernel is "
             "above 256); use ts_score + ts_vote + ts_topk_ragged",
             bt->batch, bt->max_seq_len);
  TS_REQUIRE(workspace_bytes >= w.total, TS_EWORKSPACE, "ts_select: workspace %zu bytes < required %zu",
             workspace_bytes, w.total);
  *w_out = w;
  return TS_OK;
}

int ts_select_clear(const ts_config* cfg, const ts_batch* bt, void* workspace,
                    size_t workspace_bytes, ts_stream_t stream) {
  SelectWorkspace w;
  TS_TRY(check_select(cfg, bt, workspace, workspace_bytes, &w));
  ZeroSet zero;
  select_zero_regions(cfg, w, workspace, bt->batch, &zero);
  return launch_select_zero(zero, (hipStream_t)stream);
}

int ts_select_cleared_bounded(const ts_config* cfg, const ts_batch* bt, const void* qf,
                              const void* k_pool, int64_t pool_rows, const int32_t* hit,
                              const ts_selcache* cache, int32_t* sel, int32_t* sel_pos,
                              int64_t sel_stride, int32_t* sel_len, float* votes,
                              int64_t vote_stride, void* workspace, size_t workspace_bytes,
                              uint64_t wait_ticks, int32_t absent_workgroups, ts_stream_t stream) {
  SelectWorkspace w;
  TS_REQUIRE(wait_ticks >= 1 && absent_workgroups >= 0, TS_EINVAL,
             "ts_select: wait_ticks %llu / absent_workgroups %d out of range",
             (unsigned long long)wait_ticks, absent_workgroups);
  TS_TRY(check_select(cfg, bt, workspace, workspace_bytes, &w));
  TS_REQUIRE(qf && k_pool && sel && sel_pos && sel_len, TS_EINVAL, "ts_select: NULL tensor argument");
  TS_REQUIRE_ALIGNED(qf, 16, "qf");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  const int max_sel = cfg->n_init + cfg->top_k + cfg->n_local;
  TS_REQUIRE(sel_stride >= max_sel, TS_EWORKSPACE, "sel_stride %lld < n_init+top_k+n_local = %d",
             (long long)sel_stride, max_sel);
  const int max_n = bt->max_seq_len - cfg->n_init - cfg->n_local;
  TS_REQUIRE(votes == nullptr || vote_stride >= max_n, TS_EWORKSPACE,
             "vote_stride %lld < max candidates %d", (long long)vote_stride, max_n);
  TS_REQUIRE(hit == nullptr || cache != nullptr, TS_EINVAL,
             "ts_select: hit flags need the selection cache");
  if (cache)
    TS_REQUIRE(cache->topk_cache && cache->cache_len, TS_EINVAL,
               "ts_select: selection cache has a NULL array");
  return launch_select(cfg, bt, qf, k_pool, pool_rows, hit, cache, sel, sel_pos, sel_stride, sel_len,
                       votes, vote_stride, workspace, nullptr, 0, (hipStream_t)stream, wait_ticks,
                       (uint32_t)absent_workgroups);
}

int ts_select_cleared(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
                      int64_t pool_rows, const int32_t* hit, const ts_selcache* cache, int32_t* sel,
                      int32_t* sel_pos, int64_t sel_stride, int32_t* sel_len, float* votes,
                      int64_t vote_stride, void* workspace, size_t workspace_bytes,
                      ts_stream_t stream) {
  return ts_select_cleared_bounded(cfg, bt, qf, k_pool, pool_rows, hit, cache, sel, sel_pos, sel_stride,
                                   sel_len, votes, vote_stride, workspace, workspace_bytes,
                                   bt ? select_wait_ticks(bt) : 1, bt ? std::max(bt->absent_workgroups, 0) : 0,
                                   stream);
}

int ts_select(const ts_config* cfg, const ts_batch* bt, const void* qf, const void* k_pool,
              int64_t pool_rows, const int32_t* hit, const ts_selcache* cache, int32_t* sel,
              int32_t* sel_pos, int64_t sel_stride, int32_t* sel_len, float* votes,
              int64_t vote_stride, void* workspace, size_t workspace_bytes, ts_stream_t stream) {
  TS_TRY(ts_select_clear(cfg, bt, workspace, workspace_bytes, stream));
  return ts_select_cleared(cfg, bt, qf, k_pool, pool_rows, hit, cache, sel, sel_pos, sel_stride,
                           sel_len, votes, vote_stride, workspace, workspace_bytes, stream);
}

int ts_paged_matmul(const void* query, const void* token, int64_t pool_rows,
                    const int32_t* indices, void* scores, int32_t scores_dtype, int64_t n,
                    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                    ts_stream_t stream) {
  TS_REQUIRE(query && token && indices && scores, TS_EINVAL, "ts_paged_matmul: NULL tensor argument");
  TS_REQUIRE_ALIGNED(query, 16, "query");
  TS_REQUIRE_ALIGNED(token, 16, "token");
  TS_REQUIRE(head_dim == kHeadDim, TS_ESHAPE, "head_dim %d not supported (only 128)", head_dim);
  TS_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0, TS_ESHAPE,
             "num_heads %d / num_kv_heads %d invalid", num_heads, num_kv_heads);
  TS_REQUIRE(group_supported(num_kv_heads, num_heads / num_kv_heads), TS_ESHAPE,
             "unsupported head shape: num_kv_heads=%d group=%d", num_kv_heads,
             num_heads / num_kv_heads);
  TS_REQUIRE(scores_dtype == TS_DTYPE_F32 || scores_dtype == TS_DTYPE_BF16, TS_EINVAL,
             "scores_dtype %d unknown", scores_dtype);
  TS_REQUIRE(n >= 0 && n <= 0x7fffffffLL, TS_EINVAL, "n %lld out of range", (long long)n);
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  if (n == 0) return TS_OK;

  ScoreArgs a{};
  a.qf = (const uint16_t*)query;
  a.k_pool = (const uint16_t*)token;
  a.pool_rows = (uint32_t)pool_rows;
  a.seq_lens = nullptr;
  a.table = indices;
  a.table_stride = 0;
  a.k_per_req = nullptr;
  a.skip = nullptr;
  a.n_init = a.n_local = 0;
  a.top_k = 1;
  a.max_seq_len = 0;
  a.page_size = 1;
  a.page_shift = 0;
  a.direct_n = n;
  a.scores = scores;
  a.score_stride = n;
  a.partials = nullptr;
  a.tokens_per_block = score_tokens_per_block(n, num_heads);
  a.nchunks = (int)ceil_div(n, a.tokens_per_block);
  a.num_heads = num_heads;
  a.head_map = TS_HEADMAP_MOD;
  const dim3 grid((unsigned)a.nchunks, 1);
  if (scores_dtype == TS_DTYPE_BF16)
    return launch_score<true, kScoreDirect>(num_kv_heads, num_heads / num_kv_heads, a, grid,
                                     (hipStream_t)stream);
  return launch_score<false, kScoreDirect>(num_kv_heads, num_heads / num_kv_heads, a, grid,
                                    (hipStream_t)stream);
}

}  // extern "C"
