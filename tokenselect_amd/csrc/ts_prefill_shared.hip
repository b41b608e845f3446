// The prefill attention where there are many query rows: a long chunk, or the chunks of a prompt together
// (FlashInfer paged prefill, tr.py:759-771; what is computed, and the staging area it reads, are in
// ts_prefill.hip).
//
// prefill_attn_kernel gives a workgroup 64 columns (query rows of a head) and its four wavefronts a
// quarter of the keys each, because a chunk alone has few workgroups.  Every workgroup then reads all of its
// head's tiles, 1.4 MB for 64 columns, and where several chunks have keys of their own they come from
// beyond L2: 25.7 us a workgroup, and fifteen chunks of 28 heads on 4 (13.1 workgroups per CU) 337 us.
// Here a wavefront has 64 columns of its own and all keys, so that a workgroup has 256 columns: a quarter of
// the reads, nothing to merge, and 84 tiles instead of 21 for the rotation of the queries and the first loads
// to be paid from.  68 us a workgroup, 0.70 of it the matrix unit's: 5712 products of 16.5 cycles, at the
// 2.1 GHz that the device keeps up under them.
//
// The tiles pass through LDS, past the registers.  From there the operands go to the registers as they do from
// L2 in the other kernel: an operand is refilled as soon as its last product is issued, a whole iteration
// before it is needed.  Cycles of a tile, 512 rows over 2688 keys: 1660 with the loop as in the other kernel,
// 1550 with it unrolled by two (no copies of the logits) and the weights, their packing and the maxima dealt out
// over all 68 products, a wavefront issuing hardly more than one instruction beside a product for nothing; 1530 with
// the buffers' addresses from one scalar.  Of these the exponentials are 110, the reads of LDS 110, the loads to it
// 50 and the maxima 90 more than the products alone (1165).  72.5 -> 68.5 us a workgroup and not a tenth less,
// because the clock goes down as the matrix unit's share goes up: 2.13 -> 2.08 GHz, and a probe of the products alone
// is at 2.1.  18 chunks of 28 heads 289 -> 279 us.  What did not help: 32x32x16 products (1360 cycles, but at 1.78
// GHz: their accumulators' registers are read and written twice as often for the same sums), four products in a
// row into one accumulator (3 % less in the probe, here all operands of K are refilled at the end of a pass: 1585).
//
// Jobs that are cut: 256 columns and their keys are a job, and where the jobs do not fill whole waves of a workgroup per
// CU, or are of very different lengths (a long dense chunk, whose first rows see few keys), the workgroups of the last
// wave and a bit take equal shares of what is left instead, in the order of the jobs, so that a share begins and ends within
// a job; the pieces of a job meet in memory.  A piece costs 6.5 us before its first tile (1.5 until the queries are
// asked for, 2 until all is, 2.2 for their rotation, 1 for the first logits), 2.5 to be left or 4.5 to be added up, 2.2 for
// the output: some 10 tiles.  us for a whole call, without and with: eight chunks of 28 heads on 4 (1.75 waves) 229 ->
// 198, six (1.3) 177 -> 162, six of 32 on 8 (1.5) 191 -> 183, three of 28 (0.6) 117 -> 110; 2048 dense rows of 28 heads
// 61 -> 54, 2560 of 32 75 -> 73.  That the first operands pass through LDS as the others do (each wavefront for itself
// asked for 96 KB a workgroup in place of 24: 2.7 us until all was), the scale is the rotation's, and the output is written in
// pieces of 16 bytes (3.6 -> 2.0 us) made a workgroup 79 -> 77 us, which four waves of them give back to the clock.
//
// Which columns: the query rows of a chunk are cut into tiles of 16, the G heads of a KV head that see the same
// tile are G column blocks, and these are numbered tile by tile.  A workgroup takes sixteen in a
// row, so that no column is left without a head whatever G is.
#include <algorithm>
#include <utility>

#include "ts_prefill.h"

namespace ts {

constexpr int kPsWaves = 4;
constexpr int kPsThreads = 64 * kPsWaves;
constexpr int kPsUnits = kPsWaves * kPfBlocks;             // column blocks of a workgroup
constexpr int kPsPackage = 2 * kPfOperands * 64;           // a K tile and a V^T tile, in 16 bytes
constexpr int kPsBuffers = 4;
typedef __attribute__((ext_vector_type(4))) uint32_t ps_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t ps_u32x2;
constexpr int kPsCoherent = 16;  // a buffer access past the XCD's L2 (sc1), as agent-scope atomics are
constexpr int kPsCost = 10;       // what a piece of a job costs besides its tiles, in tiles
constexpr int kPsLeast = 8;      // tiles of a piece of a job that is cut, at least
constexpr size_t kPsLdsBytes = (size_t)kPsBuffers * kPsPackage * 16;  // 64 KB

// Two kilobytes, 16 bytes per lane of each, from `at` (of the lane) bytes behind the start of `from` to `to` (a byte of
// LDS), past the registers (the offset of the second counts on both sides).  All of the offset is the lanes' own: that is
// the part of an address that a raw buffer's size bounds, so that what would lie past the end of `from` is not read (it
// arrives as zeros, and nothing uses it), wherever the memory behind it ends.  A scalar offset is not part of that check.
// Assembly, because the compiler would wait for it at the next read of LDS, wherever that reads; nothing is returned to
// a register, and the waits are in the loop.
typedef __attribute__((ext_vector_type(4))) uint32_t ps_buffer;  // a buffer resource: base, size, raw dwords
__device__ __forceinline__ ps_buffer buffer_of(const void* from, int64_t bytes) {
  const uint64_t at = (uint64_t)from;
  return ps_buffer{(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, (uint32_t)(bytes > 0 ? bytes : 0), 0x00020000u};
}
__device__ __forceinline__ void load_to_lds(uint32_t to, const ps_buffer& from, uint32_t at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:1024 lds"
               :
               : "s"(to), "v"(at), "s"(from)
               : "m0", "memory");
}

// f(0), f(1) .. f(N - 1), each with a constant.
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

// Beside the 68 products of an iteration goes an even share of what else there is to do: before product n so many
// weights are made, and so many words of two packed.
constexpr int weighed(int n) { return n <= 0 ? 0 : n <= 32 ? 20 * n / 32 : n < 54 ? 20 + 12 * (n - 32) / 22 : 32; }
constexpr int packed(int n) { return weighed(n - 1) / 2; }
constexpr int kMaxAt = 8;  // the product of the second thirty-six behind which the search for the largest logit begins

// ---- the jobs that are cut (PrefillCuts)
// The tiles that the rows of workgroup i of a chunk of m rows see, of `keys` keys.
__host__ __device__ __forceinline__ int job_tiles(int keys, int m, int i, int group) {
  const int row_end = (i * kPsUnits + kPsUnits - 1) / group * 16 + 16;
  const int last = keys - m + (row_end < m ? row_end : m) - 1;
  return last < 0 ? 1 : last / kPfKeys + 1;
}
// Job j of a KV head, the chunks one after the other, the last rows of each first.
struct PsJob {
  int chunk, m, i, tiles;
};
__host__ __device__ __forceinline__ PsJob job_at(const PrefillCuts& c, int rows, int chunk_rows, int group, int j) {
  PsJob job;
  job.chunk = j / c.per_chunk < c.chunks ? j / c.per_chunk : c.chunks - 1;
  const int begin = job.chunk * c.per_chunk;
  job.m = rows - job.chunk * chunk_rows < chunk_rows ? rows - job.chunk * chunk_rows : chunk_rows;
  job.i = (job.chunk + 1 < c.chunks ? c.per_chunk : c.jobs - begin) - 1 - (j - begin);
  job.tiles = job_tiles(c.keys, job.m, job.i, group);
  return job;
}
// Where a boundary that lies `at` tiles into a job cuts it: not so close to an end that a piece would be shorter than
// kPsLeast; 0 and `tiles` are no cut.
__host__ __device__ __forceinline__ int cut_at(int at, int tiles) {
  return at >= tiles ? tiles : at < kPsLeast ? 0 : at > tiles - kPsLeast ? tiles : at;
}

constexpr int kPsPiece = 4 * 8 * 64 * 16 + 4 * 64 * 8;  // bytes that a wavefront leaves of a piece: sums; maxima and weights
constexpr int kPsPieces = 2 * kPsSlots;                 // two of each workgroup: one cut at its start, one at its end
static_assert(kPsTicketBytes == kPsSlots * kPsWaves * 4, "a ticket per wavefront of the workgroup that has a job's first piece");
size_t prefill_cut_bytes() { return kPsTicketBytes + (size_t)kPsPieces * kPsWaves * kPsPiece; }

template <bool CAP>
__global__ __launch_bounds__(kPsThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_shared_kernel(
    PrefillArgs a, PrefillCuts cuts) {
  constexpr int CB = kPfBlocks;
  extern __shared__ __attribute__((aligned(16))) uint4 ps_lds[];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int qc = lane & 15, g4 = lane >> 4;  // query column / key group of the matrix layouts
  // The KV head fastest, as in the other kernel; the last rows, which see the most keys, start first.
  const int kvh = blockIdx.x;
  const int G = a.num_heads / a.num_kv_heads;
  // This workgroup's job; or, of those that share the last jobs, where it begins: `own` is its number among
  // them, its share the costs [own, own + 1) x quantum, `job_cost` the costs before the job, `t_from` the tile.
  int j = blockIdx.y, t_from = 0, job_cost = 0;
  const int own = (int)blockIdx.y - cuts.whole;
  if (own >= 0) {
    const int target = own * cuts.quantum;
    bool found = false;
    for (int base = cuts.whole; base < cuts.jobs && !found; base += 64) {
      const int at = base + lane;
      const int cost = at < cuts.jobs ? kPsCost + job_at(cuts, a.rows, a.chunk_rows, G, at).tiles : 0;
      int upto = cost;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int before = __shfl_up(upto, off);
        upto += lane >= off ? before : 0;
      }
      const uint64_t behind = __ballot(job_cost + upto > target);
      if (behind != 0) {
        const int l = __builtin_ctzll(behind);
        j = base + l;
        const int tiles = __builtin_amdgcn_readlane(cost, l) - kPsCost;
        job_cost += __builtin_amdgcn_readlane(upto, l) - tiles - kPsCost;
        t_from = cut_at(target - job_cost - kPsCost, tiles);
        if (t_from == tiles) {
          job_cost += tiles + kPsCost;
          t_from = 0;
          ++j;
        }
        found = j < cuts.jobs;
        break;
      }
      job_cost += __builtin_amdgcn_readlane(upto, 63);
    }
    if (!found) return;
  }
  for (;;) {  // over the jobs of a share
  j = __builtin_amdgcn_readfirstlane(j);
  t_from = __builtin_amdgcn_readfirstlane(t_from);
  job_cost = __builtin_amdgcn_readfirstlane(job_cost);
  const PsJob job = job_at(cuts, a.rows, a.chunk_rows, G, j);
  // Its end: within the job, at its end, or further on.
  int t_to = job.tiles;
  bool more = false;
  if (own >= 0) {
    const int end = (own + 1) * cuts.quantum - kPsCost;  // in tiles of this job: less job_cost
    t_to = cut_at(end - job_cost, job.tiles);
    if (t_to == job.tiles && j + 1 < cuts.jobs) {
      const int next_cost = job_cost + kPsCost + job.tiles;
      more = cut_at(end - next_cost, job_at(cuts, a.rows, a.chunk_rows, G, j + 1).tiles) > 0;
    }
  }
  const bool cut = t_from > 0 || t_to < job.tiles;
  const int chunk = job.chunk, m = job.m;
  const int unit0 = job.i * kPsUnits;
  const int first_row = chunk * a.chunk_rows;
  const int row_begin = unit0 / G * 16;                     // of the workgroup
  const int row_end = min((unit0 + kPsUnits - 1) / G * 16 + 16, m);
  int row0[CB], head[CB];      // of the column blocks: first row, head
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int unit = unit0 + CB * wave + cb;
    row0[cb] = unit / G * 16;
    head[cb] = kvh * G + unit % G;
  }

  const size_t head_at = chunk * a.stage_stride + (size_t)kvh * a.s_pad * kHeadDim;
  // ---- queries: B operand, lane (qc, g4) holds dims [32 ks + 8 g4, +8) of its column block's row.
  // Their loads do not wait for the selection's length.
  const int listed = a.sel_len[chunk];
  uint4 raw[CB][4];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const uint16_t* const row =
        a.q + (size_t)(first_row + min(row0[cb] + qc, m - 1)) * a.q_stride + head[cb] * kHeadDim + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) raw[cb][ks] = *(const uint4*)(row + 32 * ks);
  }
  // The tiles pass through LDS.  Package t, what the operands' registers are refilled with in iteration t of the loop
  // below, is the K tile t + 2 and the V^T tile t + 1: sixteen kilobytes, of which a wavefront asks for four.  The
  // first operands, the K tiles t_from and t_from + 1 and the V^T tile t_from, are the two packages before the loop's, as
  // far as they are needed.  (A tile past the staging area, asked for ahead and never used, arrives as zeros.)
  constexpr uint32_t kBytes = kPsPackage * 16, kPart = kBytes / 2 / kPsWaves;
  const uint32_t lane16 = 16 * lane, part_at = kPart * wave;
  const int64_t tiles_bytes = (int64_t)a.s_pad * kHeadDim * 2 - kPart * wave;
  {
    // (behind the queries, which are wanted first: loads return in order)
    const ps_buffer k_tiles = buffer_of(a.kr + head_at + kPart / 2 * wave, tiles_bytes);
    const ps_buffer v_tiles = buffer_of(a.vt + head_at + kPart / 2 * wave, tiles_bytes);
    const uint32_t at = lane16 + 2 * kPfTileElems * t_from;
    load_to_lds(part_at + 2 * kBytes, k_tiles, at);
    load_to_lds(part_at + 3 * kBytes, k_tiles, at + 2 * kPfTileElems);
    load_to_lds(part_at + 3 * kBytes + kBytes / 2, v_tiles, at);
  }
  const ps_buffer ask_k = buffer_of(a.kr + head_at + 2 * kPfTileElems + kPart / 2 * wave, tiles_bytes - 2 * 2 * kPfTileElems);
  const ps_buffer ask_v = buffer_of(a.vt + head_at + kPfTileElems + kPart / 2 * wave, tiles_bytes - 2 * kPfTileElems);
  uint32_t ask_at = lane16 + 2 * kPfTileElems * t_from;  // of the next package to be asked for, in the staging area
  auto ask_keys = [&](uint32_t buffer) __attribute__((always_inline)) { load_to_lds(part_at + buffer, ask_k, ask_at); };
  auto ask_values = [&](uint32_t buffer) __attribute__((always_inline)) {
    load_to_lds(part_at + buffer + kBytes / 2, ask_v, ask_at);
    ask_at += 2 * kPfTileElems;
  };
  const int S = __builtin_amdgcn_readfirstlane(min(max(listed, 0), a.max_sel_len));
  const int shift = S - m;  // query row i sits at position shift + i and sees keys <= that
  const bool rope = a.rope_mode == TS_ROPE_LLAMA;
  // (as in the other kernel: without a soft cap the softmax scale and log2(e) go into the query)
  const float qs = CAP ? 1.0f : a.sm_scale * kLog2e;
  pf_bf16x8 qb[CB][4];
  {
    // The rotation of the first rows while the queries are on their way.
    float sn[2][8], cs[2][8];
    int rotated;  // the rows that sn and cs are those of
    auto rotation = [&](int row) __attribute__((always_inline)) {
      rotated = row;
      const float pos = (float)(shift + min(row + qc, m - 1));
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float pair = (float)(32 * (e >> 3) + 8 * g4 + (e & 7));
        const float freq = a.rope_rcp_scale * exp2f(-pair * (2.0f / kHeadDim) * a.log2_theta);
        sincos_reduced(pos * freq, sn[e >> 3][e & 7], cs[e >> 3][e & 7]);
        sn[e >> 3][e & 7] *= qs;
        cs[e >> 3][e & 7] *= qs;
      }
    };
    if (rope) rotation(row0[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      if (cb == CB / 2) {
        // All queries are here: the loop's first packages are asked for now, and nothing waits for those with them.
#pragma unroll
        for (int late = CB / 2; late < CB; ++late)
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(raw[late][ks].x), "+v"(raw[late][ks].y), "+v"(raw[late][ks].z), "+v"(raw[late][ks].w));
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          ask_keys(t * kBytes);
          ask_values(t * kBytes);
        }
      }
      if (rope && row0[cb] != rotated) rotation(row0[cb]);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const uint32_t lw[4] = {raw[cb][ks].x, raw[cb][ks].y, raw[cb][ks].z, raw[cb][ks].w};
        const uint32_t hw[4] = {raw[cb][ks + 2].x, raw[cb][ks + 2].y, raw[cb][ks + 2].z, raw[cb][ks + 2].w};
        uint32_t lp[4], hp[4];
        if (rope) {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float lo[2] = {bf16_lo(lw[w]), bf16_hi(lw[w])}, hi[2] = {bf16_lo(hw[w]), bf16_hi(hw[w])};
            const float* const s = &sn[ks][2 * w];
            const float* const c = &cs[ks][2 * w];
            lp[w] = pack_bf16(lo[0] * c[0] - hi[0] * s[0], lo[1] * c[1] - hi[1] * s[1]);
            hp[w] = pack_bf16(hi[0] * c[0] + lo[0] * s[0], hi[1] * c[1] + lo[1] * s[1]);
          }
          asm volatile("" : "+v"(lp[0]));  // (two ways, not one with the results picked)
        } else {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            lp[w] = pack_bf16(bf16_lo(lw[w]) * qs, bf16_hi(lw[w]) * qs);
            hp[w] = pack_bf16(bf16_lo(hw[w]) * qs, bf16_hi(hw[w]) * qs);
          }
        }
        qb[cb][ks] = __builtin_bit_cast(pf_bf16x8, make_uint4(lp[0], lp[1], lp[2], lp[3]));
        qb[cb][ks + 2] = __builtin_bit_cast(pf_bf16x8, make_uint4(hp[0], hp[1], hp[2], hp[3]));
        keep_acc(qb[cb][ks]);
        keep_acc(qb[cb][ks + 2]);
      }
    }
  }

  // ---- main loop over the tiles that any row of this workgroup can see (none where the selection
  // reported a fault, S <= 0; rows at negative positions see no key of any: their sums stay zero, and so does
  // their output)
  const int last_visible = min(S, shift + row_end) - 1;
  const int visible = S > 0 && last_visible >= 0 ? last_visible / kPfKeys + 1 : 0;
  const int n_tiles = t_to < job.tiles ? min(t_to, visible) : visible;  // (the last piece goes to the end, wherever that is)
  const int masked = max(shift + row_begin + 1, 0) / kPfKeys;  // the first tile that some row must not see whole
  // Running maximum of each column's row: m_run (kNegBig: none yet), minus that as the
  // four-register start value of the logits' accumulators (0 while there is none), and the
  // excess over it that makes the row move (-inf while there is none: any finite logit does).
  float m_run[CB], raise_at[CB];
  pf_f32x4 minus_m[CB];  // (all zero with a soft cap, whose logits are shifted afterwards)
  pf_f32x4 o[CB][8], row_sum[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    m_run[cb] = kNegBig;
    raise_at[cb] = -INFINITY;
    minus_m[cb] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
    row_sum[cb] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      o[cb][db] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
      keep_acc(o[cb][db]);
    }
  }
  const pf_bf16x8 ones = __builtin_bit_cast(pf_bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));

  // The software pipeline of the other kernel.  Package t is asked for in iteration t - 2 (L2 takes 0.6 to 0.85 us, an
  // iteration 0.65), to buffer (t - t_from) % 4.
  // Before the barrier in the second half of iteration t a wavefront waits until its part of package t + 1
  // has come, which leaves that of package t + 2 under way, and until all but its last eight
  // reads of LDS are through.  The buffer that is asked for in iteration t had package t - 2: its reads
  // were issued in iteration t - 2 and, everybody's, through at the barrier of iteration t - 1.
  // The largest logit of the lane's eight.
  auto largest = [&](const pf_f32x4 (&s)[2]) __attribute__((always_inline)) {
    float mx = max3(s[0][0], s[0][1], s[0][2]);
    mx = max3(mx, s[0][3], s[1][0]);
    mx = max3(mx, s[1][1], s[1][2]);
    return fmaxf(mx, s[1][3]);
  };
  auto soft_cap = [&](pf_f32x4 (&s)[2], int cb) __attribute__((always_inline)) {
    const float shift_by = m_run[cb] == kNegBig ? 0.f : m_run[cb];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[kb][r] = a.logit_cap * tanhf(s[kb][r] * a.sm_scale / a.logit_cap) * kLog2e - shift_by;
  };
  // Masked logits are -inf: exp2 makes them 0 without a branch.
  auto mask = [&](int t, pf_f32x4 (&s)[2], int cb) __attribute__((always_inline)) {
    const int limit = shift + min(row0[cb] + qc, m - 1) - (t * kPfKeys + 4 * g4);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (16 * kb + r > limit) s[kb][r] = -INFINITY;
  };
  // Whether some row outgrew its maximum (or has none yet): the largest logit of all column blocks against the least
  // of their bounds.  (settle() of the other kernel)
  auto bound = [&]() __attribute__((always_inline)) { return fminf(fminf(raise_at[0], raise_at[1]), fminf(raise_at[2], raise_at[3])); };
  float raise_any = -INFINITY;
  // Agrees on the largest logit of the column's row, in the four lanes that have it, and moves the row's maximum there
  // if it outgrew that or has none; what its sums are to be multiplied by.
  auto raise = [&](pf_f32x4 (&s)[2], int cb) __attribute__((always_inline)) {
    const bool unset = m_run[cb] == kNegBig;
    float mx = largest(s);
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const bool take = mx > raise_at[cb];
    const float delta = take ? mx : 0.f;
    if (take) {
      m_run[cb] = unset ? delta : delta + m_run[cb];
      raise_at[cb] = kPfRaise;
      if (!CAP) {
        const float nm = -m_run[cb];
        minus_m[cb] = pf_f32x4{nm, nm, nm, nm};
      }
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[kb][r] -= delta;
    // (a row without a maximum has only zeros in its accumulators)
    return unset ? 1.0f : __builtin_amdgcn_exp2f(-delta);
  };
  auto settle = [&](pf_f32x4 (&s)[CB][2]) __attribute__((always_inline)) {
    mfma_settled(o);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const float scale = raise(s[cb], cb);
#pragma unroll
      for (int db = 0; db < 8; ++db) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[cb][db][r] *= scale;
        keep_acc(o[cb][db]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) row_sum[cb][r] *= scale;
    }
    raise_any = bound();
  };

  pf_bf16x8 kw[kPfOperands], vw[kPfOperands];  // the operands of the next K tile and of the current V^T tile
  // NEXT: there is a tile t + 1.  s_cur: the logits of tile t, which become its
  // weights; s_next: those of tile t + 1.
  uint32_t read_at = 0;  // the buffer of package t (that of package t + 2 is the one after the next)
  auto iteration = [&](int t, pf_f32x4 (&s_cur)[CB][2], pf_f32x4 (&s_next)[CB][2], auto next)
      __attribute__((always_inline)) {
    constexpr bool NEXT = decltype(next)::value;
    const pf_bf16x8* const from = (const pf_bf16x8*)((const char*)ps_lds + lane16 + read_at);
    uint32_t pw[CB][4];  // the weights, two to a word
    auto weigh = [&](int x) __attribute__((always_inline)) {  // x: 8 column block + element
      float p = s_cur[x >> 3][(x >> 2) & 1][x & 3];
      s_cur[x >> 3][(x >> 2) & 1][x & 3] = __builtin_amdgcn_exp2f(p);
    };
    auto pack = [&](int w) __attribute__((always_inline)) {  // w: two weights
      const pf_f32x4& p = s_cur[w >> 2][(w >> 1) & 1];
      pw[w >> 2][w & 3] = pack_bf16(p[2 * (w & 1)], p[2 * (w & 1) + 1]);
    };
    auto share = [&](auto at) __attribute__((always_inline)) {
      constexpr int n = decltype(at)::value;
      each<weighed(n + 1) - weighed(n)>([&](auto x) __attribute__((always_inline)) { weigh(weighed(n) + decltype(x)::value); });
      each<packed(n + 1) - packed(n)>([&](auto w) __attribute__((always_inline)) { pack(packed(n) + decltype(w)::value); });
    };
    each<32>([&](auto at) __attribute__((always_inline)) {
      constexpr int n = decltype(at)::value, i = n >> 2, cb = n & 3, kb = i >> 2, ks = i & 3;
      if (NEXT) s_next[cb][kb] = mfma_logits(ks == 0 ? minus_m[cb] : s_next[cb][kb], __builtin_bit_cast(uint4, kw[i]), qb[cb][ks]);
      share(at);
      if (NEXT && n == 1) ask_keys(read_at ^ 2 * kBytes);
      if (NEXT && n == 5) ask_values(read_at ^ 2 * kBytes);
      if (NEXT && cb == 3) kw[i] = from[64 * i];
      __builtin_amdgcn_sched_barrier(0);
    });
    float part[4];
    uint64_t moves = 0;
    pf_bf16x8 pb;
    each<36>([&](auto at) __attribute__((always_inline)) {
      constexpr int n = decltype(at)::value, cb = n / 9, db = n % 9;  // (the ninth: the sums of the weights)
      if (db == 0) {
        pb = __builtin_bit_cast(pf_bf16x8, make_uint4(pw[cb][0], pw[cb][1], pw[cb][2], pw[cb][3]));
        weights_settled(pb);
      }
      if (db < 8) mfma_acc(o[cb][db & 7], vw[db & 7], pb);
      else row_sum[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb, row_sum[cb], 0, 0, 0);
      share(std::integral_constant<int, 32 + n>{});
      if (NEXT && CAP && n < CB) soft_cap(s_next[n & 3], n & 3);
      // the largest of the thirty-two logits, an instruction at a time
      if (NEXT && n >= kMaxAt && n < kMaxAt + 17) {
        constexpr int step = n - kMaxAt, c = (step & 15) >> 2;
        const pf_f32x4 (&s)[2] = s_next[c];
        if (step == 16) moves = __ballot(max3(max3(part[0], part[1], part[2]), part[3], part[3]) > raise_any);
        else if ((step & 3) == 0) part[c] = max3(s[0][0], s[0][1], s[0][2]);
        else if ((step & 3) == 1) part[c] = max3(part[c], s[0][3], s[1][0]);
        else if ((step & 3) == 2) part[c] = max3(part[c], s[1][1], s[1][2]);
        else part[c] = max3(part[c], s[1][3], s[1][3]);
      }
      if (NEXT && n == 24) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(8)\n\ts_barrier" ::: "memory");
      if (NEXT && cb == 3 && db < 8) vw[db & 7] = from[64 * (kPfOperands + (db & 7))];
      __builtin_amdgcn_sched_barrier(0);
    });
    if (NEXT) {
      if (__builtin_expect((int)(t + 1 >= masked) | (int)(moves != 0), 0)) {
        if (t + 1 >= masked) {
          float mx = -INFINITY;
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) {
            mask(t + 1, s_next[cb], cb);
            mx = max3(mx, mx, largest(s_next[cb]));
          }
          moves = __ballot(mx > raise_any);
        }
        if (moves != 0) settle(s_next);
      }
      read_at = (read_at + kBytes) & (kPsBuffers * kBytes - 1);
    }
  };

  if (t_from < n_tiles) {
    pf_bf16x8 k_second[kPfOperands];
    pf_f32x4 s_even[CB][2], s_odd[CB][2];  // the logits of the even and of the odd tiles: [column block][key block]
    // The first operands, once everybody's parts have come.
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    {
      const pf_bf16x8* const from = (const pf_bf16x8*)((const char*)ps_lds + lane16 + 2 * kBytes);
#pragma unroll
      for (int i = 0; i < kPfOperands; ++i) {
        kw[i] = from[64 * i];
        k_second[i] = from[kPsPackage + 64 * i];
        vw[i] = from[kPsPackage + 64 * (kPfOperands + i)];
      }
    }
    // the first tile's logits: nothing comes before them
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        s_even[cb][i >> 2] = mfma_logits((i & 3) == 0 ? minus_m[cb] : s_even[cb][i >> 2], __builtin_bit_cast(uint4, kw[i]), qb[cb][i & 3]);
      kw[i] = k_second[i];
    }
    // (no sums yet that a maximum would move)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      if (CAP) soft_cap(s_even[cb], cb);
      if (masked <= t_from) mask(t_from, s_even[cb], cb);
      raise(s_even[cb], cb);
    }
    raise_any = bound();
    // (the compiler waits for the operands here, and not in every iteration for what may be the first's)
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) asm volatile("" : "+v"(kw[i]), "+v"(vw[i]));
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    using Yes = std::true_type;
    using No = std::false_type;
    int t = t_from;
    for (; t + 2 < n_tiles; t += 2) {
      iteration(t, s_even, s_odd, Yes{});
      iteration(t + 1, s_odd, s_even, Yes{});
    }
    if (t + 1 < n_tiles) {
      iteration(t++, s_even, s_odd, Yes{});
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        s_even[cb][0] = s_odd[cb][0];
        s_even[cb][1] = s_odd[cb][1];
      }
    }
    iteration(t, s_even, s_odd, No{});
    mfma_settled(o);
  }
  // What was asked for past the end comes before the space may be another workgroup's.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // The length of a dense chunk, whose gather is through (nothing here reads it).
  if (a.new_len && j == 0 && t_from == 0 && kvh == 0 && threadIdx.x == 0) *a.new_len = min(*a.new_len + m, a.len_cap);
  bool write = true;
  if (cut) {
    // A wavefront leaves what it has of its columns and draws a ticket of the job's; the last to draw adds up the
    // pieces.  Nobody waits.  (What is left is visible by the time the ticket is drawn: written past the L2, and waited
    // for.)  Of two pieces the one that finds the other's ticket drawn is not left anywhere.
    const int first_cut = (job_cost + kPsCost + kPsLeast + cuts.quantum - 1) / cuts.quantum;
    const int pieces = (job_cost + kPsCost + job.tiles - kPsLeast) / cuts.quantum - first_cut + 2;
    const int mine = own - first_cut + 1;
    const int slot0 = kvh * cuts.streams + first_cut - 1;  // of the workgroup with the first piece
    uint32_t* const ticket = cuts.tickets + slot0 * kPsWaves + wave;
    auto piece = [&](int p) __attribute__((always_inline)) {
      return __builtin_amdgcn_make_buffer_rsrc(
          cuts.pieces + ((size_t)(2 * (slot0 + p) + (p == 0)) * kPsWaves + wave) * kPsPiece, 0, kPsPiece, 0x00020000);
    };
    const bool two = pieces == 2;
    write = two && __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
    if (!write) {
      const auto to = piece(mine);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
        for (int db = 0; db < 8; ++db)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(ps_u32x4, o[cb][db]), to, lane16, (8 * cb + db) * 1024, kPsCoherent);
        const ps_u32x2 ml = {__float_as_uint(m_run[cb]), __float_as_uint(row_sum[cb][0])};
        __builtin_amdgcn_raw_buffer_store_b64(ml, to, 8 * lane, 32 * 1024 + cb * 512, kPsCoherent);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      uint32_t before = 0;
      if (lane == 0) before = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      write = __builtin_amdgcn_readfirstlane((int)before) + 1 == pieces;
    }
    if (write) {
      // Two pieces: the other one to this one, the same sums whichever came last.  More: from the first on.
      if (!two) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          m_run[cb] = kNegBig;
          row_sum[cb][0] = 0.f;
#pragma unroll
          for (int db = 0; db < 8; ++db) {
            o[cb][db] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
            keep_acc(o[cb][db]);
          }
        }
      }
      for (int p = two ? 1 - mine : 0; p < (two ? 2 - mine : pieces); ++p) {
#pragma clang fp contract(off)
        const auto from = piece(p);
        pf_f32x4 x[CB][8];
        ps_u32x2 ml[CB];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          ml[cb] = __builtin_bit_cast(ps_u32x2, __builtin_amdgcn_raw_buffer_load_b64(from, 8 * lane, 32 * 1024 + cb * 512, kPsCoherent));
#pragma unroll
          for (int db = 0; db < 8; ++db)
            x[cb][db] = __builtin_bit_cast(pf_f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, lane16, (8 * cb + db) * 1024, kPsCoherent));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const float m_p = __uint_as_float(ml[cb].x), m_new = fmaxf(m_run[cb], m_p);
          const float e0 = __builtin_amdgcn_exp2f(m_run[cb] - m_new), e1 = __builtin_amdgcn_exp2f(m_p - m_new);
          m_run[cb] = m_new;
          row_sum[cb][0] = row_sum[cb][0] * e0 + __uint_as_float(ml[cb].y) * e1;
#pragma unroll
          for (int db = 0; db < 8; ++db) {
#pragma unroll
            for (int r = 0; r < 4; ++r) o[cb][db][r] = o[cb][db][r] * e0 + x[cb][db][r] * e1;
            keep_acc(o[cb][db]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  // o[cb][db][r] = O[query qc][dim 16 db + 4 g4 + r]; the row sum is complete in every lane.  Of two blocks of 16 dims the
  // even lane groups take the first, the odd ones the second, so that a lane has eight dims in a row.
  if (write) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int row = row0[cb] + qc;
      const float l = row_sum[cb][0], inv = l > 0.f ? 1.0f / l : 0.f;
      uint16_t* const to = a.out + ((size_t)(first_row + row) * a.num_heads + head[cb]) * kHeadDim + 16 * (g4 & 1) + 8 * (g4 >> 1);
#pragma unroll
      for (int db = 0; db < 8; db += 2) {
        const auto first = [&](int at) { return pack_bf16(o[cb][db][at] * inv, o[cb][db][at + 1] * inv); };
        const auto second = [&](int at) { return pack_bf16(o[cb][db + 1][at] * inv, o[cb][db + 1][at + 1] * inv); };
        const ps_u32x2 x = __builtin_amdgcn_permlane16_swap(first(0), second(0), false, false);
        const ps_u32x2 y = __builtin_amdgcn_permlane16_swap(first(2), second(2), false, false);
        if (row < m) *(uint4*)(to + 16 * db) = make_uint4(x.x, y.x, x.y, y.y);
      }
    }
  }
  if (!more) return;
  job_cost += kPsCost + job.tiles;
  t_from = 0;
  ++j;
  __syncthreads();  // (everybody is through with the buffers)
  }
}

int64_t prefill_shared_workgroups(int num_heads, int num_kv_heads, int chunk_rows) {
  return ceil_div(ceil_div(chunk_rows, 16) * (num_heads / num_kv_heads), kPsUnits) * num_kv_heads;
}

PrefillCuts prefill_cuts(int num_heads, int num_kv_heads, int rows, int chunk_rows, int keys, void* workspace) {
  PrefillCuts c{};
  const int group = num_heads / num_kv_heads, streams = kPsSlots / num_kv_heads;
  auto workgroups = [&](int m) { return (int)ceil_div(ceil_div(m, 16) * group, kPsUnits); };
  c.chunks = (int)ceil_div(rows, chunk_rows);
  c.per_chunk = workgroups(std::min(rows, chunk_rows));
  c.jobs = (c.chunks - 1) * c.per_chunk + workgroups(rows - (c.chunks - 1) * chunk_rows);
  c.keys = keys;
  c.whole = c.jobs;
  // Shares are of all jobs where these are of very different lengths (2048 rows of a dense chunk, a wave: 62 -> 56 us), and
  // otherwise of what is left of whole waves and of one wave more (of what is left alone, 0.2 to 0.7 waves: six chunks
  // of 32 heads 188 us, 183 so).  A last wave that is 0.85 full is left as it is.
  const int rest = c.jobs % streams, m = std::min(rows, chunk_rows);
  const bool even = 2 * job_tiles(keys, m, 0, group) >= job_tiles(keys, m, c.per_chunk - 1, group);
  if (workspace == nullptr || (even && (rest == 0 || 100 * rest >= 85 * streams))) return c;
  c.streams = streams;
  c.whole = even ? std::max(c.jobs / streams - 1, 0) * streams : 0;
  int64_t cost = 0;
  for (int j = c.whole; j < c.jobs; ++j) cost += kPsCost + job_at(c, rows, chunk_rows, group, j).tiles;
  c.quantum = (int)std::max<int64_t>(ceil_div(cost, c.streams), kPsCost + 2 * kPsLeast);
  c.tickets = (uint32_t*)workspace;
  c.pieces = (char*)workspace + kPsTicketBytes;
  return c;
}

// Whether the jobs of one long dense chunk are shared out, by what the launch would take either way, in tiles.  Cut, all
// of a head's jobs and ten tiles each divided by its workgroups, and 26 for what is cut on top.  As they are, the longest start
// first and whoever is through takes the next, sixteen tiles each besides their own: within a wave the longest, within
// two also two from the middle (whose lengths go down evenly, so that any such two are as long), within three the longest
// of the third on top of these; with more, and below 0.87 waves, sharing pays nowhere.  By four tiles at least, this says the
// right thing for all of 73 sizes of 16 to 64 heads, 1024 to 4700 rows.  us for a whole call uncut and cut, where it says cut: 24 on 8, 2560
// rows (0.94 waves) 75 and 65, 32 on 8, 2048 (1) 63 and 59, 2688 (1.31) 79 and 75, 28 on 4, 2560 (1.09) 73 and 68, 64 on 8, 2304 (2.25) 104 and
// 101; where it says not: 64 on 8, 1024 rows (1) 44.5 and 50, 1536 (1.5) 59 and 67, 40 on 8, 1792 (1.09) 59 and 61, 32 on 8, 3200 (1.56) 92.5 and 97,
// 4000 (1.97) 127 and 135, 28 on 4, 4000 (1.72) 115 and 124, 56 on 8, 4000 (3.44) 213 and 224.
bool prefill_dense_cuts_pay(int num_heads, int num_kv_heads, int rows, int keys) {
  const int group = num_heads / num_kv_heads, streams = kPsSlots / num_kv_heads;
  const int jobs = (int)ceil_div(ceil_div(rows, 16) * group, kPsUnits);
  if (jobs * num_kv_heads < 224 || jobs > 3 * streams) return false;
  auto tiles = [&](int j) { return job_tiles(keys, rows, jobs - 1 - j, group); };  // of the j-th to start
  constexpr int kUncut = 16, kCut = 26, kLeastGain = 4;
  int64_t cost = 0;
  for (int j = 0; j < jobs; ++j) cost += kPsCost + tiles(j);
  int whole = tiles(0) + kUncut;
  if (jobs > streams) whole = std::max(whole, tiles(streams - 1) + tiles(streams) + 2 * kUncut);
  if (jobs > 2 * streams) whole += tiles(2 * streams) + kUncut;
  return ceil_div(cost, streams) + kCut + kLeastGain <= whole;
}

int launch_prefill_shared(const PrefillArgs& a, const PrefillCuts& cuts, hipStream_t stream) {
  const dim3 grid((unsigned)a.num_kv_heads, (unsigned)(cuts.whole + cuts.streams));
  const auto kernel = a.logit_cap > 0.f ? prefill_shared_kernel<true> : prefill_shared_kernel<false>;
  static const hipError_t ok[2] = {
      hipFuncSetAttribute((const void*)prefill_shared_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPsLdsBytes),
      hipFuncSetAttribute((const void*)prefill_shared_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPsLdsBytes)};
  if (ok[0] != hipSuccess || ok[1] != hipSuccess)
    return fail(TS_EHIP, "prefill attention: %zu bytes of LDS refused", kPsLdsBytes);
  hipLaunchKernelGGL(kernel, grid, dim3(kPsThreads), kPsLdsBytes, stream, a, cuts);
  return check_launch("prefill_shared_kernel");
}

}  // namespace ts
