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
// Which columns: the query rows of a chunk are cut into tiles of 16, the G heads of a KV head that see the same
// tile are G column blocks, and these are numbered tile by tile.  A workgroup takes sixteen in a
// row, so that no column is left without a head whatever G is.
#include <utility>

#include "ts_prefill.h"

namespace ts {

constexpr int kPsWaves = 4;
constexpr int kPsThreads = 64 * kPsWaves;
constexpr int kPsUnits = kPsWaves * kPfBlocks;             // column blocks of a workgroup
constexpr int kPsPackage = 2 * kPfOperands * 64;           // a K tile and a V^T tile, in 16 bytes
constexpr int kPsBuffers = 4;
constexpr size_t kPsLdsBytes = (size_t)kPsBuffers * kPsPackage * 16;  // 64 KB

// Two kilobytes, 16 bytes per lane of each, from `at` bytes behind the start of `from` to `to` (a byte of LDS), past
// the registers (the offset of the second counts on both sides; what lies past the end of `from` arrives as zeros).
// Assembly, because the compiler would wait for it at the next read of LDS, wherever that reads; nothing is returned to
// a register, and the waits are in the loop.
typedef __attribute__((ext_vector_type(4))) uint32_t ps_buffer;  // a buffer resource: base, size, raw dwords
__device__ __forceinline__ ps_buffer buffer_of(const void* from, int64_t bytes) {
  const uint64_t at = (uint64_t)from;
  return ps_buffer{(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, (uint32_t)(bytes > 0 ? bytes : 0), 0x00020000u};
}
__device__ __forceinline__ void load_to_lds(uint32_t to, const ps_buffer& from, uint32_t at, uint32_t lane16) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\tbuffer_load_dwordx4 %1, %2, %3 offen offset:1024 lds"
               :
               : "s"(to), "v"(lane16), "s"(from), "s"(at)
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

template <bool CAP>
__global__ __launch_bounds__(kPsThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_shared_kernel(
    PrefillArgs a) {
  constexpr int CB = kPfBlocks;
  extern __shared__ __attribute__((aligned(16))) uint4 ps_lds[];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int qc = lane & 15, g4 = lane >> 4;  // query column / key group of the matrix layouts
  // The KV head fastest, as in the other kernel; the last rows, which see the most keys, start first.
  const int kvh = blockIdx.x, chunk = blockIdx.z;
  const int G = a.num_heads / a.num_kv_heads;
  const int unit0 = (int)(gridDim.y - 1 - blockIdx.y) * kPsUnits;
  const int first_row = chunk * a.chunk_rows;
  const int m = min(a.chunk_rows, a.rows - first_row);
  const int row_begin = unit0 / G * 16;                     // of the workgroup
  if (row_begin >= m) return;  // (the last chunk of several may be shorter)
  const int row_end = min((unit0 + kPsUnits - 1) / G * 16 + 16, m);
  int row0[CB], head[CB];      // of the column blocks: first row, head
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int unit = unit0 + CB * wave + cb;
    row0[cb] = unit / G * 16;
    head[cb] = kvh * G + unit % G;
  }

  const size_t head_at = chunk * a.stage_stride + (size_t)kvh * a.s_pad * kHeadDim;
  const int last_tile = a.s_pad / kPfKeys - 1;
  // (a tile past the staging area, asked for ahead and never used, is replaced by the last one)
  auto tile_at = [&](const uint16_t* base, int t) __attribute__((always_inline)) {
    return (const pf_bf16x8*)(base + head_at + (size_t)min(t, last_tile) * kPfTileElems);
  };
  // ---- queries: B operand, lane (qc, g4) holds dims [32 ks + 8 g4, +8) of its column block's row.
  // Their loads do not wait for the selection's length.
  const int S = min(max(a.sel_len[chunk], 0), a.max_sel_len);
  uint4 raw[CB][4];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const uint16_t* const row =
        a.q + (size_t)(first_row + min(row0[cb] + qc, m - 1)) * a.q_stride + head[cb] * kHeadDim + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) raw[cb][ks] = *(const uint4*)(row + 32 * ks);
  }
  // (behind the queries, which are wanted first: loads return in order)
  pf_bf16x8 kw[kPfOperands], vw[kPfOperands], k_second[kPfOperands];  // the operands of the next K tile and of the current V^T tile
  {
    const pf_bf16x8 *const k0 = tile_at(a.kr, 0), *const k1 = tile_at(a.kr, 1), *const v0 = tile_at(a.vt, 0);
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) kw[i] = k0[64 * i + lane];
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) k_second[i] = k1[64 * i + lane];
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) vw[i] = v0[64 * i + lane];
  }
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
      }
    };
    if (rope) rotation(row0[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      if (rope && row0[cb] != rotated) rotation(row0[cb]);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const uint32_t lw[4] = {raw[cb][ks].x, raw[cb][ks].y, raw[cb][ks].z, raw[cb][ks].w};
        const uint32_t hw[4] = {raw[cb][ks + 2].x, raw[cb][ks + 2].y, raw[cb][ks + 2].z, raw[cb][ks + 2].w};
        uint32_t lp[4], hp[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float lo[2] = {bf16_lo(lw[w]), bf16_hi(lw[w])}, hi[2] = {bf16_lo(hw[w]), bf16_hi(hw[w])};
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            if (rope) {
              const float s = sn[ks][2 * w + x], c = cs[ks][2 * w + x];
              const float l2 = lo[x] * c - hi[x] * s;
              hi[x] = hi[x] * c + lo[x] * s;
              lo[x] = l2;
            }
            lo[x] *= qs;
            hi[x] *= qs;
          }
          lp[w] = pack_bf16(lo[0], lo[1]);
          hp[w] = pack_bf16(hi[0], hi[1]);
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
  const int n_tiles = S > 0 && last_visible >= 0 ? last_visible / kPfKeys + 1 : 0;
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

  // The software pipeline of the other kernel.  Package t, what the operands' registers are refilled with in
  // iteration t, is the K tile t + 2 and the V^T tile t + 1: sixteen kilobytes, of which a wavefront asks
  // for four, straight to LDS, in iteration t - 2 (L2 takes 0.6 to 0.85 us, an iteration 0.65), buffer t % 4.
  // Before the barrier in the second half of iteration t a wavefront waits until its part of package t + 1
  // has come, which leaves that of package t + 2 under way, and until all but its last eight
  // reads of LDS are through.  The buffer that is asked for in iteration t had package t - 2: its reads
  // were issued in iteration t - 2 and, everybody's, through at the barrier of iteration t - 1.
  constexpr uint32_t kBytes = kPsPackage * 16, kPart = kBytes / 2 / kPsWaves;
  const int64_t tiles_bytes = (int64_t)a.s_pad * kHeadDim * 2 - kPart * wave;
  const ps_buffer ask_k = buffer_of(a.kr + head_at + 2 * kPfTileElems + kPart / 2 * wave, tiles_bytes - 2 * 2 * kPfTileElems);
  const ps_buffer ask_v = buffer_of(a.vt + head_at + kPfTileElems + kPart / 2 * wave, tiles_bytes - 2 * kPfTileElems);
  uint32_t ask_at = 0;  // of the next package to be asked for, in the staging area
  const uint32_t lane16 = 16 * lane, part_at = kPart * wave;
  auto ask_keys = [&](uint32_t buffer) __attribute__((always_inline)) { load_to_lds(part_at + buffer, ask_k, ask_at, lane16); };
  auto ask_values = [&](uint32_t buffer) __attribute__((always_inline)) {
    load_to_lds(part_at + buffer + kBytes / 2, ask_v, ask_at, lane16);
    ask_at += 2 * kPfTileElems;
  };

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

  if (n_tiles > 0) {
    pf_f32x4 s_even[CB][2], s_odd[CB][2];  // the logits of the even and of the odd tiles: [column block][key block]
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      ask_keys(t * kBytes);
      ask_values(t * kBytes);
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
      if (masked <= 0) mask(0, s_even[cb], cb);
      raise(s_even[cb], cb);
    }
    raise_any = bound();
    // (the compiler waits for the operands here, and not in every iteration for what may be the first's)
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) asm volatile("" : "+v"(kw[i]), "+v"(vw[i]));
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    using Yes = std::true_type;
    using No = std::false_type;
    int t = 0;
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
    // What was asked for past the end comes before the space may be another workgroup's.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // The length of a dense chunk, whose gather is through (nothing here reads it).
  if (a.new_len && blockIdx.x == 0 && blockIdx.z == 0 && blockIdx.y + 1 == gridDim.y && threadIdx.x == 0)
    *a.new_len = min(*a.new_len + m, a.len_cap);
  // o[cb][db][r] = O[query qc][dim 16 db + 4 g4 + r]; the row sum is complete in every lane.
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int row = row0[cb] + qc;
    if (row >= m) continue;
    const float l = row_sum[cb][0], inv = l > 0.f ? 1.0f / l : 0.f;
    uint16_t* const to = a.out + ((size_t)(first_row + row) * a.num_heads + head[cb]) * kHeadDim + 4 * g4;
#pragma unroll
    for (int db = 0; db < 8; ++db)
      *(uint2*)(to + 16 * db) = make_uint2(pack_bf16(o[cb][db][0] * inv, o[cb][db][1] * inv),
                                           pack_bf16(o[cb][db][2] * inv, o[cb][db][3] * inv));
  }
}

int64_t prefill_shared_workgroups(int num_heads, int num_kv_heads, int chunk_rows) {
  return ceil_div(ceil_div(chunk_rows, 16) * (num_heads / num_kv_heads), kPsUnits) * num_kv_heads;
}

int launch_prefill_shared(const PrefillArgs& a, int chunks, hipStream_t stream) {
  const int64_t per_head = prefill_shared_workgroups(a.num_heads, a.num_kv_heads, a.chunk_rows) / a.num_kv_heads;
  const dim3 grid((unsigned)a.num_kv_heads, (unsigned)per_head, (unsigned)chunks);
  const auto kernel = a.logit_cap > 0.f ? prefill_shared_kernel<true> : prefill_shared_kernel<false>;
  static const hipError_t ok[2] = {
      hipFuncSetAttribute((const void*)prefill_shared_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPsLdsBytes),
      hipFuncSetAttribute((const void*)prefill_shared_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPsLdsBytes)};
  if (ok[0] != hipSuccess || ok[1] != hipSuccess)
    return fail(TS_EHIP, "prefill attention: %zu bytes of LDS refused", kPsLdsBytes);
  hipLaunchKernelGGL(kernel, grid, dim3(kPsThreads), kPsLdsBytes, stream, a);
  return check_launch("prefill_shared_kernel");
}

}  // namespace ts
