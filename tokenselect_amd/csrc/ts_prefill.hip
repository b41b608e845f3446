// Chunked prefill (patched_radix_attention_extend_forward_flashinfer, tr.py:703-775):
// the fingerprint of a chunk (mean of its rotated query rows, tr.py:380-392) and the
// causal attention of the chunk's rows over the selected KV slots (FlashInfer paged
// prefill, tr.py:759-771, page size 1, in-kernel Llama RoPE).
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "ts_prefill.h"
#include "ts_store.h"

// ts_prefill_chunks.hip is this file's attention once more, for chunks that each have keys of their own, and nothing else
// of it.

namespace ts {

#ifndef TS_PREFILL_CHUNKS
// ------------------------------------------------------------------ fingerprint
// Four workgroups per head (16 rotation pairs each), 512 threads = 4 quads of pairs
// x 128 row groups, so that a chunk of 512 rows is one step of four independent rows
// per thread (the kernel is bound by the latency of its loads).  Row r
// is rotated with table row first_pos + r exactly like the rotation kernel (every
// product and sum rounded on its own, result rounded to bf16, tr.py:104-107); the
// bf16 values are summed in fp32, row group by row group in a fixed order, divided
// by the row count and rounded to bf16 (torch.mean on a bf16 tensor, tr.py:392).
constexpr int kFpRowGroups = 128;
constexpr int kFpInFlight = 4;  // rows per step of a row group
constexpr int kFpVec = 4;       // rotation pairs per thread
constexpr int kFpSplit = 4;     // workgroups per head
constexpr int kFpClear = 16;    // workgroups that clear
constexpr int kFpHeads = 2;     // heads of a workgroup where chunks are taken together
constexpr int kFpThreads = kHeadDim / 2 / kFpSplit / kFpVec * kFpRowGroups;

// Heads [h0, h0 + NH) below `heads`, the quarter's rotation pairs, of one chunk of `rows` rows: the tables' rows are
// read once for all of them.
template <int NH>
__device__ __forceinline__ void fingerprint_quarter(
    const uint16_t* __restrict__ q, int q_stride, uint16_t* __restrict__ qf, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int64_t table_rows, int first_pos, int rows, int heads, int h0, int quarter) {
#pragma clang fp contract(off)
  constexpr int half = kHeadDim / 2;
  constexpr int kPairs = half / kFpSplit;   // rotation pairs of this workgroup
  constexpr int kLanes = kPairs / kFpVec;   // threads per row
  static_assert(kFpThreads == kLanes * kFpRowGroups && kFpThreads == 2 * kPairs * kFpRowGroups / 8,
                "a thread per row group and four pairs, and per eight row groups and column");
  const int first_pair = quarter * kPairs;
  const int i = first_pair + (threadIdx.x % kLanes) * kFpVec, rg = threadIdx.x / kLanes;
  float lo_sum[NH][kFpVec] = {}, hi_sum[NH][kFpVec] = {};
  // Four rows per step: their loads are independent and go out together; the sums
  // are still taken in row order.
  for (int r0 = rg; r0 < rows; r0 += kFpInFlight * kFpRowGroups) {
    uint2 x1[NH][kFpInFlight], x2[NH][kFpInFlight];
    float4 c1[kFpInFlight], c2[kFpInFlight], s1[kFpInFlight], s2[kFpInFlight];
#pragma unroll
    for (int j = 0; j < kFpInFlight; ++j) {
      const int r = min(r0 + j * kFpRowGroups, rows - 1);
      int64_t pos = (int64_t)first_pos + r;
      pos = pos < table_rows ? pos : table_rows - 1;
      const float* c = cos_table + pos * kHeadDim;
      const float* s = sin_table + pos * kHeadDim;
#pragma unroll
      for (int x = 0; x < NH; ++x) {
        const size_t base = (size_t)r * q_stride + (NH == 1 ? h0 : min(h0 + x, heads - 1)) * kHeadDim;
        x1[x][j] = *(const uint2*)(q + base + i);
        x2[x][j] = *(const uint2*)(q + base + i + half);
      }
      c1[j] = *(const float4*)(c + i);
      c2[j] = *(const float4*)(c + i + half);
      s1[j] = *(const float4*)(s + i);
      s2[j] = *(const float4*)(s + i + half);
    }
#pragma unroll
    for (int j = 0; j < kFpInFlight; ++j) {
      if (r0 + j * kFpRowGroups < rows) {
        const float cc1[kFpVec] = {c1[j].x, c1[j].y, c1[j].z, c1[j].w};
        const float cc2[kFpVec] = {c2[j].x, c2[j].y, c2[j].z, c2[j].w};
        const float ss1[kFpVec] = {s1[j].x, s1[j].y, s1[j].z, s1[j].w};
        const float ss2[kFpVec] = {s2[j].x, s2[j].y, s2[j].z, s2[j].w};
#pragma unroll
        for (int x = 0; x < NH; ++x) {
          const uint2 y1 = x1[x][j], y2 = x2[x][j];
          const float a1[kFpVec] = {bf16_to_f32((uint16_t)y1.x), bf16_to_f32((uint16_t)(y1.x >> 16)),
                                    bf16_to_f32((uint16_t)y1.y), bf16_to_f32((uint16_t)(y1.y >> 16))};
          const float a2[kFpVec] = {bf16_to_f32((uint16_t)y2.x), bf16_to_f32((uint16_t)(y2.x >> 16)),
                                    bf16_to_f32((uint16_t)y2.y), bf16_to_f32((uint16_t)(y2.y >> 16))};
#pragma unroll
          for (int e = 0; e < kFpVec; ++e) {
            const float lo = a1[e] * cc1[e] + (-a2[e]) * ss1[e];
            const float hi = a2[e] * cc2[e] + a1[e] * ss2[e];
            const uint32_t rounded = pack_bf16(lo, hi);  // (a NaN stays one, and is one in the mean)
            lo_sum[x][e] += bf16_lo(rounded);
            hi_sum[x][e] += bf16_hi(rounded);
          }
        }
      }
    }
  }
  // Columns of this workgroup: its kPairs low halves, then its kPairs high halves.
  // The row groups are added in order, eight at a time and then the sixteen eights.
  // (A head's sums are written again two heads on: by then everybody has read them.)
  constexpr int kBuffers = NH > 1 ? 2 : 1;
  __shared__ float part[kBuffers][kFpRowGroups][2 * kPairs];
  __shared__ float part8[NH][kFpRowGroups / 8][2 * kPairs];
  const int col = i - first_pair;
#pragma unroll
  for (int x = 0; x < NH; ++x) {
#pragma unroll
    for (int e = 0; e < kFpVec; ++e) {
      part[x % kBuffers][rg][col + e] = lo_sum[x][e];
      part[x % kBuffers][rg][col + e + kPairs] = hi_sum[x][e];
    }
    __syncthreads();
    const int c = threadIdx.x % (2 * kPairs), set = threadIdx.x / (2 * kPairs);
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) sum += part[x % kBuffers][set * 8 + g][c];
    part8[x][set][c] = sum;
  }
  __syncthreads();
  if (threadIdx.x < NH * 2 * kPairs) {
    const int x = threadIdx.x / (2 * kPairs), c = threadIdx.x % (2 * kPairs);
    float total = 0.f;
    for (int g = 0; g < kFpRowGroups / 8; ++g) total += part8[x][g][c];
    const int dim = c < kPairs ? first_pair + c : half + first_pair + (c - kPairs);
    if (NH == 1 || h0 + x < heads) qf[(size_t)(h0 + x) * kHeadDim + dim] = f32_to_bf16(total / (float)rows);
  }
}

__global__ __launch_bounds__(kFpThreads) void fingerprint_kernel(
    const uint16_t* __restrict__ q, int q_stride, uint16_t* __restrict__ qf, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int64_t table_rows, int first_pos, int rows, int heads,
    ZeroSet zero, ChunkStore cs) {
  // On the side: the workgroups past the fingerprint's own store the chunk's K/V rows (the
  // caller's store of the chunk, which the selection after this launch must find done, riding here
  // instead of in a launch of its own), and the last kFpClear of them clear the words that the
  // selection counts into.
  if ((int)blockIdx.y >= kFpSplit) {
    const int wg = ((int)blockIdx.y - kFpSplit) * (int)gridDim.x + (int)blockIdx.x;
    const int stores = cs.k != nullptr ? cs.workgroups : 0;
    if (wg < stores)
      store_chunk_rows<true>(cs, wg, kFpThreads);
    else if (wg < stores + kFpClear)
      clear_regions(zero, (uint32_t)(wg - stores) * (kFpThreads / 64) + (threadIdx.x >> 6),
                    kFpClear * (kFpThreads / 64));
    return;
  }
  fingerprint_quarter<1>(q, q_stride, qf, cos_table, sin_table, table_rows, first_pos, rows, heads, (int)blockIdx.x,
                         (int)blockIdx.y);
}

// The same for several chunks of a prompt: the store of their rows (whose positions follow from the length before
// the first chunk, which the launch after this one advances), the words their selections count into and their
// lengths, by the first workgroups, cs.workgroups + 1 per chunk; then the fingerprints, two heads of a chunk to
// a workgroup, their quarters eight workgroups apart: on one XCD, whose L2 has the lines of the queries
// that they share.  With a workgroup per head and quarter the tables were four times the queries, and the two bf16
// roundings of a pair eleven instructions instead of one: 19 chunks of 28 heads 46.8 -> 38.8 us, 6 of 32 20.8 ->
// 19.1, 3 of 32 12.5 -> 11.6 (the rows alone, read and stored, are 110 MB of the first: 22 us).  Four heads, whose
// registers leave one workgroup to a CU, 59.
__global__ __launch_bounds__(kFpThreads) void prompt_fingerprint_kernel(
    const uint16_t* __restrict__ q, int q_stride, uint16_t* __restrict__ qf, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int64_t table_rows, int first_pos, int heads, PromptChunks pc, ChunkStore cs) {
  const int on_the_side = pc.chunks * (cs.workgroups + 1);
  if ((int)blockIdx.x < on_the_side) {
    const int chunk = (int)blockIdx.x / (cs.workgroups + 1), wg = (int)blockIdx.x % (cs.workgroups + 1);
    const int first = chunk * pc.chunk_rows, rows = min(pc.chunk_rows, pc.rows - first);
    const int len = *cs.seq_len;
    if (wg < cs.workgroups) {
      store_rows_at(cs, len, first + wg * (kFpThreads / kChunkThreadsPerRow) + (int)threadIdx.x / kChunkThreadsPerRow,
                    first + rows);
    } else {
      uint32_t* const counters = pc.counters + (size_t)chunk * pc.counters_stride;
      for (int w = threadIdx.x; w < pc.counter_words; w += kFpThreads) counters[w] = 0u;
      if (threadIdx.x == 0) pc.lens[chunk] = min(len + first + rows, cs.max_tokens);
    }
    return;
  }
  const int id = (int)blockIdx.x - on_the_side, per_chunk = (heads + kFpHeads - 1) / kFpHeads;
  const int unit = id / (8 * kFpSplit) * 8 + id % 8, quarter = id / 8 % kFpSplit;
  if (unit >= pc.chunks * per_chunk) return;
  const int chunk = unit / per_chunk, first = chunk * pc.chunk_rows;
  fingerprint_quarter<kFpHeads>(q + (size_t)first * q_stride, q_stride, qf + (size_t)chunk * heads * kHeadDim, cos_table,
                          sin_table, table_rows, first_pos, min(pc.chunk_rows, pc.rows - first), heads,
                          unit % per_chunk * kFpHeads, quarter);
}

#endif  // TS_PREFILL_CHUNKS

// ------------------------------------------------------------ prefill attention
// Two launches.
//
// prefill_gather_kernel: the selected rows are gathered once per chunk into a
// contiguous staging area, K rotated to its index in the selected list (in fp32,
// rounded to bf16 like the queries) and V transposed, so that the attention kernel, whose
// query tiles would otherwise each repeat the gather, the rotation and the transposition,
// only loads operands: per KV head and tile of 32 keys kr and vt hold the eight A operands
// of the tile one after the other, 1 KB each, 16 bytes per lane in lane order.  The keys of
// a V^T operand are in the order in which the logits' product leaves them (kv_pos below).
//
// prefill_attn_kernel<G>: grid (KV heads, query tiles, head blocks x chunks); 256 threads = four
// wavefronts, one per SIMD, each a key group of its own: group g takes the 32-key tiles
// g, g + 4, g + 8, ... for all 64 query columns of the workgroup (kPfBlocks column blocks of
// 16 query rows of one head: four heads x 16 rows, two x 32 or one x 64, whatever divides G
// with the least waste), held in registers.  The four groups' (max, sum, acc) are merged
// through LDS at the end, a column block per wavefront.
//
// Why one wavefront per SIMD with 64 columns: every K and V^T operand that a wavefront
// fetches feeds four matrix instructions, and nobody shares its tiles, so that they go from
// L2 straight into the operand registers.  With two wavefronts per SIMD of 32 columns the
// tiles went through LDS (written once, read by two wavefronts): 192 KB of LDS traffic per
// round and counters in LDS to hand buffers over, which a wavefront, issuing in order,
// waited for.  The staging area is laid out so that an operand is 1 KB in a row, lane l's 16
// bytes at 16 l; an operand's registers are refilled for the next tile as soon as its last
// product is issued, so that a load has a whole round (some 1400 cycles) to arrive.
//
// A wavefront computes S^T = K Q^T with v_mfma_f32_16x16x32_bf16 (A = 16 keys x 32 dims,
// B = 16 rotated queries of one head, pre-multiplied by the softmax scale and log2 e), which
// leaves lane (query l%16, key group l/16) with base-2 logits of 8 keys of the tile.  The
// accumulator starts at minus the running maximum of the row, so the products come out
// already shifted; the running maximum is only raised when a logit exceeds it by more than 8
// (the weights then stay below 2^8, harmless in fp32 sums and invisible after the final
// division), so the common path per logit is one maximum, one exp2 and half a conversion.
// The 8 probabilities, rounded to bf16, are directly the B operand of O^T += V^T P^T
// (A = 16 dims x 32 keys from the V^T tile); a ninth product with an all-ones A operand
// accumulates the row sums.  fp32 accumulation throughout.
//
// Measured, 512 rows over 2688 selected keys: 32 heads on 8 KV heads 37.3 -> 28.8 us, 28 on 4
// 32.8 -> 25.4 us (68 matrix instructions of 7 ns per tile: 10 us; the 1.4 MB of tiles per
// CU at the 110 GB/s that L2 delivers to one: 13 us).  What is left over is mostly the
// loads' latency: 64 KB per CU in flight, 0.6 to 0.85 us from L2 under this load.
// Alternating products and exp2 in the source order of the logits' steps changed nothing.
// The merge area: per group and column block eight vectors of accumulators and (max, sum),
// four floats per lane each.  (The rotated queries pass through the same space at the start.)
constexpr size_t kPfLdsBytes = (size_t)kPfGroups * kPfBlocks * 9 * 64 * 16;  // 144 KB

#ifndef TS_PREFILL_CHUNKS
constexpr int kPfVRow = kPfKeys + 8;   // halfwords per V^T row in the gather kernel's LDS (80 B)

// Position of key kk (0..31 within its block) in a V^T row: the matrix instruction
// that made the logits left lane group g4 with keys 16 kb + 4 g4 + r (kb < 2, r < 4),
// and the next one wants those 8 as one 16-byte operand, in the order 4 kb + r.
__device__ __forceinline__ int kv_pos(int kk) { return 8 * ((kk >> 2) & 3) + 4 * (kk >> 4) + (kk & 3); }

// 16 bytes of the staging area.  With eight KV heads the workgroup that gathers a head's keys runs
// on the XCD whose workgroups attend to them (the KV head is the fastest index of both grids), and
// what it leaves in that XCD's L2 is read from there.  With fewer, several XCDs read a head, most of
// what is written waits in the wrong L2, and the writes go past it.  Gather + attention, us: 28 heads
// on 4 7.75 + 24.8 with the tile as the fastest index, 6.6 + 24.6 with the head, 5.6 + 24.8 past the
// L2 as well; 32 on 8 7.4 + 27.4, 6.5 + 27.6, 6.7 + 28.3.  A prompt of 31600 tokens, 28 heads on 4:
// 3675 us kept, 3651 past the L2.  On two heads and on one (whose keys are a quarter and an eighth) it is the
// same either way: 28.6 and 27.0 us for both launches, prompts of 12000 tokens 1250 and 1198.
typedef __attribute__((ext_vector_type(4))) unsigned int pf_u32x4;
__device__ __forceinline__ void stage(const PrefillArgs& a, void* to, const uint4& w) {
  if (a.num_kv_heads < 8)
    __builtin_nontemporal_store(__builtin_bit_cast(pf_u32x4, w), (pf_u32x4*)to);
  else
    *(uint4*)to = w;
}

// Grid (32-key tiles x KV heads, the head fastest; all on x: the device reports 65536 as the end of y, 2.1 M keys),
// by chunks.
// Thread (key kk, chunk c) moves dims [8c, 8c+8) and
// [64+8c, +8) of key j = tile + kk.  Keys past S are written as zeros.
// DENSE (PrefillDense): key j is position j, its slot the table's or, from the length on, one of the
// chunk's new rows, which is read where the caller has it and stored on the way.  A dense chunk was
// a store that also wrote the list (4.6 us and a gap), this (5.4) and the attention; this is 6.2 now: three
// prompts of 700 to 5200 tokens and 8 tokens 2475 -> 2400 us a pass.
// MANY: chunk blockIdx.y of several.  One chunk leaves out what finds its own.
template <bool DENSE, bool MANY>
__device__ __forceinline__ void gather_tile(const PrefillArgs& a, const PrefillDense& dense) {
  __shared__ __attribute__((aligned(16))) uint16_t vt_lds[kHeadDim * kPfVRow];
  const int tid = threadIdx.x;
  const int kk = tid >> 3, c8 = tid & 7;
  const int head_bits = __builtin_ctz((unsigned)a.num_kv_heads);  // (1, 2, 4 or 8 of them)
  const int kvh = blockIdx.x & (a.num_kv_heads - 1);
  const uint32_t tile = blockIdx.x >> head_bits, tiles = gridDim.x >> head_bits;
  const int j = tile * kPfKeys + kk;
  const int chunk = MANY ? (int)blockIdx.y : 0;
  // (the slot is asked for together with the length, not after it)
  uint32_t slot;
  if (DENSE) {
    const PrefillDense& d = dense;
    slot = ((uint32_t)d.table[min(j, d.list_bound - 1) >> d.page_shift] << d.page_shift) +
           (uint32_t)(j & ((1 << d.page_shift) - 1));
  } else {
    slot = (uint32_t)a.sel[chunk * a.sel_stride + min(j, a.max_sel_len - 1)];
  }
  const int len = DENSE ? *dense.seq_len : 0;
  const bool appends = DENSE && dense.store.k != nullptr;
  const int end = appends ? min(len + dense.store.rows, dense.store.max_tokens) : len;  // of what is stored
  const int S = DENSE ? min(max(end, 0), dense.list_bound) : min(max(a.sel_len[chunk], 0), a.max_sel_len);
  const int row = j - len;  // of the chunk
  const bool fresh = appends && len >= 0 && row >= 0 && j < end;
  // A row of the chunk to its slot (clamped to the pool, as ts_kv_store_chunk does).
  auto chunk_slot = [&](int r) {
    const int64_t at = dense.store.loc[r];
    return (uint32_t)(at < 0 ? 0 : at >= (int64_t)a.pool_rows ? (int64_t)a.pool_rows - 1 : at);
  };
  auto chunk_piece = [&](const uint4* rows, int r, int half) {
    return rows[(size_t)r * dense.store.kv_stride + kvh * (kHeadDim / 8) + c8 + 8 * half];
  };
  auto store_piece = [&](uint32_t to, int half, const uint4& k, const uint4& v) {
    const size_t at = ((size_t)to * a.num_kv_heads + kvh) * (kHeadDim / 8) + c8 + 8 * half;
    dense.store.k_pool[at] = k;
    dense.store.v_pool[at] = v;
  };
  if (DENSE) {
    // Rows past the tiles (a bound below the length is the caller's error, but they are stored).
    if (appends && len >= 0 && tile + 1 == tiles)
      for (int at = max((int)tiles * kPfKeys, len) + kk; at < end; at += kPfKeys) {
        const uint32_t to = chunk_slot(at - len);
        for (int half = 0; half < 2; ++half)
          store_piece(to, half, chunk_piece(dense.store.k, at - len, half), chunk_piece(dense.store.v, at - len, half));
        if (kvh == 0 && c8 == 0) dense.store.table[at] = (int32_t)to;
      }
    if (kvh == 0 && j == 0 && c8 == 0) *dense.sel_len = S;
    slot = fresh ? chunk_slot(row) : min(slot, a.pool_rows - 1);
    if (kvh == 0 && c8 == 0) {
      if (j < S) {
        dense.sel_pos[j] = j;
        dense.sel[j] = (int32_t)slot;
      }
      if (fresh) dense.store.table[j] = (int32_t)slot;
    }
  }
  // Whole blocks of kPfPadKeys: the keys between S and the next multiple are written as
  // zeros too (their weights are zero, but 0 x garbage is not).
  if (tile * kPfKeys >= (S + kPfPadKeys - 1) / kPfPadKeys * kPfPadKeys && !(DENSE && tile * kPfKeys < (unsigned)max(end, 0)))
    return;
  const bool live = j < S;
  uint4 kraw[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
  uint4 vraw[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
  if (fresh) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      kraw[half] = chunk_piece(dense.store.k, row, half);
      vraw[half] = chunk_piece(dense.store.v, row, half);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      store_piece(slot, half, kraw[half], vraw[half]);
      if (!live) kraw[half] = vraw[half] = make_uint4(0, 0, 0, 0);
    }
  } else if (live) {
    slot = slot < a.pool_rows ? slot : a.pool_rows - 1;
    const size_t at = ((size_t)slot * a.num_kv_heads + kvh) * kHeadDim + 8 * c8;
    kraw[0] = *(const uint4*)(a.k_pool + at);
    kraw[1] = *(const uint4*)(a.k_pool + at + 64);
    vraw[0] = *(const uint4*)(a.v_pool + at);
    vraw[1] = *(const uint4*)(a.v_pool + at + 64);
  }
  const uint32_t klo[4] = {kraw[0].x, kraw[0].y, kraw[0].z, kraw[0].w};
  const uint32_t khi[4] = {kraw[1].x, kraw[1].y, kraw[1].z, kraw[1].w};
  float lo[8], hi[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    lo[2 * e] = bf16_lo(klo[e]);
    lo[2 * e + 1] = bf16_hi(klo[e]);
    hi[2 * e] = bf16_lo(khi[e]);
    hi[2 * e + 1] = bf16_hi(khi[e]);
  }
  if (a.rope_mode == TS_ROPE_LLAMA) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int pair = 8 * c8 + e;
      const float freq = a.rope_rcp_scale * exp2f(-(float)pair * (2.0f / kHeadDim) * a.log2_theta);
      float sn, cs;
      sincos_reduced((float)j * freq, sn, cs);
      // (which product is rounded is said here: both forms of the gather give the same keys)
      const float l2 = fmaf(lo[e], cs, -(hi[e] * sn));
      hi[e] = fmaf(hi[e], cs, lo[e] * sn);
      lo[e] = l2;
    }
  }
  // key kk = 16 kb + qc, dims 32 ks + 8 g4: operand 4 kb + ks, lane 16 g4 + qc
  const size_t tile_at = chunk * a.stage_stride + ((size_t)kvh * a.s_pad + (size_t)tile * kPfKeys) * kHeadDim;
  uint16_t* kout = a.kr + tile_at + ((4 * (kk >> 4) + (c8 >> 2)) * 64 + 16 * (c8 & 3) + (kk & 15)) * 8;
  stage(a, kout, make_uint4(pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(lo[4], lo[5]),
                            pack_bf16(lo[6], lo[7])));
  stage(a, kout + 2 * 64 * 8, make_uint4(pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3]),
                                         pack_bf16(hi[4], hi[5]), pack_bf16(hi[6], hi[7])));
  // transpose the 32 x 128 V tile through LDS (key kk to column kv_pos(kk)), then write its
  // eight operands: piece p is lane p % 64 of operand p / 64, dim 16 (p / 64) + p % 16,
  // columns [8 g4, +8) with g4 = p % 64 / 16
  const uint32_t vlo[4] = {vraw[0].x, vraw[0].y, vraw[0].z, vraw[0].w};
  const uint32_t vhi[4] = {vraw[1].x, vraw[1].y, vraw[1].z, vraw[1].w};
  const int col = kv_pos(kk);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    vt_lds[(8 * c8 + 2 * e) * kPfVRow + col] = (uint16_t)(vlo[e] & 0xffffu);
    vt_lds[(8 * c8 + 2 * e + 1) * kPfVRow + col] = (uint16_t)(vlo[e] >> 16);
    vt_lds[(64 + 8 * c8 + 2 * e) * kPfVRow + col] = (uint16_t)(vhi[e] & 0xffffu);
    vt_lds[(64 + 8 * c8 + 2 * e + 1) * kPfVRow + col] = (uint16_t)(vhi[e] >> 16);
  }
  __syncthreads();
  uint4* vout = (uint4*)(a.vt + tile_at);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 256 * i;
    stage(a, vout + p, *(const uint4*)(vt_lds + (16 * (p >> 6) + (p & 15)) * kPfVRow + 8 * ((p >> 4) & 3)));
  }
}
// The tickets of the attention's jobs that are cut (PrefillCuts), if there are any.
__device__ __forceinline__ void clear_tickets(uint32_t* tickets) {
  if (tickets && blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < kPsTicketBytes / 4; i += 256) tickets[i] = 0u;
}
template <bool MANY>
__global__ __launch_bounds__(256) void prefill_gather_kernel(PrefillArgs a, uint32_t* tickets) {
  clear_tickets(tickets);
  gather_tile<false, MANY>(a, PrefillDense{});
}
__global__ __launch_bounds__(256) void prefill_gather_dense_kernel(PrefillArgs a, PrefillDense dense, uint32_t* tickets) {
  clear_tickets(tickets);
  gather_tile<true, false>(a, dense);
}

#endif  // TS_PREFILL_CHUNKS

// Heads of a workgroup's column blocks; the kPfBlocks / heads blocks of a head are
// consecutive query tiles.  The choice that leaves the fewest columns of the last head block
// without a head, and of those the one with the most heads (which share a row's rotation).
constexpr int prefill_heads(int group) { return group % 4 == 0 || group % 4 == 3 ? 4 : group % 2 == 0 ? 2 : 1; }

// One wavefront per SIMD by construction (four per workgroup, one workgroup per CU by its
// LDS): saying so lets the compiler use all 512 registers.
// MANY: a chunk of several, which the workgroup finds first.  One chunk leaves that out: 512 rows behind 131072
// tokens 25.8 us with it, 25.3 without (with both in one kernel, chosen by its arguments, 25.5, and two or three
// chunks of a prompt half a microsecond more).
template <int G, bool CAP, bool MANY>
__global__ __launch_bounds__(64 * kPfGroups) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_attn_kernel(
    PrefillArgs a) {
  constexpr int CB = kPfBlocks;
  constexpr int NH = prefill_heads(G);   // heads of the workgroup
  constexpr int RT = CB / NH;            // query tiles of 16 rows
  constexpr int kRows = 16 * RT;
  constexpr int kHeadBlocks = (G + NH - 1) / NH;
  // Column block cb: head cb % NH of the workgroup's, query tile cb / NH.
  extern __shared__ __attribute__((aligned(16))) uint16_t pf_lds[];
  const int group = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // wavefront = key group
  const int lane = threadIdx.x & 63;
  const int qc = lane & 15, g4 = lane >> 4;  // query column / key group of the matrix layouts
  // The KV head is the fastest-moving workgroup index: consecutive workgroups go to
  // consecutive XCDs, so with eight KV heads each XCD's L2 holds the keys and values of one
  // head (1.4 MB of 11 MB) and every query tile of that head finds them there.  The last
  // query tiles, which see the most keys, start first.
  const int kvh = blockIdx.x;
  const int q_row0 = (int)(gridDim.y - 1 - blockIdx.y) * kRows;
  const int H = a.num_heads;
  const int chunk = MANY ? (int)blockIdx.z / kHeadBlocks : 0;
  const int head_block = (int)blockIdx.z - chunk * kHeadBlocks;
  const int first_row = chunk * a.chunk_rows;
  const int m = MANY ? min(a.chunk_rows, a.rows - first_row) : a.rows;
  if (MANY && q_row0 >= m) return;  // (the last chunk of several may be shorter)
  auto head_in_group = [&](int cb) { return head_block * NH + cb % NH; };
  auto head_of = [&](int cb) { return kvh * G + min(head_in_group(cb), G - 1); };
  auto row_of = [&](int cb) { return q_row0 + 16 * (cb / NH) + qc; };

  // Tile t of this group holds the keys [(t kPfGroups + group) kPfKeys, + kPfKeys).  A tile
  // past the staging area (asked for ahead, never used) is replaced by the last one.
  const uint16_t* const k_base = a.kr + chunk * a.stage_stride + (size_t)kvh * a.s_pad * kHeadDim;
  const uint16_t* const v_base = a.vt + chunk * a.stage_stride + (size_t)kvh * a.s_pad * kHeadDim;
  const int last_tile = a.s_pad / kPfKeys - 1;
  auto tile_at = [&](const uint16_t* base, int t) __attribute__((always_inline)) {
    return (const uint4*)(base + (size_t)min(t * kPfGroups + group, last_tile) * kPfTileElems);
  };
  uint4 kw[kPfOperands], vw[kPfOperands];  // the operands of the next K tile and of the current V^T tile
  {
    const uint4* const k0 = tile_at(k_base, 0);
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) kw[i] = k0[64 * i + lane];
  }

  // ---- queries: B operand, lane (qc, g4) holds dims [32 ks + 8 g4, +8) of its column block's
  // row, rotated to position shift + row (partner dims d and d + 64 are k-steps ks and ks + 2).
  // All wavefronts need all of them; each prepares a quarter, four dims of every eight of one
  // k-step and their partners, and they meet in LDS.
  // The queries' loads do not wait for the selection's length.
  const int my_ks = group >> 1, my_half = 4 * (group & 1);
  uint2 q_raw[CB][2];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const uint16_t* qrow = a.q + (size_t)(first_row + min(row_of(cb), m - 1)) * a.q_stride + head_of(cb) * kHeadDim +
                           32 * my_ks + 8 * g4 + my_half;
    q_raw[cb][0] = *(const uint2*)qrow;
    q_raw[cb][1] = *(const uint2*)(qrow + 64);
  }
  const int S = min(max(a.sel_len[chunk], 0), a.max_sel_len);
  // The length of a dense chunk, whose gather is through (nothing here reads it), by one of the
  // workgroups of the first rows, which see the fewest keys.
  auto commit_length = [&]() {
    if (a.new_len && blockIdx.x == 0 && blockIdx.z == 0 && blockIdx.y + 1 == gridDim.y && threadIdx.x == 0)
      *a.new_len = min(*a.new_len + m, a.len_cap);
  };
  const int shift = S - m;  // query row i sits at position shift + i and sees keys <= that
  if (S <= 0) {
    // No keys (a selection that reported a fault): the rows attend to nothing and the
    // output is defined as zero.  (With fewer keys than rows, 0 < S < m, the rows whose
    // position S - m + i is negative see no key either: every tile is masked for them,
    // their sums stay zero and so does their output; the others attend as usual.)
    const int cb = group;  // a column block per wavefront
    if (head_in_group(cb) < G)
      for (int i = lane; i < 16 * (kHeadDim / 8); i += 64) {
        const int row = q_row0 + 16 * (cb / NH) + i / (kHeadDim / 8);
        if (row < m)
          *(uint4*)(a.out + ((size_t)(first_row + row) * H + head_of(cb)) * kHeadDim + 8 * (i % (kHeadDim / 8))) =
              make_uint4(0u, 0u, 0u, 0u);
      }
    commit_length();
    return;
  }
  {
    const bool rope = a.rope_mode == TS_ROPE_LLAMA;
    // Without a soft cap the softmax scale and log2(e) go into the query, so that the
    // products come out as base-2 logits and every key costs one exp2 and no multiply.
    const float qs = CAP ? 1.0f : a.sm_scale * kLog2e;
    float freq[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int pair = 32 * my_ks + 8 * g4 + my_half + e;
      freq[e] = a.rope_rcp_scale * exp2f(-(float)pair * (2.0f / kHeadDim) * a.log2_theta);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float sn[4], cs[4];
      if (rope) {
        const float pos = (float)(shift + min(q_row0 + 16 * rt + qc, m - 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) sincos_reduced(pos * freq[e], sn[e], cs[e]);
      }
#pragma unroll
      for (int hh = 0; hh < NH; ++hh) {
        const int cb = rt * NH + hh;
        float lo[4] = {bf16_lo(q_raw[cb][0].x), bf16_hi(q_raw[cb][0].x), bf16_lo(q_raw[cb][0].y),
                       bf16_hi(q_raw[cb][0].y)};
        float hi[4] = {bf16_lo(q_raw[cb][1].x), bf16_hi(q_raw[cb][1].x), bf16_lo(q_raw[cb][1].y),
                       bf16_hi(q_raw[cb][1].y)};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (rope) {
            const float l2 = lo[e] * cs[e] - hi[e] * sn[e];
            hi[e] = hi[e] * cs[e] + lo[e] * sn[e];
            lo[e] = l2;
          }
          lo[e] *= qs;
          hi[e] *= qs;
        }
        uint16_t* const to = pf_lds + ((cb * 4 + my_ks) * 64 + lane) * 8 + my_half;
        *(uint2*)to = make_uint2(pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]));
        *(uint2*)(to + 2 * 64 * 8) = make_uint2(pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3]));
      }
    }
  }
  __syncthreads();
  pf_bf16x8 qb[CB][4];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qb[cb][ks] = __builtin_bit_cast(pf_bf16x8, *(const uint4*)(pf_lds + ((cb * 4 + ks) * 64 + lane) * 8));
      keep_acc(qb[cb][ks]);
    }
  __syncthreads();  // (the space is the merge area from here on)

  // ---- main loop over the tiles any row of this workgroup can see
  const int last_visible = min(S - 1, shift + min(q_row0 + kRows - 1, m - 1));
  // tiles of this group that hold a visible key
  const int n_tiles = last_visible >= group * kPfKeys
                          ? (last_visible - group * kPfKeys) / (kPfGroups * kPfKeys) + 1
                          : 0;
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

  // The loop is a software pipeline, because a wavefront issues in order and the matrix unit
  // and the vector ALU only run side by side when their instructions alternate in one stream.
  // Iteration t:
  //   logits(t + 1): S^T = K_{t+1} Q^T (32 matrix instructions in eight steps, one per K
  //                  operand), shifted by the running maximum through the accumulators' start
  //                  values; in between, a step's share of the exp2 of tile t, and the
  //                  operand's registers are filled with tile t + 2's;
  //   output(t):     O^T += V_t^T P^T and the row sums (36 matrix instructions); in between the
  //                  largest logit of each row of tile t + 1, and the V^T operands of tile t + 1
  //                  are asked for;
  //   settle(t + 1): when a row outgrew its maximum by kPfRaise, the move to a new one.
  // Only the last tile of a group can hold keys that some row must not see (a group's tiles
  // are 128 keys apart, and a workgroup has at most 64 rows): the mask is on that one alone.
  pf_f32x4 s_cur[CB][2];  // logits of the tile whose output comes next: [column block][key block]

  // The soft cap, and the mask of the last tile; the largest logit of the lane's eight.
  auto largest = [&](int t, pf_f32x4 (&s)[2], int cb, bool last) __attribute__((always_inline)) {
    if (CAP) {
      const float shift_by = m_run[cb] == kNegBig ? 0.f : m_run[cb];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[kb][r] = a.logit_cap * tanhf(s[kb][r] * a.sm_scale / a.logit_cap) * kLog2e - shift_by;
    }
    if (last) {
      // Masked logits are -inf: exp2 makes them 0 without a branch.
      const int limit = shift + min(row_of(cb), m - 1) - ((t * kPfGroups + group) * kPfKeys + 4 * g4);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * kb + r > limit) s[kb][r] = -INFINITY;
    }
    float mx = max3(s[0][0], s[0][1], s[0][2]);
    mx = max3(mx, s[0][3], s[1][0]);
    mx = max3(mx, s[1][1], s[1][2]);
    return fmaxf(mx, s[1][3]);
  };
  auto settle = [&](pf_f32x4 (&s)[CB][2], const float (&mx_lane)[CB]) __attribute__((always_inline)) {
    bool any = false;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) any = any || mx_lane[cb] > raise_at[cb];
    if (__ballot(any) == 0ull) return;
    // Some row has no maximum yet, or outgrew it: agree on the row's maximum over the four
    // key groups of lanes and move to it.  (All column blocks, and one vector at a time: a
    // row that stays where it is is multiplied by one, and a branch per block or more
    // vectors at once would cost the loop around this its registers.)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const bool unset = m_run[cb] == kNegBig;
      float mx = mx_lane[cb];
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const bool take = mx > raise_at[cb];
      const float delta = take ? mx : 0.f;
      // (a row without a maximum has only zeros in its accumulators)
      const float scale = unset ? 1.0f : __builtin_amdgcn_exp2f(-delta);
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
        for (int r = 0; r < 4; ++r) s[cb][kb][r] -= delta;
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
  };

  // NEXT: there is a tile t + 1; LAST: that one is the group's last.
  auto iteration = [&](int t, auto next, auto last) __attribute__((always_inline)) {
    constexpr bool NEXT = decltype(next)::value, LAST = decltype(last)::value;
    const uint4* const k2 = tile_at(k_base, t + 2);
    const uint4* const v1 = tile_at(v_base, t + 1);
    pf_f32x4 s_next[CB][2];
    uint32_t pw[CB][4];
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) {
      const int kb = i >> 2, ks = i & 3;
      // this step's share of the weights: column block i / 2, key block i % 2
      const int pcb = i >> 1, pkb = i & 1;
      float p[4];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        if (NEXT) s_next[cb][kb] = mfma_logits(ks == 0 ? minus_m[cb] : s_next[cb][kb], kw[i], qb[cb][ks]);
        p[cb] = __builtin_amdgcn_exp2f(s_cur[pcb][pkb][cb]);
      }
      if (NEXT && !LAST) kw[i] = k2[64 * i + lane];
      pw[pcb][2 * pkb] = pack_bf16(p[0], p[1]);
      pw[pcb][2 * pkb + 1] = pack_bf16(p[2], p[3]);
      if (NEXT) {  // in the order: product, exp2, product, exp2, ...
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // matrix
          __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);  // transcendental
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    pf_bf16x8 pb[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
      pb[cb] = __builtin_bit_cast(pf_bf16x8, make_uint4(pw[cb][0], pw[cb][1], pw[cb][2], pw[cb][3]));
    packed_settled(pb);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
      row_sum[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[cb], row_sum[cb], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    float mx[CB];
#pragma unroll
    for (int db = 0; db < 8; ++db) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) mfma_acc(o[cb][db], __builtin_bit_cast(pf_bf16x8, vw[db]), pb[cb]);
      if (NEXT) {
        vw[db] = v1[64 * db + lane];
        if (db >= 3 && db < 3 + CB) mx[db - 3] = largest(t + 1, s_next[db - 3], db - 3, LAST);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    mfma_settled(o);
    __builtin_amdgcn_sched_barrier(0);
    if (NEXT) {
      settle(s_next, mx);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        s_cur[cb][0] = s_next[cb][0];
        s_cur[cb][1] = s_next[cb][1];
      }
    }
  };

  if (n_tiles > 0) {
    // the first tile's logits: nothing comes before them
    const uint4* const k1 = tile_at(k_base, 1);
    const uint4* const v0 = tile_at(v_base, 0);
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        s_cur[cb][i >> 2] = mfma_logits((i & 3) == 0 ? minus_m[cb] : s_cur[cb][i >> 2], kw[i], qb[cb][i & 3]);
      kw[i] = k1[64 * i + lane];
      __builtin_amdgcn_sched_barrier(0);
    }
    // (after the second K tile, in the order of the loop: loads return in order, and at the
    // loop's head the compiler waits for the later of the two orders it may have come from)
#pragma unroll
    for (int i = 0; i < kPfOperands; ++i) vw[i] = v0[64 * i + lane];
    __builtin_amdgcn_sched_barrier(0);
    float mx[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) mx[cb] = largest(0, s_cur[cb], cb, n_tiles == 1);
    settle(s_cur, mx);
    for (int t = 0; t + 2 < n_tiles; ++t) iteration(t, std::true_type{}, std::false_type{});
    if (n_tiles > 1) iteration(n_tiles - 2, std::true_type{}, std::true_type{});
    iteration(n_tiles - 1, std::false_type{}, std::false_type{});
  }

  // ---- merge of the four key groups: every wavefront hands all its column blocks over (per
  // lane 8 vectors of acc and one of (max, sum)) and merges one of them.
  pf_f32x4* const merge = (pf_f32x4*)pf_lds;  // [group][column block][9][64 lanes]
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    pf_f32x4* const mine = merge + (group * CB + cb) * (9 * 64) + lane;
#pragma unroll
    for (int db = 0; db < 8; ++db) mine[db * 64] = o[cb][db];
    mine[8 * 64] = pf_f32x4{m_run[cb], row_sum[cb][0], 0.f, 0.f};
  }
  __syncthreads();
  static_assert(CB == kPfGroups, "a column block per wavefront");
  const int cb = group;
  const pf_f32x4* const all = merge + cb * (9 * 64) + lane;
  pf_f32x4 ml = all[8 * 64];
  float m_all = ml[0], l_all = ml[1];
  pf_f32x4 sum[8];
#pragma unroll
  for (int db = 0; db < 8; ++db) sum[db] = all[db * 64];
#pragma unroll
  for (int g = 1; g < kPfGroups; ++g) {
    const pf_f32x4* const other = all + g * CB * (9 * 64);
    ml = other[8 * 64];
    const float m_new = fmaxf(m_all, ml[0]);
    const float e0 = __builtin_amdgcn_exp2f(m_all - m_new), e1 = __builtin_amdgcn_exp2f(ml[0] - m_new);
    m_all = m_new;
    // (which product is rounded is said here: the compiler chooses by what is around, and a chunk's bits with it)
    l_all = fmaf(l_all, e0, ml[1] * e1);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const pf_f32x4 od = other[db * 64];
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[db][r] = fmaf(od[r], e1, sum[db][r] * e0);
    }
  }

  commit_length();
  // sum[db][r] = O[query qc][dim 16 db + 4 g4 + r]; the row sum is complete in every lane.
  const int row = row_of(cb);
  if (row >= m || head_in_group(cb) >= G) return;
  const float inv = l_all > 0.f ? 1.0f / l_all : 0.f;
  uint16_t* orow = a.out + ((size_t)(first_row + row) * H + head_of(cb)) * kHeadDim;
#pragma unroll
  for (int db = 0; db < 8; ++db)
    *(uint2*)(orow + 16 * db + 4 * g4) = make_uint2(pack_bf16(sum[db][0] * inv, sum[db][1] * inv),
                                                    pack_bf16(sum[db][2] * inv, sum[db][3] * inv));
}

template <bool MANY>
static int launch_attention(const PrefillArgs& a, int chunks, hipStream_t stream) {
  const int group = a.num_heads / a.num_kv_heads, heads = prefill_heads(group);
  const dim3 grid((unsigned)a.num_kv_heads, (unsigned)ceil_div(std::min(a.chunk_rows, a.rows), 16 * (kPfBlocks / heads)),
                  (unsigned)(ceil_div(group, heads) * chunks));
  const bool cap = a.logit_cap > 0.f;
#define TS_PF_LAUNCH(G_, C_)                                                                        \
  {                                                                                                 \
    static const hipError_t lds_ok = hipFuncSetAttribute(                                           \
        (const void*)prefill_attn_kernel<G_, C_, MANY>, hipFuncAttributeMaxDynamicSharedMemorySize, \
        (int)kPfLdsBytes);                                                                          \
    if (lds_ok != hipSuccess) return fail(TS_EHIP, "prefill attention: %zu bytes of LDS refused", kPfLdsBytes); \
    hipLaunchKernelGGL((prefill_attn_kernel<G_, C_, MANY>), grid, dim3(64 * kPfGroups), kPfLdsBytes, stream, a); \
  }
#define TS_PF_CASE(G_)               \
  case G_:                           \
    if (cap) TS_PF_LAUNCH(G_, true)  \
    else TS_PF_LAUNCH(G_, false)     \
    break;
  switch (group) {
    TS_PF_CASE(1)
    TS_PF_CASE(2)
    TS_PF_CASE(3)
    TS_PF_CASE(4)
    TS_PF_CASE(5)
    TS_PF_CASE(6)
    TS_PF_CASE(7)
    TS_PF_CASE(8)
    default: return fail(TS_ESHAPE, "unsupported head group %d", group);
  }
#undef TS_PF_CASE
#undef TS_PF_LAUNCH
  return check_launch("prefill_attn_kernel");
}

#ifdef TS_PREFILL_CHUNKS
int launch_prefill_several(const PrefillArgs& a, int chunks, hipStream_t stream) {
  return launch_attention<true>(a, chunks, stream);
}
#else
int check_fingerprint(const void* q, int32_t rows, const float* cos_table, const float* sin_table,
                      int64_t table_rows, const void* qf, int32_t n_local) {
  TS_REQUIRE(q && cos_table && sin_table && qf, TS_EINVAL, "ts_fingerprint: NULL tensor argument");
  TS_REQUIRE_ALIGNED(q, 16, "q");
  TS_REQUIRE_ALIGNED(cos_table, 16, "cos_table");
  TS_REQUIRE_ALIGNED(sin_table, 16, "sin_table");
  TS_REQUIRE(rows >= 1, TS_EINVAL, "ts_fingerprint: rows %d < 1", rows);
  TS_REQUIRE(table_rows >= (int64_t)n_local + rows, TS_EINVAL,
             "ts_fingerprint: cos/sin tables have %lld rows, need n_local + rows = %lld",
             (long long)table_rows, (long long)n_local + rows);
  return TS_OK;
}

int launch_fingerprint(const ts_config* cfg, const void* q, int q_stride, int32_t rows, const float* cos_table,
                       const float* sin_table, int64_t table_rows, void* qf, const ZeroSet& zero,
                       hipStream_t stream, const ChunkStore* store) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(!zero.overflow, TS_EINVAL, "internal: more than %d regions to clear in one launch", kZeroRegions);
  TS_TRY(check_fingerprint(q, rows, cos_table, sin_table, table_rows, qf, cfg->n_local));
  ChunkStore cs{};
  if (store) {  // 32 threads per row
    cs = *store;
    cs.workgroups = (int)ceil_div(cs.rows, kFpThreads / kChunkThreadsPerRow);
    TS_REQUIRE(cs.workgroups <= kChunkCountedWgs && cs.max_tokens <= kLenMask, TS_EINVAL,
               "internal: a chunk store of %d rows does not ride in the fingerprint launch", cs.rows);
  }
  const unsigned grid_y =
      kFpSplit + (unsigned)ceil_div(cs.workgroups + (zero.used ? kFpClear : 0), cfg->num_heads);
  hipLaunchKernelGGL(fingerprint_kernel, dim3((unsigned)cfg->num_heads, grid_y), dim3(kFpThreads), 0, stream,
                     (const uint16_t*)q, q_stride, (uint16_t*)qf, cos_table, sin_table, table_rows,
                     cfg->n_local, rows, cfg->num_heads, zero, cs);
  return check_launch("fingerprint_kernel");
}

int launch_prompt_fingerprint(const ts_config* cfg, const void* q, int q_stride, const float* cos_table,
                              const float* sin_table, int64_t table_rows, void* qf, const PromptChunks& pc,
                              const ChunkStore& store, hipStream_t stream) {
  TS_TRY(check_fingerprint(q, pc.chunk_rows, cos_table, sin_table, table_rows, qf, cfg->n_local));
  ChunkStore cs = store;
  cs.workgroups = (int)ceil_div(pc.chunk_rows, kFpThreads / kChunkThreadsPerRow);
  const int64_t units = ceil_div(cfg->num_heads, kFpHeads) * pc.chunks;
  const dim3 grid((unsigned)(pc.chunks * (int64_t)(cs.workgroups + 1) + ceil_div(units, 8) * 8 * kFpSplit));
  hipLaunchKernelGGL(prompt_fingerprint_kernel, grid, dim3(kFpThreads), 0, stream, (const uint16_t*)q, q_stride,
                     (uint16_t*)qf, cos_table, sin_table, table_rows, cfg->n_local, cfg->num_heads, pc, cs);
  return check_launch("prompt_fingerprint_kernel");
}

// Chunks, from the first on, whose attention takes the workgroups of 256 columns where no job is cut: for a workspace
// without room for the pieces, or jobs too few.  A wave of those over the device, a workgroup per CU, takes 68 us for 2688 keys, and one
// of the workgroups of 64 columns 20 where all of them read the same 1.4 MB per head, 26 where each chunk has its own: so they get all
// chunks where their last wave is at least 0.8 full, else as many as fill whole waves.  us for a whole call of chunks of 512 rows in
// workgroups of 64 columns, with whole waves, and with all: 28 heads on 4, two chunks (0.44 waves) 106, 106 and 125, four
// (0.88) 152, 152 and 132, nine (1.97) 285, 269 and 224, 18 (3.94) 530, 447 and 402.  The line is that of a loop that took 75 us;
// with this one it would lie at some 0.6 (three chunks, 0.66, 130, 130 and 128, eight, 1.75, 264, 247 and 219; 32 on 8, six,
// 1.5, 219, 206 and 211), of use only to who has no room for pieces: jobs are cut from 0.59 waves on.  The rows of a long dense chunk see
// fewer keys the earlier they are, and the early ones fill the last wave up: 28 heads on 4, 2048 rows (0.88) 66 and 66, 2336 (1) 83 and
// 73, 2688 (1.16) 96 and 83.
static int shared_chunks(int num_heads, int num_kv_heads, int rows, int chunk_rows) {
  const int64_t each = prefill_shared_workgroups(num_heads, num_kv_heads, chunk_rows), chunks = ceil_div(rows, chunk_rows);
  // (small chunks would leave most of a workgroup without columns)
  if (4 * chunk_rows * (int64_t)num_heads < 3 * each * 256) return 0;
  const int64_t full = each * chunks / 256, rest = each * chunks - full * 256;
  if (rest >= 205 || rest == 0 || (chunks == 1 && each >= 256)) return (int)chunks;
  return (int)(full * 256 / each);
}

// Whether the workgroups of 256 columns take all rows, with jobs that are cut: one long dense chunk by what it would take
// either way (prefill_dense_cuts_pay), several chunks from 0.59 waves of jobs on.  us for a whole call, in workgroups of 64 columns
// and so: two full chunks of 28 heads (0.44) 95 and 96, of 32 (0.5) 99 and 103; 1436 rows in chunks of 512 of 28 heads (0.61) 117 and 110, of 32
// (0.7) 124 and 122, 1948 of 24 on 8 (0.72) 149 and 125.  And from 1024 keys on: the start of a piece costs ten tiles of 32.
bool prefill_cuts_pay(int num_heads, int num_kv_heads, int rows, int chunk_rows, int keys) {
  if (keys < 1024) return false;
  const PrefillCuts c = prefill_cuts(num_heads, num_kv_heads, rows, chunk_rows, 1, nullptr);
  // (small chunks would leave most of a workgroup without columns)
  if (4 * (int64_t)std::min(rows, chunk_rows) * num_heads < 3 * (int64_t)c.per_chunk * num_kv_heads * 256) return false;
  if (c.chunks == 1) return prefill_dense_cuts_pay(num_heads, num_kv_heads, rows, keys);
  return c.jobs * num_kv_heads >= 152;
}

static int prefill_s_pad(int max_sel_len) { return (int)ceil_div(max_sel_len, kPfPadKeys) * kPfPadKeys; }

int launch_prefill_attn(const ts_config* cfg, const void* q, int q_stride, int32_t rows, const void* k_pool,
                        const void* v_pool, int64_t pool_rows, const int32_t* sel, const int32_t* sel_len,
                        int32_t max_sel_len, void* out, void* workspace, size_t workspace_bytes,
                        hipStream_t stream, const PrefillDense* dense, void* cut_space) {
  return launch_prefill_attn_chunks(cfg, q, q_stride, rows, rows, k_pool, v_pool, pool_rows, sel, 0, sel_len,
                                    max_sel_len, out, workspace, workspace_bytes, stream, dense, cut_space);
}

int launch_prefill_attn_chunks(const ts_config* cfg, const void* q, int q_stride, int32_t rows, int32_t chunk_rows,
                               const void* k_pool, const void* v_pool, int64_t pool_rows, const int32_t* sel,
                               int64_t sel_stride, const int32_t* sel_len, int32_t max_sel_len, void* out,
                               void* workspace, size_t workspace_bytes, hipStream_t stream,
                               const PrefillDense* dense, void* cut_space) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(q && k_pool && v_pool && sel && sel_len && out, TS_EINVAL,
             "ts_sparse_prefill_attn: NULL tensor argument");
  TS_REQUIRE(rows >= 1 && rows <= 65535 * 16, TS_EINVAL, "rows %d out of range", rows);
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  const unsigned chunks = (unsigned)ceil_div(rows, chunk_rows);
  const size_t per_chunk = ts_prefill_attn_workspace_bytes(cfg, max_sel_len), need = chunks * per_chunk;
  TS_REQUIRE(workspace != nullptr && workspace_bytes >= need, TS_EWORKSPACE,
             "ts_sparse_prefill_attn: workspace %zu bytes < required %zu", workspace_bytes, need);
  TS_REQUIRE_ALIGNED(workspace, 256, "workspace");
  TS_REQUIRE_ALIGNED(q, 16, "q");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(v_pool, 16, "v_pool");
  TS_REQUIRE_ALIGNED(out, 16, "out");
  PrefillArgs a;
  a.q = (const uint16_t*)q;
  a.q_stride = q_stride;
  a.k_pool = (const uint16_t*)k_pool;
  a.v_pool = (const uint16_t*)v_pool;
  a.pool_rows = (uint32_t)pool_rows;
  a.sel = sel;
  a.sel_len = sel_len;
  a.max_sel_len = max_sel_len;
  a.s_pad = prefill_s_pad(max_sel_len);
  a.rows = rows;
  a.chunk_rows = chunk_rows;
  a.sel_stride = sel_stride;
  a.stage_stride = per_chunk / 2;  // (a chunk's kr, then its vt: bytes to elements, twice as far apart)
  a.num_heads = cfg->num_heads;
  a.num_kv_heads = cfg->num_kv_heads;
  a.rope_mode = cfg->rope_mode;
  a.log2_theta = cfg->rope_mode == TS_ROPE_LLAMA ? (float)log2((double)cfg->rope_theta) : 0.f;
  a.rope_rcp_scale = cfg->rope_mode == TS_ROPE_LLAMA ? 1.0f / cfg->rope_scale : 1.0f;
  a.sm_scale = cfg->sm_scale;
  a.logit_cap = cfg->logit_cap;
  a.kr = (uint16_t*)workspace;
  a.vt = (uint16_t*)((char*)workspace + per_chunk / 2);
  a.out = (uint16_t*)out;
  a.new_len = dense && dense->store.k ? dense->seq_len : nullptr;
  a.len_cap = dense ? dense->store.max_tokens : 0;
  hipStream_t st = stream;
  const dim3 gather_grid((unsigned)cfg->num_kv_heads * (unsigned)(a.s_pad / kPfKeys), chunks);
  const bool cut = cut_space != nullptr && prefill_cuts_pay(cfg->num_heads, cfg->num_kv_heads, rows, chunk_rows, max_sel_len);
  const int together = cut ? (int)chunks : shared_chunks(cfg->num_heads, cfg->num_kv_heads, rows, chunk_rows);
  PrefillArgs first = a;
  first.rows = (int)std::min<int64_t>(rows, (int64_t)together * chunk_rows);
  PrefillCuts cuts{};
  if (together > 0)
    cuts = prefill_cuts(cfg->num_heads, cfg->num_kv_heads, first.rows, chunk_rows, max_sel_len, cut ? cut_space : nullptr);
  if (dense)
    hipLaunchKernelGGL(prefill_gather_dense_kernel, gather_grid, dim3(256), 0, st, a, *dense, cuts.tickets);
  else
    hipLaunchKernelGGL(chunks > 1 ? prefill_gather_kernel<true> : prefill_gather_kernel<false>, gather_grid, dim3(256), 0,
                       st, a, cuts.tickets);
  TS_TRY(check_launch("prefill_gather_kernel"));
  if (together > 0) {
    TS_TRY(launch_prefill_shared(first, cuts, st));
    if (together == (int)chunks) return TS_OK;
    a.q += (size_t)first.rows * q_stride;
    a.out += (size_t)first.rows * cfg->num_heads * kHeadDim;
    a.sel_len += together;
    a.kr += together * a.stage_stride;
    a.vt += together * a.stage_stride;
    a.rows -= first.rows;
  }
  return together < (int)chunks - 1 ? launch_prefill_several(a, (int)chunks - together, st)
                                    : launch_attention<false>(a, 1, st);
}
#endif  // TS_PREFILL_CHUNKS

}  // namespace ts

#ifndef TS_PREFILL_CHUNKS
using namespace ts;

extern "C" {

int ts_fingerprint(const ts_config* cfg, const void* q, int32_t rows, const float* cos_table,
                   const float* sin_table, int64_t table_rows, void* qf, ts_stream_t stream) {
  return launch_fingerprint(cfg, q, cfg ? cfg->num_heads * cfg->head_dim : 0, rows, cos_table, sin_table, table_rows, qf, ZeroSet{},
                            (hipStream_t)stream);
}

size_t ts_prefill_attn_workspace_bytes(const ts_config* cfg, int32_t max_sel_len) {
  if (validate_config(cfg) != TS_OK || max_sel_len < 1) return 0;
  return 2 * align_up((size_t)cfg->num_kv_heads * prefill_s_pad(max_sel_len) * kHeadDim * 2, 256);
}

int ts_sparse_prefill_attn(const ts_config* cfg, const void* q, int32_t rows, const void* k_pool,
                           const void* v_pool, int64_t pool_rows, const int32_t* sel,
                           const int32_t* sel_len, int32_t max_sel_len, void* out, void* workspace,
                           size_t workspace_bytes, ts_stream_t stream) {
  return launch_prefill_attn(cfg, q, cfg ? cfg->num_heads * cfg->head_dim : 0, rows, k_pool, v_pool, pool_rows, sel,
                             sel_len, max_sel_len, out, workspace, workspace_bytes, (hipStream_t)stream);
}

}  // extern "C"
#endif  // TS_PREFILL_CHUNKS
