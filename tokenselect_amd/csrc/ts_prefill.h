// What the prefill's kernels share: their arguments, the staging area's layout, and the products of the attention.
#pragma once

#include <type_traits>

#include "ts_common.h"

namespace ts {

struct PrefillArgs {
  const uint16_t* q;  // [rows, H, 128] bf16, un-rotated, rows q_stride elements apart
  int q_stride;
  const uint16_t* k_pool;
  const uint16_t* v_pool;
  uint32_t pool_rows;
  const int32_t* sel;      // [chunk][S] selected slots in attention order
  const int32_t* sel_len;  // [chunk] S
  int max_sel_len;
  int s_pad;               // keys in kr and vt per KV head: max_sel_len rounded up to kPfPadKeys
  int rows;                // of all chunks
  int chunk_rows;          // of a chunk (the last one may have fewer): a selection for each of them
  int64_t sel_stride;      // entries between the chunks' lists
  size_t stage_stride;     // elements between their parts of kr, and of vt
  int32_t* new_len;        // the length that the attention advances by `rows`, up to len_cap, or NULL
  int len_cap;
  int num_heads, num_kv_heads, rope_mode;
  float log2_theta, rope_rcp_scale, sm_scale, logit_cap;
  uint16_t* kr;   // [Hkv, s_pad / 32, operand 4 kb + ks, lane, 8] bf16 rotated keys
  uint16_t* vt;   // [Hkv, s_pad / 32, operand db, lane, 8] bf16 transposed values
  uint16_t* out;  // [rows, H, 128] bf16
};

typedef __attribute__((ext_vector_type(8))) __bf16 pf_bf16x8;
typedef __attribute__((ext_vector_type(4))) float pf_f32x4;
constexpr float kLog2e = 1.4426950408889634f;

constexpr int kPfKeys = 32;            // keys per tile: of the gather kernel and of the attention kernel
constexpr int kPfPadKeys = 64;         // the staging area holds whole multiples of this many keys
constexpr int kPfGroups = 4;           // key groups of an attention workgroup: its wavefronts
constexpr int kPfBlocks = 4;           // column blocks (16 query rows of one head) of a wavefront
constexpr int kPfTileElems = kPfKeys * kHeadDim;      // a K tile; a V^T tile is as large
constexpr int kPfOperands = kPfTileElems / (64 * 8);  // operands of a tile: 16 bytes per lane each
static_assert(kPfOperands == 8, "a tile has eight operands");
constexpr float kPfRaise = 8.0f;       // a row's maximum is raised when a logit exceeds it by this much

// Largest of three, without the NaN-quieting copies fmaxf brings along.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

// The products, with their registers in the half of the register file that suits them: the
// accumulators of the output and the queries in the accumulation registers, the logits,
// which vector instructions read, in the others.  Written as assembly because the compiler,
// left to choose, moves accumulators to and fro around every product (480 moves per tile).
// What it does not see it does not keep apart: between a product and any use of its result other
// than as the same product's next accumulator there must be eight instructions' issue, and two
// between a vector instruction and a product that reads its result.  The two fences below make
// that order a dependency of the values themselves; tests/test_prefill_hazards_cpu.py looks
// through the compiler's listing for what register copies could still have put in between.
__device__ __forceinline__ void mfma_acc(pf_f32x4& acc, const pf_bf16x8& a, const pf_bf16x8& b) {
  asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ pf_f32x4 mfma_logits(const pf_f32x4& s, const uint4& k, const pf_bf16x8& q) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pf_bf16x8, k), q, s, 0, 0, 0);
}
// Says that acc lives in the accumulation registers here, so that where paths join it stays there.
template <typename V>
__device__ __forceinline__ void keep_acc(V& acc) { asm("" : "+a"(acc)); }
// The accumulators behind this are those before it, sixteen idle instructions later: no use of
// one can come before the idling, and no product that makes one after it.
template <int CB>
__device__ __forceinline__ void mfma_settled(pf_f32x4 (&o)[CB][8]) {
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int db = 0; db < 8; ++db) asm volatile("" : "+a"(o[cb][db]));
  asm volatile("s_nop 15" ::: "memory");
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int db = 0; db < 8; ++db) asm volatile("" : "+a"(o[cb][db]));
}
// The weights behind this are those before it, two idle instructions later.
__device__ __forceinline__ void packed_settled(pf_bf16x8 (&pb)[4]) {
  asm("s_nop 1" : "+v"(pb[0]), "+v"(pb[1]), "+v"(pb[2]), "+v"(pb[3]));
}
__device__ __forceinline__ void weights_settled(pf_bf16x8& p) { asm("s_nop 1" : "+v"(p)); }

// The attention over a staging area that has been filled, in workgroups of 256 columns, and how many of
// them a chunk is (ts_prefill_shared.hip).
int64_t prefill_shared_workgroups(int num_heads, int num_kv_heads, int chunk_rows);
// Their jobs, per KV head: a workgroup each for the first `whole`, and the others shared out evenly between
// `streams` workgroups, by what they cost, so that a share may begin and end within a job.
struct PrefillCuts {
  int chunks, per_chunk, jobs;  // chunks, jobs of a chunk (the last one may have fewer), of all
  int whole, streams;
  int keys;                     // that the last row of a chunk sees, by the host's knowledge
  int quantum;                  // cost of a share
  uint32_t* tickets;            // zero at launch: of the jobs that are cut
  char* pieces;                 // and what there is of each
};
constexpr int kPsSlots = 256;   // workgroups that share jobs, of all KV heads: one per CU
constexpr int kPsTicketBytes = kPsSlots * 4 * 4;
// (without a workspace of prefill_cut_bytes() no job is cut)
PrefillCuts prefill_cuts(int num_heads, int num_kv_heads, int rows, int chunk_rows, int keys, void* workspace);
bool prefill_dense_cuts_pay(int num_heads, int num_kv_heads, int rows, int keys);
int launch_prefill_shared(const PrefillArgs& a, const PrefillCuts& cuts, hipStream_t stream);
// The same in workgroups of 64 columns, for several chunks (ts_prefill_chunks.hip).
int launch_prefill_several(const PrefillArgs& a, int chunks, hipStream_t stream);

}  // namespace ts
