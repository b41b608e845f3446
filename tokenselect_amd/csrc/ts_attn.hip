// Decode attention over the selected KV slots: the FlashInfer paged decode the
// reference calls at tr.py:815-823 (page size 1, in-kernel Llama RoPE).
//
// Split-K in one launch: grid (splits, Hkv, B).  A workgroup owns a contiguous range of
// the request's selected list for one KV head and all G = H/Hkv query heads that read it;
// its four wavefronts walk a quarter of the range each, in tiles of 32 tokens, on the
// matrix cores (see attn_kernel).  Keys are rotated to their index in the selected list,
// the query to S-1; softmax is online in fp32.  A dense decode step on a per-token or paged
// table is this one launch (AttnDense): the list is the table itself.  Partial (max, sum, acc) triples are merged
// across the wavefronts, written with device-coherent stores, and the workgroup that draws
// the last ticket of its (request, KV head) merges the splits and writes the bf16 output; or, in a layer without a selection
// cache, all of them merge a share each (attn_finish_shared).
#include <math.h>

#include <algorithm>

#include <mutex>
#include <type_traits>

#include "ts_common.h"

namespace ts {

constexpr int kAttnThreads = 64 * kAttnWaves;

struct AttnArgs {
  const uint16_t* q;  // [B,H,128] bf16, un-rotated, rows q_stride elements apart
  int q_stride;
  const uint16_t* k_pool;
  const uint16_t* v_pool;
  uint32_t pool_rows;
  const int32_t* sel;
  int64_t sel_stride;
  const int32_t* sel_len;
  int num_heads, num_kv_heads;
  int group;          // query heads per KV head
  int rope_mode;
  float log2_theta, rope_rcp_scale, sm_scale, logit_cap;
  int nsplit, max_sel_len;
  float* part_acc;    // [B,H,nsplit,128]
  float* part_ml;     // [B,H,nsplit,2]
  uint32_t* tickets;  // [B][Hkv + 1], zero at launch and again when the kernel ends
  uint16_t* out;      // [B,H,128] bf16
  ZeroSet zero;       // cleared on the side (counters of the stream's next selection)
  // A dense step (AttnDense): sel is the table, in pages of 1 << list_shift, sel_len the lengths;
  // list_bound: positions whose entries are there to be read.
  int list_shift, list_bound;
  AttnDense step;
  StepCommit commit;  // what the step's store left to be written (batch 0: nothing)
};
struct AttnSharedArgs : AttnArgs {
  AttnShare share;  // the splits merged by everybody
};

// The last three wavefronts' share of the regions to clear.
__device__ __forceinline__ void attn_clear_on_the_side(const AttnArgs& a) {
  if (a.zero.used == 0) return;
  const uint32_t wg = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  clear_regions(a.zero, wg * (kAttnWaves - 1) + wave - 1, gridDim.x * gridDim.y * gridDim.z * (kAttnWaves - 1));
}

__device__ __forceinline__ float2 load_coherent2(const float* p) {
  const uint64_t v =
      __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}
// (Plain stores, waited for before the ticket is drawn: exchanges whose old value is
// awaited, the faster way to publish a few words elsewhere, are slower for a
// workgroup's 2 KB of partials.)
__device__ __forceinline__ void store_coherent2(float* p, float x, float y) {
  const uint64_t v = (uint64_t)__float_as_uint(x) | ((uint64_t)__float_as_uint(y) << 32);
  __hip_atomic_store((uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The lengths, table entries and page count that a store within the selection left to be written
// (StepCommit), by one wavefront.  Nothing of this launch reads them.
__device__ __forceinline__ void attn_commit(const StepCommit& c) {
  const int b = threadIdx.x & 63;
  if (b >= c.batch) return;
  const int4 note = c.notes[b];
  if (note.x >= 0) {
    if (note.z >= 0) c.table[(int64_t)b * c.table_stride + note.y] = note.z;
    c.seq_lens[b] = note.x;
  }
  if (b == 0 && c.free_count) *c.free_count = max(*c.free_count, 0) - note.w;
}

__device__ __forceinline__ bool attn_appends(const AttnArgs& a, int slot, int len) {
  return a.step.loc != nullptr && append_fits(slot, len, a.pool_rows, a.step.max_tokens);
}

// What a dense step leaves behind besides the output, after a workgroup's share of the attention:
// the new token's row of this KV head in the pool (by the workgroup whose range holds it), the
// list (by the workgroups of the first KV head), and, by the last workgroup of the request's last
// KV head (`last`), when all of them have read the length, the table's entry and the length.
// Nobody waits for any of it in this launch: the new row was read where the caller has it.
__device__ __forceinline__ void attn_dense_epilogue(const AttnArgs& a, int b, int kvh, int lo, int hi, int S,
                                                    int slot, int len, bool ok, bool last) {
  const int tid = threadIdx.x;
  // (a host bound below the length is the caller's error, but the row is stored: the table lists it)
  if (ok && lo <= len && (len < hi || (int)blockIdx.x + 1 == a.nsplit) && tid < 2 * (kHeadDim / 8)) {
    const bool is_v = tid >= kHeadDim / 8;
    const int at = 8 * (tid % (kHeadDim / 8));
    const uint16_t* row = (is_v ? a.step.v : a.step.k) + (size_t)b * a.step.kv_stride + kvh * kHeadDim + at;
    uint16_t* to = (uint16_t*)(is_v ? a.v_pool : a.k_pool) + ((size_t)slot * a.num_kv_heads + kvh) * kHeadDim + at;
    *(uint4*)to = *(const uint4*)row;
  }
  if (kvh == 0) {
    const int32_t* tab = a.sel + (int64_t)b * a.sel_stride;
    int32_t* const sel = a.step.sel + (int64_t)b * a.step.sel_stride;
    int32_t* const sel_pos = a.step.sel_pos + (int64_t)b * a.step.sel_stride;
    for (int pos = lo + tid; pos < min(hi, S); pos += kAttnThreads) {
      const uint32_t entry = ((uint32_t)tab[min(pos, a.list_bound - 1) >> a.list_shift] << a.list_shift) +
                             (uint32_t)(pos & ((1 << a.list_shift) - 1));
      sel_pos[pos] = pos;
      sel[pos] = ok && pos == len ? slot : (int32_t)min(entry, a.pool_rows - 1);
    }
  }
  if (last && tid == 0) {
    uint32_t* const heads = a.tickets + (size_t)b * (a.num_kv_heads + 1) + a.num_kv_heads;
    if (__hip_atomic_fetch_add(heads, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
        (uint32_t)a.num_kv_heads) {
      __hip_atomic_store(heads, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      a.step.sel_len[b] = S;
      if (ok) {
        a.step.table[(int64_t)b * a.sel_stride + len] = slot;
        a.step.seq_lens[b] = len + 1;
      }
    }
  }
}

// The end of an attention workgroup: its four wavefronts' partial (max, sum, acc) triples
// of G head slots lie in LDS; they are merged, written with device-coherent stores, and the
// workgroup that draws the last ticket of its (request, KV head) merges the splits and
// writes the bf16 output.  Whether this was that workgroup.
template <int G>
__device__ __forceinline__ bool attn_finish(const AttnArgs& a, int b, int kvh, int split,
                                            float (*sm_acc)[G][kHeadDim], float (*sm_m)[G],
                                            float (*sm_l)[G], uint32_t* s_last_ptr) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int H = a.num_heads;
  auto head_of_slot = [&](int g) { return kvh * G + g; };
  uint32_t& s_last = *s_last_ptr;
  __syncthreads();
  // A thread owns two adjacent dims of one head: one 64-bit coherent store.
  for (int idx = tid; idx < G * (kHeadDim / 2); idx += kAttnThreads) {
    const int g = idx / (kHeadDim / 2), d = (idx % (kHeadDim / 2)) * 2;
    float mm = kNegBig;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) mm = fmaxf(mm, sm_m[w][g]);
    float o0 = 0.f, o1 = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      const float sc = __expf(sm_m[w][g] - mm);
      o0 += sm_acc[w][g][d] * sc;
      o1 += sm_acc[w][g][d + 1] * sc;
      ll += sm_l[w][g] * sc;
    }
    const size_t ph = ((size_t)b * H + head_of_slot(g)) * a.nsplit + split;
    store_coherent2(a.part_acc + ph * kHeadDim + d, o0, o1);
    if (d == 0) store_coherent2(a.part_ml + ph * 2, mm, ll);
  }

  // Ticket: the stores above are acknowledged before the workgroup is counted.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* ticket = a.tickets + (size_t)b * (a.num_kv_heads + 1) + kvh;
  if (tid == 0) {
    const uint32_t before =
        __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before + 1 == (uint32_t)a.nsplit ? 1u : 0u;
  } else if (tid >= 64) {
    // (While the ticket is drawn, not ahead of the first loads: 0.6 us of the 38 that a layer of a
    // 32K request takes, 2.0 of 98 with eight of 8K.)
    attn_clear_on_the_side(a);
    if (tid >= kAttnThreads - 64 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) attn_commit(a.commit);
  }
  __syncthreads();
  if (!s_last) return false;

  // out[b,h,:] = sum_s exp(m_s - M) acc_s / sum_s exp(m_s - M) l_s, rounded to bf16.
  // A wavefront per head slot (a thread owns two adjacent dims, and a head has 64 such
  // pairs): lane s fetches the (max, sum) of split s, so that the wave takes the maximum and
  // lane s the weight of its split while the accumulators, all requested at once, are on their
  // way, and they are added up with weights that are ready (read lane by lane): no chain of
  // dependent exponentials, and one statistics load per wave instead of one per split and thread.
  // With more than four head slots a wavefront has two of them, and works on both at once:
  // one after the other they would be two chains of loads (as they are behind a branch).
  static_assert(kHeadDim / 2 == 64, "one wavefront per head slot");
  constexpr int SLOTS = (G + kAttnWaves - 1) / kAttnWaves;  // head slots per wavefront
  const int wave_id = tid >> 6, d = lane * 2;
  size_t ph[SLOTS];
  float mm[SLOTS], ll[SLOTS], o0[SLOTS], o1[SLOTS];
#pragma unroll
  for (int it = 0; it < SLOTS; ++it) {
    // (a slot past the last head repeats the last one and is not written)
    ph[it] = ((size_t)b * H + head_of_slot(min(wave_id + kAttnWaves * it, G - 1))) * a.nsplit;
    mm[it] = kNegBig;
    ll[it] = o0[it] = o1[it] = 0.f;
  }
  // COUNT splits from s0 on, branch-free: loads past the last split repeat it and get the weight
  // zero.  As few as hold the launch's splits: this step takes what one CU needs to fetch their
  // accumulators, some 10 ns per load of 512 bytes.  With 32 loads for any number of splits it was 3
  // to 3.7 us of an attention of 10 to 11; now 0.8 us for 3 splits, 2.4 for 21.  (Wavefronts that share
  // a workgroup of eight, for half as many splits, share a SIMD: 2.5 us more for the tiles.)
  auto add_splits = [&](int s0, auto count_c) __attribute__((always_inline)) {
    constexpr int COUNT = decltype(count_c)::value;
    float2 ac[SLOTS][COUNT], ml[SLOTS];
#pragma unroll
    for (int it = 0; it < SLOTS; ++it) {
#pragma unroll
      for (int i = 0; i < COUNT; ++i)
        ac[it][i] = load_coherent2(a.part_acc + (ph[it] + min(s0 + i, a.nsplit - 1)) * kHeadDim + d);
      ml[it] = (lane < COUNT && s0 + lane < a.nsplit) ? load_coherent2(a.part_ml + (ph[it] + s0 + lane) * 2)
                                                      : make_float2(kNegBig, 0.f);
    }
#pragma unroll
    for (int it = 0; it < SLOTS; ++it) {
      float mx = ml[it].x;
      mx = fmaxf(mx, dpp_move<kRowRor8>(mx));
      mx = fmaxf(mx, dpp_move<kRowRor4>(mx));
      mx = fmaxf(mx, dpp_move<kRowRor2>(mx));
      mx = fmaxf(mx, dpp_move<kRowRor1>(mx));
      if (COUNT > 16) mx = fmaxf(mx, __shfl_xor(mx, 16));
      const float mn = fmaxf(mm[it], __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mx))));
      const float keep = __expf(mm[it] - mn);  // what earlier batches hold
      const float w = (lane < COUNT && s0 + lane < a.nsplit) ? __expf(ml[it].x - mn) : 0.f;
      const float wl = ml[it].y * w;
      o0[it] *= keep;
      o1[it] *= keep;
      ll[it] *= keep;
      mm[it] = mn;
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i));
        ll[it] += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), i));
        o0[it] += ac[it][i].x * wi;
        o1[it] += ac[it][i].y * wi;
      }
    }
  };
  if (a.nsplit <= 4)
    add_splits(0, std::integral_constant<int, 4>{});
  else if (a.nsplit <= 8)
    add_splits(0, std::integral_constant<int, 8>{});
  else if (a.nsplit <= 16)
    add_splits(0, std::integral_constant<int, 16>{});
  else
    for (int s0 = 0; s0 < a.nsplit; s0 += 24) add_splits(s0, std::integral_constant<int, 24>{});
#pragma unroll
  for (int it = 0; it < SLOTS; ++it) {
    const int g = wave_id + kAttnWaves * it;
    if (g < G) {
      const uint32_t packed = (uint32_t)f32_to_bf16(ll[it] > 0.f ? o0[it] / ll[it] : 0.f) |
                              ((uint32_t)f32_to_bf16(ll[it] > 0.f ? o1[it] / ll[it] : 0.f) << 16);
      *(uint32_t*)(a.out + ((size_t)b * H + head_of_slot(g)) * kHeadDim + d) = packed;
    }
  }
  if (tid == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// The end of a workgroup where the splits are merged by everybody (AttnShare): each sends its partial sums as
// words that are not zero, so that each word is its own flag, and then merges, of one head, the columns that are its
// own share: it asks for them until they have come.  A word has one reader, who leaves it zero again for the next
// launch.  In place of the acknowledgement of the partials, the ticket and one workgroup that fetches the partials of all
// there is the time that the last words take.  In-kernel clock, one request, us after the first workgroup's start: 32 heads
// on 8, tiles done 5.3, partials sent 6.2, then ticket 7.3 (the last 8.3) and end 10.2, or all words seen 7.4 (8.0) and end
// 8.5.  28 on 4: as before end 10.6; and since more splits cost the merge nothing now, with 64 entries each tiles done 3.9
// in place of 5.2, sent 5.0, seen 6.4, end 7.4.
// Nothing of a word is lost: the bits are sent inverted, and the one pattern that would be zero, two NaN that no
// computation makes, as its neighbour.
__device__ __forceinline__ uint64_t share_word(float x, float y) {
  const uint64_t w = ~((uint64_t)__float_as_uint(x) | ((uint64_t)__float_as_uint(y) << 32));
  return w ? w : 1ull;
}
__device__ __forceinline__ float2 shared_pair(uint64_t w) {
  return make_float2(__uint_as_float(~(uint32_t)w), __uint_as_float(~(uint32_t)(w >> 32)));
}
template <int G>
__device__ __forceinline__ void attn_finish_shared(const AttnSharedArgs& a, int b, int kvh, int split,
                                                   float (*sm_acc)[G][kHeadDim], float (*sm_m)[G], float (*sm_l)[G],
                                                   float2 (*sm_sum)[kHeadDim / 2]) {
  constexpr int kColumns = kHeadDim / 2;  // two adjacent dims each
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ns = a.nsplit, parts = a.share.parts, cols = a.share.cols;
  const int stride = G * (kColumns + parts);  // words of a split: its sums, then its (max, sum) for every reader
  uint64_t* const words = a.share.words + (size_t)(b * a.num_kv_heads + kvh) * ns * stride;
  auto head_of = [&](int reader) { return (int)((uint32_t)reader * a.share.parts_magic >> 16); };
  __syncthreads();
  auto merged = [&](int g, float (&sc)[kAttnWaves], float& mm) {
    mm = kNegBig;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) mm = fmaxf(mm, sm_m[w][g]);
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) sc[w] = __expf(sm_m[w][g] - mm);
  };
  if (split >= a.share.absent) {
    uint64_t* const to = words + (size_t)split * stride;
    for (int idx = tid; idx < G * kColumns; idx += kAttnThreads) {
      const int g = idx / kColumns, d = (idx % kColumns) * 2;
      float sc[kAttnWaves], mm, o0 = 0.f, o1 = 0.f;
      merged(g, sc, mm);
#pragma unroll
      for (int w = 0; w < kAttnWaves; ++w) {
        o0 += sm_acc[w][g][d] * sc[w];
        o1 += sm_acc[w][g][d + 1] * sc[w];
      }
      __hip_atomic_store(&to[idx], share_word(o0, o1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (tid < G * parts) {  // (at most kAttnShareSplits of them)
      const int g = head_of(tid);
      float sc[kAttnWaves], mm, ll = 0.f;
      merged(g, sc, mm);
#pragma unroll
      for (int w = 0; w < kAttnWaves; ++w) ll += sm_l[w][g] * sc[w];
      __hip_atomic_store(&to[G * kColumns + tid], share_word(mm, ll), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (tid >= 64) {
    attn_clear_on_the_side(a);
    if (tid >= kAttnThreads - 64 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) attn_commit(a.commit);
  }
  if (split >= G * parts) return;

  // Sixteen lanes have a column each (and sixteen further on, the next), the sixteen groups of them a split each.
  const int g = head_of(split), first = (split - g * parts) * cols, here = min(cols, kColumns - first);
  const int c = lane & 15, group = tid >> 4;
  uint64_t* const sums = words + g * kColumns + first;
  uint64_t* const ml = words + G * kColumns + split;
  float m_all = kNegBig, l_all = 0.f;
  auto collect = [&](auto count_c, auto passes_c) __attribute__((always_inline)) {
    constexpr int COUNT = decltype(count_c)::value, PASSES = decltype(passes_c)::value;
    uint64_t w[COUNT][PASSES], x[COUNT];
    const uint64_t t0 = wall_clock64();
    bool lost = false;
    for (uint32_t polls = 1;; ++polls) {
      bool come = true;
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        const int mine = group + 16 * i, s = c + 16 * i;
        x[i] = s < ns ? __hip_atomic_load(&ml[(size_t)s * stride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : share_word(kNegBig, 0.f);
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
          w[i][p] = mine < ns && c + 16 * p < here
                        ? __hip_atomic_load(&sums[(size_t)mine * stride + c + 16 * p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                        : ~0ull;
      }
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        come = come && x[i] != 0ull;
#pragma unroll
        for (int p = 0; p < PASSES; ++p) come = come && w[i][p] != 0ull;
      }
      if (__all(come)) break;
      if ((polls & 15u) == 0 && wall_clock64() - t0 > a.share.ticks) {
        lost = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    // What every wait of a layer does that gives up: the request has no result, and says so.
    if (lost) {
      if (lane == 0) {
        __hip_atomic_store(&a.share.sel_len[b], -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.share.fault_out) __hip_atomic_store(a.share.fault_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        x[i] = share_word(kNegBig, 0.f);
#pragma unroll
        for (int p = 0; p < PASSES; ++p) w[i][p] = ~0ull;
      }
    }
    float2 pair[COUNT];
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
      pair[i] = shared_pair(x[i]);
      m_all = fmaxf(m_all, pair[i].x);
    }
    m_all = fmaxf(m_all, dpp_move<kRowRor8>(m_all));
    m_all = fmaxf(m_all, dpp_move<kRowRor4>(m_all));
    m_all = fmaxf(m_all, dpp_move<kRowRor2>(m_all));
    m_all = fmaxf(m_all, dpp_move<kRowRor1>(m_all));
    float o0[PASSES], o1[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) o0[p] = o1[p] = 0.f;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
      const float e = c + 16 * i < ns ? __expf(pair[i].x - m_all) : 0.f;
      l_all += pair[i].y * e;
      const float weight = __shfl(e, (lane & 48) | group);
#pragma unroll
      for (int p = 0; p < PASSES; ++p) {
        const float2 o = shared_pair(w[i][p]);
        o0[p] += o.x * weight;
        o1[p] += o.y * weight;
      }
    }
    l_all = row16_sum(l_all);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      o0[p] += __shfl_xor(o0[p], 16);
      o1[p] += __shfl_xor(o1[p], 16);
      o0[p] += __shfl_xor(o0[p], 32);
      o1[p] += __shfl_xor(o1[p], 32);
      if (lane < 16) sm_sum[wave][lane + 16 * p] = make_float2(o0[p], o1[p]);
    }
    __syncthreads();
    if (tid < here) {
      float2 o = sm_sum[0][tid];
#pragma unroll
      for (int v = 1; v < kAttnWaves; ++v) {
        o.x += sm_sum[v][tid].x;
        o.y += sm_sum[v][tid].y;
      }
      *(uint32_t*)(a.out + ((size_t)b * a.num_heads + kvh * G + g) * kHeadDim + 2 * (first + tid)) =
          (uint32_t)f32_to_bf16(l_all > 0.f ? o.x / l_all : 0.f) | ((uint32_t)f32_to_bf16(l_all > 0.f ? o.y / l_all : 0.f) << 16);
    }
    // Zero again, for the next launch (nobody else reads them; the maxima are every wavefront's of this workgroup).
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
      const int mine = group + 16 * i;
#pragma unroll
      for (int p = 0; p < PASSES; ++p)
        if (mine < ns && c + 16 * p < here) sums[(size_t)mine * stride + c + 16 * p] = 0ull;
    }
    for (int s = tid; s < ns; s += kAttnThreads) ml[(size_t)s * stride] = 0ull;
  };
  auto for_columns = [&](auto count_c) __attribute__((always_inline)) {
    if (cols <= 16) collect(count_c, std::integral_constant<int, 1>{});
    else if (cols <= 32) collect(count_c, std::integral_constant<int, 2>{});
    else collect(count_c, std::integral_constant<int, 4>{});
  };
  if (ns <= 16) for_columns(std::integral_constant<int, 1>{});
  else if (ns <= 32) for_columns(std::integral_constant<int, 2>{});
  else if (ns <= 48) for_columns(std::integral_constant<int, 3>{});
  else for_columns(std::integral_constant<int, 5>{});
}

// ---------------------------------------------------------------------------------------
// attn_kernel<G, ROPE, CAP, FORM>: G = H / Hkv query heads per workgroup (1 to 8), on the matrix
// cores.  A wavefront walks a contiguous quarter of the workgroup's range in tiles of 32
// tokens.  v_mfma_f32_16x16x32_bf16 three times over:
//   logits   S[token][head] = K' Q'^T : A = 16 rotated keys x 32 dims (lane (token l%16,
//            l/16) loads 16 bytes of its token's row per 32 dims and rotates them in fp32 -
//            the partner dims d and d + 64 are in the same lane), B = the query heads as
//            columns (G of 16 used), rotated to S - 1 once.
//   V^T      a value row arrives like a key row (a lane holds 8 consecutive dims of one
//            token); the matrix product with a 0/1 matrix that selects 16 of 32 dims leaves
//            lane (dim l%16, l/16) with that dim of four consecutive tokens, exactly (bf16
//            values summed with zeros in fp32): the transposition, without LDS.
//   output   O^T[dim][head] += V^T P : A = 16 dims x 32 tokens from the step above, B = the
//            weights of the tile, which the logits' product left in the lanes that need them
//            (lane (head l%16, l/16): tokens 4 (l/16) + r of both 16-token halves).
// The matrix instructions take bf16, the reference's attention works in fp32 on rotated keys:
// every fp32 operand (rotated key, rotated query, softmax weight) is therefore split into a
// bf16 value and the bf16 of what the rounding left, x = hi + lo to 2^-18 of x, and the
// products are taken as hi hi + lo hi + hi lo (fp32 accumulation; the values are bf16 as
// stored).  The results match an fp32 evaluation to the rounding of the bf16 output; with
// single bf16 operands the mean error was a hundred times larger and the largest one
// exceeded 2e-2 for outputs of magnitude 2 under a peaked softmax.
// Everything of a head lives in the four lanes of its column: the running maximum moves once
// per tile (two exchanges between the lane groups), the sums stay per lane until the end.
// The loads of the next tile's keys are issued when this tile's have been rotated, those of
// its values after this tile's have been consumed: some 8 KB per wavefront are in flight at
// any time.
typedef __attribute__((ext_vector_type(8))) __bf16 at_bf16x8;
typedef __attribute__((ext_vector_type(4))) float at_f32x4;
constexpr float kAttnLog2e = 1.4426950408889634f, kAttnLn2 = 0.6931471805599453f;
constexpr uint32_t kNewRow = 0xffffffffu;  // the slot of a row that is not in the pool (no pool has as many)

__device__ __forceinline__ at_bf16x8 pack8(const float* x) {
  const uint4 w = make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]),
                             pack_bf16(x[6], x[7]));
  return __builtin_bit_cast(at_bf16x8, w);
}
__device__ __forceinline__ void unpack8(const uint4& w, float* f) {
  f[0] = bf16_lo(w.x);
  f[1] = bf16_hi(w.x);
  f[2] = bf16_lo(w.y);
  f[3] = bf16_hi(w.y);
  f[4] = bf16_lo(w.z);
  f[5] = bf16_hi(w.z);
  f[6] = bf16_lo(w.w);
  f[7] = bf16_hi(w.w);
}

// x = hi + lo with both halves in bf16: hi = x rounded, lo = the remainder rounded (the
// subtraction is exact); what is lost is 2^-18 of x.
__device__ __forceinline__ void split8(const float* x, at_bf16x8& hi, at_bf16x8& lo) {
  const uint4 h = make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]),
                             pack_bf16(x[6], x[7]));
  const float r[8] = {x[0] - bf16_lo(h.x), x[1] - bf16_hi(h.x), x[2] - bf16_lo(h.y), x[3] - bf16_hi(h.y),
                      x[4] - bf16_lo(h.z), x[5] - bf16_hi(h.z), x[6] - bf16_lo(h.w), x[7] - bf16_hi(h.w)};
  hi = __builtin_bit_cast(at_bf16x8, h);
  lo = pack8(r);
}

// An index offset of zero that the compiler cannot see through, produced after `after` is:
// LDS reads addressed with it stay where they are written (inside the loop, next to their
// use) instead of being gathered at the top, where they would hold dozens of registers.
__device__ __forceinline__ int opaque_zero(uint32_t after) {
  int z = 0;
  asm volatile("" : "+v"(z) : "v"(after));
  return z;
}

// DENSE (AttnDense) is an instantiation of its own: with its few instructions in the one kernel the
// attention over a list took 1 us more.
enum AttnForm { kAttnList, kAttnDenseStep, kAttnShared, kAttnSharedHalf };
template <int G, bool ROPE, bool CAP, int FORM>
__global__ __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_kernel(
    std::conditional_t<(FORM >= kAttnShared), AttnSharedArgs, AttnArgs> a) {
  constexpr bool DENSE = FORM == kAttnDenseStep, SHARED = FORM >= kAttnShared;
  constexpr bool HALF = FORM == kAttnSharedHalf;  // a wavefront has 16 tokens: half a tile is all there is
  constexpr int TILES = HALF ? 1 : 2;
  static_assert(G >= 1 && G <= 8, "the query heads of a KV head are columns of one tile");
  const int split = blockIdx.x, b = blockIdx.z, kvh = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, qd = lane >> 4;
  const int chunk = attn_chunk(a.max_sel_len, a.nsplit);
  const int wlen = chunk / kAttnWaves;
  const int32_t* sel = a.sel + (int64_t)b * a.sel_stride;
  const size_t row_elems = (size_t)a.num_kv_heads * kHeadDim;

  // What every wavefront reads again and again lives in LDS, not in registers (the loop
  // below needs them all): the query operand, the 0/1 matrices, the rotation of one step.
  __shared__ __attribute__((aligned(16))) uint4 sm_q[4][64];     // B operand per 32 dims, per lane
  __shared__ __attribute__((aligned(16))) uint4 sm_q_lo[4][64];  // its low halves
  __shared__ __attribute__((aligned(16))) uint4 sm_pick[2][64];  // B operand per half, per lane
  __shared__ __attribute__((aligned(16))) float2 sm_step[kHeadDim / 2];  // (cos, sin) of 16 tokens
  __shared__ float sm_acc[kAttnWaves][G][kHeadDim];
  __shared__ float sm_m[kAttnWaves][G], sm_l[kAttnWaves][G];
  __shared__ uint32_t s_last;
  __shared__ float2 sm_sum[SHARED ? kAttnWaves : 1][kHeadDim / 2];

  // Column n of the logits: query head n of the KV head (zeros beyond its heads).  Wavefront
  // kb2 < 2 prepares the dims [32 kb2, +32) and their partners 64 further on.
  const bool real = n < G;
  const int head = kvh * G + min(n, G - 1);
  // (No load of the start-up sits behind a branch: where a branch joins, the compiler waits
  // for every load that either side may have issued.)
  uint4 q_raw[2];
  {
    const uint16_t* qrow = a.q + (size_t)b * a.q_stride + head * kHeadDim + 32 * (wave & 1) + 8 * qd;
    q_raw[0] = *(const uint4*)qrow;
    q_raw[1] = *(const uint4*)(qrow + 64);
  }
  // The first tile's slots are asked for together with the list's length, not after it.
  // An entry past the wavefront's range (its token gets the weight zero) is replaced by the
  // slot of the range's first token: its row must still be one that holds numbers.
  const int wlo = split * chunk + wave * wlen;
  auto raw_slot = [&](int j) {
    if (!DENSE) return (uint32_t)sel[min(j, a.max_sel_len - 1)];
    return ((uint32_t)sel[min(j, a.list_bound - 1) >> a.list_shift] << a.list_shift) +
           (uint32_t)(j & ((1 << a.list_shift) - 1));
  };
  uint32_t slot_cur[2] = {raw_slot(wlo + n), HALF ? 0u : raw_slot(wlo + 16 + n)};
  uint32_t slot_next[2] = {HALF ? 0u : raw_slot(wlo + kAttnTile + n), HALF ? 0u : raw_slot(wlo + kAttnTile + 16 + n)};
  // A dense step's list is the table and, at the end, the new token, whose row is not in the pool
  // yet: it is read where the caller has it, as slot kNewRow.  (With no new token some word that can
  // be read is loaded in place of its slot.)
  const int length = a.sel_len[b];
  const int new_slot = DENSE ? (a.step.loc ? a.step.loc : a.sel_len)[b] : -1;
  const bool appends = DENSE && attn_appends(a, new_slot, length);
  const int new_pos = appends ? length : -1;
  const uint32_t own_slot = appends ? (uint32_t)new_slot : kNewRow;
  const int S = min(max(length + (appends ? 1 : 0), 0), DENSE ? a.list_bound : a.max_sel_len);
  const int whi = min(S, wlo + wlen);
  uint32_t first_slot =
      min((uint32_t)__builtin_amdgcn_readfirstlane((int)slot_cur[0]), a.pool_rows - 1);
  if (DENSE && wlo == new_pos) first_slot = kNewRow;
  auto checked = [&](uint32_t slot, int j) {
    if (!DENSE) return j < whi && slot < a.pool_rows ? slot : first_slot;
    // (an entry that is no slot: as it is listed; one that the table lists already, as a padded
    // request's does: the row that is about to be there)
    const uint32_t entry = j < whi ? min(slot, a.pool_rows - 1) : first_slot;
    return (j == new_pos) | (entry == own_slot) ? kNewRow : entry;
  };
  slot_cur[0] = checked(slot_cur[0], wlo + n);
  slot_cur[1] = checked(slot_cur[1], wlo + 16 + n);
  slot_next[0] = checked(slot_next[0], wlo + kAttnTile + n);
  slot_next[1] = checked(slot_next[1], wlo + kAttnTile + 16 + n);
  // ... and the first tile's rows before the set-up below, which then runs while they travel.
  uint4 kr[2][4], vr[2][4];
  // (from_new: elements from the pool to the new token's row)
  auto request = [&](const uint16_t* pool, int64_t from_new, const uint32_t* slots, uint4 (&dst)[2][4]) {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      size_t at = (size_t)slots[t] * row_elems;
      if (DENSE && slots[t] == kNewRow) at = (size_t)from_new;
      const uint16_t* row = pool + at + (size_t)kvh * kHeadDim + 8 * qd;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) dst[t][kb] = *(const uint4*)(row + 32 * kb);
    }
  };
  const int64_t new_k = a.step.k_from_pool + (int64_t)b * a.step.kv_stride;
  const int64_t new_v = a.step.v_from_pool + (int64_t)b * a.step.kv_stride;
  // (a wavefront without tokens asks too: rows of some entry of the list, never used)
  request(a.k_pool, new_k, slot_cur, kr);
  request(a.v_pool, new_v, slot_cur, vr);

  if (tid < kHeadDim / 2) {
    float sn = 0.f, cs = 1.f;
    if (ROPE) {
      const float freq =
          a.rope_rcp_scale * __builtin_amdgcn_exp2f(-(float)tid * (2.0f / kHeadDim) * a.log2_theta);
      sincos_reduced(16.0f * freq, sn, cs);
    }
    sm_step[tid] = make_float2(cs, sn);
    // 0/1 matrices that pick the dims [16 h, 16 h + 16) of a 32-dim block: B operand, lane
    // (column n, qd) holds rows 8 qd .. 8 qd + 7, of which row 16 h + n is the one.
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      if (qd == 2 * h + (n >> 3)) w[(n & 7) >> 1] = (n & 1) ? 0x3f800000u : 0x00003f80u;
      sm_pick[h][lane] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  if (wave < 2) {  // the query rotated to position S - 1, rounded once
    float x[8], y[8];
    unpack8(real ? q_raw[0] : make_uint4(0u, 0u, 0u, 0u), x);
    unpack8(real ? q_raw[1] : make_uint4(0u, 0u, 0u, 0u), y);
    if (ROPE) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int pair = 32 * wave + 8 * qd + e;
        const float freq =
            a.rope_rcp_scale * __builtin_amdgcn_exp2f(-(float)pair * (2.0f / kHeadDim) * a.log2_theta);
        float sn, cs;
        sincos_reduced((float)(S - 1) * freq, sn, cs);
        // (which product is rounded is said here and for the keys below: left to the compiler it
        // changed with code elsewhere in the kernel, and one output in some 3000 by an ulp)
        const float xr = fmaf(x[e], cs, -(y[e] * sn));
        y[e] = fmaf(y[e], cs, x[e] * sn);
        x[e] = xr;
      }
    }
    at_bf16x8 hi, lo;
    split8(x, hi, lo);
    sm_q[wave][lane] = __builtin_bit_cast(uint4, hi);
    sm_q_lo[wave][lane] = __builtin_bit_cast(uint4, lo);
    split8(y, hi, lo);
    sm_q[wave + 2][lane] = __builtin_bit_cast(uint4, hi);
    sm_q_lo[wave + 2][lane] = __builtin_bit_cast(uint4, lo);
  }
  // This lane's 16 rotation pairs: dims 32 kb2 + 8 qd + e (kb2 < 2, e < 8) and their partners
  // 64 further on; key state at token wlo + n, 16 tokens per step.
  float kc[16], ks[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    kc[i] = 1.f;
    ks[i] = 0.f;
    if (ROPE) {
      const int pair = 32 * (i >> 3) + 8 * qd + (i & 7);
      const float freq =
          a.rope_rcp_scale * __builtin_amdgcn_exp2f(-(float)pair * (2.0f / kHeadDim) * a.log2_theta);
      sincos_reduced((float)(wlo + n) * freq, ks[i], kc[i]);
    }
  }
  __syncthreads();  // sm_q, sm_pick, sm_step

  float m = kNegBig, l = 0.f;  // base-2 running maximum, this lane's share of the sum
  at_f32x4 acc[8];             // O^T: dims 16 dt + 4 qd + r of head n
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) acc[dt] = at_f32x4{0.f, 0.f, 0.f, 0.f};

  if (wlo < whi) {
    const float scale2 = a.sm_scale * kAttnLog2e;

    // One tile; `more` (a compile-time flag: the last tile is a copy of the loop's body
    // without the requests) says that another tile follows.  Its loads are unconditional:
    // behind a branch the compiler would wait for all loads where the branch joins, the ones
    // just issued included.
    // `half` (compile-time as well, last tile only): the range ends within the tile's first 16
    // tokens, and nothing is computed for the other 16.
    auto tile = [&](const int j0, auto more_flag, auto half_flag) __attribute__((always_inline)) {
      constexpr bool more = decltype(more_flag)::value;
      constexpr bool half = decltype(half_flag)::value;
      static_assert(!(more && half), "only a last tile ends early");
      // The slots of the tile after the next are asked for before the next tile's rows, so
      // that waiting for them does not mean waiting for those rows (loads return in order).
      uint32_t slot_after[2] = {0u, 0u};
      if (more) {
        slot_after[0] = raw_slot(j0 + 2 * kAttnTile + n);
        slot_after[1] = raw_slot(j0 + 2 * kAttnTile + 16 + n);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- keys, 16 tokens at a time: rotate, round, multiply, step the rotation
      at_f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int t = 0; t < (half ? 1 : 2); ++t) {
        at_bf16x8 ka[4], ka_lo[4];
#pragma unroll
        for (int kb2 = 0; kb2 < 2; ++kb2) {
          float x[8], y[8];
          unpack8(kr[t][kb2], x);
          unpack8(kr[t][kb2 + 2], y);
          if (ROPE) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float c = kc[8 * kb2 + e], sn = ks[8 * kb2 + e];
              const float xr = fmaf(x[e], c, -(y[e] * sn));
              y[e] = fmaf(y[e], c, x[e] * sn);
              x[e] = xr;
            }
          }
          split8(x, ka[kb2], ka_lo[kb2]);
          split8(y, ka[kb2 + 2], ka_lo[kb2 + 2]);
        }
        const int zq = opaque_zero(__builtin_bit_cast(uint4, ka[3]).w);
        s[t] = at_f32x4{0.f, 0.f, 0.f, 0.f};
        // (k_hi + k_lo) (q_hi + q_lo) without the product of the two low halves: three
        // chains that do not wait for each other, added up at the end.
        at_f32x4 s_lh = {0.f, 0.f, 0.f, 0.f}, s_hl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const at_bf16x8 q_hi = __builtin_bit_cast(at_bf16x8, sm_q[kb][lane + zq]);
          const at_bf16x8 q_lo = __builtin_bit_cast(at_bf16x8, sm_q_lo[kb][lane + zq]);
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[kb], q_hi, s[t], 0, 0, 0);
          s_lh = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka_lo[kb], q_hi, s_lh, 0, 0, 0);
          s_hl = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[kb], q_lo, s_hl, 0, 0, 0);
        }
        s[t] += s_lh + s_hl;
        __builtin_amdgcn_sched_barrier(0);
        if (ROPE && (more || (t == 0 && !half))) {  // the same rows of the next 16 tokens
#pragma unroll
          for (int kb2 = 0; kb2 < 2; ++kb2) {
            const int zs = opaque_zero(__float_as_uint(kc[8 * kb2]));
            const float4* step = (const float4*)&sm_step[32 * kb2 + 8 * qd + zs];
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {
              const float4 d = step[e2];
              const float dcs[2] = {d.x, d.z}, dsn[2] = {d.y, d.w};
#pragma unroll
              for (int o = 0; o < 2; ++o) {
                const int i = 8 * kb2 + 2 * e2 + o;
                const float c2 = fmaf(kc[i], dcs[o], -(ks[i] * dsn[o]));
                ks[i] = fmaf(kc[i], dsn[o], ks[i] * dcs[o]);
                kc[i] = c2;
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      // the next tile's keys, into the registers just read
      if (more) request(a.k_pool, new_k, slot_next, kr);
      __builtin_amdgcn_sched_barrier(0);
      // ---- weights of 32 tokens x 16 head columns
      float p[8];
      float mx = kNegBig;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (half && t == 1) {
            p[4 + r] = -INFINITY;
            continue;
          }
          float v;
          if (CAP)
            v = a.logit_cap * tanhf(s[t][r] * a.sm_scale / a.logit_cap) * kAttnLog2e;
          else
            v = s[t][r] * scale2;
          v = j0 + 16 * t + 4 * qd + r < whi ? v : -INFINITY;
          p[4 * t + r] = v;
          mx = fmaxf(mx, v);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = half && i >= 4 ? 0.f : __builtin_amdgcn_exp2f(p[i] - mn);
        sum += p[i];
      }
      l = l * alpha + sum;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[dt] *= alpha;
      at_bf16x8 pb, pb_lo;
      split8(p, pb, pb_lo);
      // ---- values: transpose 16 dims at a time, accumulate
      const int zp = opaque_zero(__builtin_bit_cast(uint4, pb).x);
      at_bf16x8 pick[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) pick[h] = __builtin_bit_cast(at_bf16x8, sm_pick[h][lane + zp]);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const at_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          const at_f32x4 d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(at_bf16x8, vr[0][c]), pick[h], zero, 0, 0, 0);
          const at_f32x4 d1 = half ? zero
                                   : __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                         __builtin_bit_cast(at_bf16x8, vr[1][c]), pick[h], zero, 0, 0, 0);
          const float vt[8] = {d0[0], d0[1], d0[2], d0[3], d1[0], d1[1], d1[2], d1[3]};
          const at_bf16x8 vta = pack8(vt);
          acc[2 * c + h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vta, pb, acc[2 * c + h], 0, 0, 0);
          acc[2 * c + h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vta, pb_lo, acc[2 * c + h], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        request(a.v_pool, new_v, slot_next, vr);
        slot_next[0] = checked(slot_after[0], j0 + 2 * kAttnTile + n);
        slot_next[1] = checked(slot_after[1], j0 + 2 * kAttnTile + 16 + n);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // (Lowering a wavefront's priority as it advances, which evens out the two workgroups of
    // a CU in the kernel above, evens them out here too and gains nothing: the rows arrive
    // as fast as the memory system delivers them either way.)
    if constexpr (HALF) {
      tile(wlo, std::false_type{}, std::true_type{});
    } else {
      int j0 = wlo;
      for (; j0 + kAttnTile < whi; j0 += kAttnTile) tile(j0, std::true_type{}, std::false_type{});
      if (whi - j0 <= kAttnTile / 2)
        tile(j0, std::false_type{}, std::true_type{});
      else
        tile(j0, std::false_type{}, std::false_type{});
    }
  }

  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (n < G) {
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      *(float4*)&sm_acc[wave][n][16 * dt + 4 * qd] = make_float4(acc[dt][0], acc[dt][1], acc[dt][2], acc[dt][3]);
    if (qd == 0) {
      sm_m[wave][n] = m * kAttnLn2;  // natural-log units, as the merge expects
      sm_l[wave][n] = l;
    }
  }
  if constexpr (SHARED) {
    attn_finish_shared<G>(a, b, kvh, split, sm_acc, sm_m, sm_l, sm_sum);
  } else {
    const bool last = attn_finish<G>(a, b, kvh, split, sm_acc, sm_m, sm_l, &s_last);
    if (DENSE) attn_dense_epilogue(a, b, kvh, split * chunk, (split + 1) * chunk, S, new_slot, length, appends, last);
  }
}

__global__ __launch_bounds__(256) void attn_zero_kernel(uint32_t* tickets, int count) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) tickets[i] = 0u;
}

// Tickets per request (the words to clear): one per KV head, and one for the heads of a dense step.
int attn_tickets_per_request(const ts_config* cfg) { return cfg->num_kv_heads + 1; }

static int attn_splits(int batch, int num_kv_heads, int max_sel_len) {
  // One tile per wavefront (128 entries per workgroup) as long as the grid stays within the
  // 512 workgroups that are resident at once (two per CU): a second round of workgroups pays
  // the start-up and merge latencies again, which costs more than longer ranges do.
  int64_t want = ceil_div(max_sel_len, kAttnRange);
  const int64_t cap = ceil_div(2048 / kAttnWaves, (int64_t)batch * num_kv_heads);
  if (want > cap) want = cap;
  if (want < 1) want = 1;
  // (ranges are whole multiples of 64 entries: the last splits may have nothing left)
  return (int)ceil_div(max_sel_len, attn_chunk(max_sel_len, (int)want));
}

// The tickets come first, where they lie whatever the length of the lists: a completed call of any
// of them leaves the words of the next one zero.
struct AttnWorkspace {
  size_t tickets, acc, ml, total;
};
static AttnWorkspace attn_workspace(const ts_config* cfg, int batch, int max_sel_len) {
  const size_t ns = (size_t)attn_splits(batch, cfg->num_kv_heads, max_sel_len);
  const size_t heads = (size_t)batch * cfg->num_heads;
  AttnWorkspace w;
  w.tickets = 0;
  w.acc = align_up((size_t)batch * attn_tickets_per_request(cfg) * 4, 256);
  w.ml = w.acc + align_up(heads * ns * kHeadDim * 4, 256);
  w.total = w.ml + align_up(heads * ns * 2 * 4, 256);
  return w;
}

uint32_t* attn_tickets(void* workspace) { return (uint32_t*)workspace; }

size_t attn_workspace_bytes(const ts_config* cfg, int batch, int max_sel_len) {
  return attn_workspace(cfg, batch, max_sel_len).total;
}

// The kernel of a call whose splits are shared, 64 entries each or more.
template <int G>
static const void* shared_kernel_of(bool rope, bool cap, bool half) {
  if (half)
    return rope ? (cap ? (const void*)&attn_kernel<G, true, true, kAttnSharedHalf> : (const void*)&attn_kernel<G, true, false, kAttnSharedHalf>)
                : (cap ? (const void*)&attn_kernel<G, false, true, kAttnSharedHalf> : (const void*)&attn_kernel<G, false, false, kAttnSharedHalf>);
  return rope ? (cap ? (const void*)&attn_kernel<G, true, true, kAttnShared> : (const void*)&attn_kernel<G, true, false, kAttnShared>)
              : (cap ? (const void*)&attn_kernel<G, false, true, kAttnShared> : (const void*)&attn_kernel<G, false, false, kAttnShared>);
}
static const void* shared_kernel_of(int group, bool rope, bool cap, bool half) {
  switch (group) {
    case 1: return shared_kernel_of<1>(rope, cap, half);
    case 2: return shared_kernel_of<2>(rope, cap, half);
    case 3: return shared_kernel_of<3>(rope, cap, half);
    case 4: return shared_kernel_of<4>(rope, cap, half);
    case 5: return shared_kernel_of<5>(rope, cap, half);
    case 6: return shared_kernel_of<6>(rope, cap, half);
    case 7: return shared_kernel_of<7>(rope, cap, half);
    case 8: return shared_kernel_of<8>(rope, cap, half);
    default: return nullptr;
  }
}
// What the current device holds of them (nothing: it did not answer, and is asked again).
static AttnRoom attn_room(int group, bool rope, bool cap) {
  struct Entry { int device, kind; AttnRoom room; };
  constexpr int kMemo = 8;
  static thread_local Entry memo[kMemo] = {};
  static thread_local int next = 0;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return AttnRoom{};
  const int kind = group * 4 + rope * 2 + cap;
  for (const Entry& e : memo)
    if (e.kind == kind && e.device == device) return e.room;
  int cus = 0, per_cu[2] = {0, 0};
  bool ok = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess;
  for (int half = 0; half < 2; ++half) {
    const void* fn = shared_kernel_of(group, rope, cap, half != 0);
    ok = ok && fn && hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu[half], fn, kAttnThreads, 0) == hipSuccess;
  }
  if (!ok) {
    (void)hipGetLastError();
    return AttnRoom{};
  }
  const AttnRoom room{cus, cus * per_cu[1], cus * per_cu[0]};
  memo[next] = Entry{device, kind, room};
  next = (next + 1) % kMemo;
  return room;
}

AttnShare attn_share(const ts_config* cfg, int batch, int max_sel_len, void* words, size_t bytes) {
  const AttnRoom room =
      attn_room(cfg->num_heads / cfg->num_kv_heads, cfg->rope_mode == TS_ROPE_LLAMA, cfg->logit_cap > 0.f);
  AttnShare s = plan_attn_share(batch, cfg->num_heads, cfg->num_kv_heads, max_sel_len, room);
  if (s.nsplit == 0 || s.bytes > bytes) return AttnShare{};
  s.words = (uint64_t*)words;
  return s;
}

int launch_attn(const ts_config* cfg, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                int64_t pool_rows, const int32_t* sel, int64_t sel_stride, const int32_t* sel_len,
                int batch, int max_sel_len, void* out, void* workspace, bool tickets_clear,
                hipStream_t st, const ZeroSet* clear_after, const AttnDense* dense, const StepCommit* commit,
                const AttnShare* share) {
  const AttnWorkspace w = attn_workspace(cfg, batch, max_sel_len);
  AttnSharedArgs a;
  a.step = AttnDense{};
  a.commit = commit ? *commit : StepCommit{};
  a.list_shift = a.list_bound = 0;
  if (dense) {
    a.step = *dense;
    a.list_shift = page_shift_of(cfg->page_size);
    a.list_bound = dense->list_bound;
    TS_REQUIRE(!dense->loc || a.list_shift == 0, TS_EINVAL, "internal: a dense step appends to per-token tables only");
  }
  if (clear_after) {
    TS_REQUIRE(!clear_after->overflow, TS_EINVAL, "internal: more than %d regions to clear in one launch",
               kZeroRegions);
    a.zero = *clear_after;
  }
  a.q = (const uint16_t*)q;
  a.q_stride = q_stride;
  a.k_pool = (const uint16_t*)k_pool;
  a.v_pool = (const uint16_t*)v_pool;
  a.pool_rows = (uint32_t)pool_rows;
  a.sel = sel;
  a.sel_stride = sel_stride;
  a.sel_len = sel_len;
  a.num_heads = cfg->num_heads;
  a.num_kv_heads = cfg->num_kv_heads;
  a.group = cfg->num_heads / cfg->num_kv_heads;
  a.rope_mode = cfg->rope_mode;
  a.log2_theta = cfg->rope_mode == TS_ROPE_LLAMA ? (float)log2((double)cfg->rope_theta) : 0.f;
  a.rope_rcp_scale = cfg->rope_mode == TS_ROPE_LLAMA ? 1.0f / cfg->rope_scale : 1.0f;
  a.sm_scale = cfg->sm_scale;
  a.logit_cap = cfg->logit_cap;
  a.nsplit = attn_splits(batch, cfg->num_kv_heads, max_sel_len);
  a.max_sel_len = max_sel_len;
  a.part_acc = (float*)((char*)workspace + w.acc);
  a.part_ml = (float*)((char*)workspace + w.ml);
  a.tickets = (uint32_t*)((char*)workspace + w.tickets);
  a.out = (uint16_t*)out;
  a.share = share ? *share : AttnShare{};
  if (share) a.nsplit = share->nsplit;

  if (!tickets_clear) {
    const int count = batch * attn_tickets_per_request(cfg);
    hipLaunchKernelGGL(attn_zero_kernel, dim3((unsigned)ceil_div(count, 256)), dim3(256), 0, st,
                       a.tickets, count);
    TS_TRY(check_launch("attn_zero_kernel"));
  }
  const dim3 grid((unsigned)a.nsplit, (unsigned)cfg->num_kv_heads, (unsigned)batch);
  const bool rope = cfg->rope_mode == TS_ROPE_LLAMA, cap = cfg->logit_cap > 0.f;
#define TS_ATTN_LAUNCH(G_, R_, C_)                                                                    \
  do {                                                                                                \
    if (dense) hipLaunchKernelGGL((attn_kernel<G_, R_, C_, kAttnDenseStep>), grid, dim3(kAttnThreads), 0, st, a); \
    else if (share && share->half) hipLaunchKernelGGL((attn_kernel<G_, R_, C_, kAttnSharedHalf>), grid, dim3(kAttnThreads), 0, st, a); \
    else if (share) hipLaunchKernelGGL((attn_kernel<G_, R_, C_, kAttnShared>), grid, dim3(kAttnThreads), 0, st, a); \
    else hipLaunchKernelGGL((attn_kernel<G_, R_, C_, kAttnList>), grid, dim3(kAttnThreads), 0, st, a);         \
  } while (0)
#define TS_ATTN_CASE(G_)                              \
  case G_:                                            \
    if (rope && cap) TS_ATTN_LAUNCH(G_, true, true);  \
    else if (rope) TS_ATTN_LAUNCH(G_, true, false);   \
    else if (cap) TS_ATTN_LAUNCH(G_, false, true);    \
    else TS_ATTN_LAUNCH(G_, false, false);            \
    break;
  switch (a.group) {
    TS_ATTN_CASE(1)
    TS_ATTN_CASE(2)
    TS_ATTN_CASE(3)
    TS_ATTN_CASE(4)
    TS_ATTN_CASE(5)
    TS_ATTN_CASE(6)
    TS_ATTN_CASE(7)
    TS_ATTN_CASE(8)
    default: return fail(TS_ESHAPE, "unsupported head group %d", a.group);
  }
#undef TS_ATTN_CASE
#undef TS_ATTN_LAUNCH
  return check_launch("attn_kernel");
}

// Scratch of ts_sparse_decode_attn_static: the split-K partials and tickets of one
// launch, held by every device the library runs on until the process ends.
constexpr size_t kStaticScratchBytes = 4u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Device address of `scratch` on the current device, looked up once per device (each
// device holds its own copy at its own address); NULL with the error set on failure.
constexpr int kMaxDevices = 64;
static void* static_scratch() {
  static std::mutex mu;
  static void* ptr_of_device[kMaxDevices] = {};
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess || device < 0 || device >= kMaxDevices) {
    (void)hipGetLastError();
    fail(TS_EHIP, "ts_sparse_decode_attn_static: no current device (%s)", hipGetErrorString(e));
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (ptr_of_device[device] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      fail(TS_EHIP, "ts_sparse_decode_attn_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return nullptr;
    }
    ptr_of_device[device] = ptr;
  }
  return ptr_of_device[device];
}

}  // namespace ts

using namespace ts;

extern "C" {

size_t ts_attn_workspace_bytes(const ts_config* cfg, int32_t batch, int32_t max_sel_len) {
  if (validate_config(cfg) != TS_OK || batch < 1 || max_sel_len < 1) return 0;
  return attn_workspace(cfg, batch, max_sel_len).total;
}

int ts_sparse_decode_attn(const ts_config* cfg, const void* q, const void* k_pool,
                          const void* v_pool, int64_t pool_rows, const int32_t* sel,
                          int64_t sel_stride, const int32_t* sel_len, int32_t batch,
                          int32_t max_sel_len, void* out, void* workspace,
                          size_t workspace_bytes, ts_stream_t stream) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(q && k_pool && v_pool && sel && sel_len && out, TS_EINVAL,
             "ts_sparse_decode_attn: NULL tensor argument");
  TS_REQUIRE(batch >= 1 && batch <= 65535, TS_EINVAL, "batch %d out of range", batch);
  TS_REQUIRE(max_sel_len >= 1, TS_EINVAL, "max_sel_len %d < 1", max_sel_len);
  TS_REQUIRE(sel_stride >= max_sel_len || batch == 1, TS_EWORKSPACE,
             "sel_stride %lld < max_sel_len %d", (long long)sel_stride, max_sel_len);
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  const size_t need = ts_attn_workspace_bytes(cfg, batch, max_sel_len);
  TS_REQUIRE(workspace != nullptr && workspace_bytes >= need, TS_EWORKSPACE,
             "ts_sparse_decode_attn: workspace %zu bytes < required %zu", workspace_bytes, need);
  TS_REQUIRE_ALIGNED(workspace, 256, "workspace");
  TS_REQUIRE_ALIGNED(q, 16, "q");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(v_pool, 16, "v_pool");
  TS_REQUIRE_ALIGNED(out, 16, "out");
  return launch_attn(cfg, q, cfg->num_heads * cfg->head_dim, k_pool, v_pool, pool_rows, sel, sel_stride, sel_len, batch, max_sel_len,
                     out, workspace, /*tickets_clear=*/false, (hipStream_t)stream);
}

size_t ts_attn_static_scratch_bytes(void) {
  // The query a caller makes at set-up also looks up the buffer's address on the current
  // device, so that a first call under graph capture makes no runtime query of its own.
  // (Without a device there is nothing to look up, and the size is still the answer.)
  int devices = 0;
  if (hipGetDeviceCount(&devices) == hipSuccess && devices > 0) (void)static_scratch();
  (void)hipGetLastError();
  return kStaticScratchBytes;
}

int ts_sparse_decode_attn_static(const ts_config* cfg, const void* q, const void* k_pool,
                                 const void* v_pool, int64_t pool_rows, const int32_t* sel,
                                 int64_t sel_stride, const int32_t* sel_len, int32_t batch,
                                 int32_t max_sel_len, void* out, ts_stream_t stream) {
  TS_TRY(validate_config(cfg));
  TS_REQUIRE(q && k_pool && v_pool && sel && sel_len && out, TS_EINVAL,
             "ts_sparse_decode_attn_static: NULL tensor argument");
  TS_REQUIRE(batch >= 1 && batch <= 65535, TS_EINVAL, "batch %d out of range", batch);
  TS_REQUIRE(max_sel_len >= 1, TS_EINVAL, "max_sel_len %d < 1", max_sel_len);
  TS_REQUIRE(sel_stride >= max_sel_len || batch == 1, TS_EWORKSPACE,
             "sel_stride %lld < max_sel_len %d", (long long)sel_stride, max_sel_len);
  TS_REQUIRE(pool_rows >= 1 && pool_rows <= 0x7fffffffLL, TS_EINVAL, "pool_rows %lld out of range",
             (long long)pool_rows);
  const size_t need = attn_workspace(cfg, batch, max_sel_len).total;
  TS_REQUIRE(need <= kStaticScratchBytes, TS_EWORKSPACE,
             "ts_sparse_decode_attn_static: batch %d x %d heads x %d selected needs %zu bytes of "
             "scratch, the built-in buffer holds %zu; use ts_sparse_decode_attn with a workspace",
             batch, cfg->num_heads, max_sel_len, need, kStaticScratchBytes);
  TS_REQUIRE_ALIGNED(q, 16, "q");
  TS_REQUIRE_ALIGNED(k_pool, 16, "k_pool");
  TS_REQUIRE_ALIGNED(v_pool, 16, "v_pool");
  TS_REQUIRE_ALIGNED(out, 16, "out");
  void* ptr = static_scratch();
  if (ptr == nullptr) return TS_EHIP;
  // The tickets are cleared by a fill kernel on the caller's stream (the previous call
  // may have been interrupted), so the call can be captured into a HIP graph.
  return launch_attn(cfg, q, cfg->num_heads * cfg->head_dim, k_pool, v_pool, pool_rows, sel, sel_stride, sel_len, batch, max_sel_len,
                     out, ptr, /*tickets_clear=*/false, (hipStream_t)stream);
}

}  // extern "C"
