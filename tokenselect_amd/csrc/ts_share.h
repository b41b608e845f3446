// How a decode attention's splits are dealt out where all of their workgroups merge them (attn_finish_shared,
// ts_attn.hip): nothing but arithmetic, for any host compiler.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace ts {

constexpr int kHeadDim = 128;
constexpr int kAttnWaves = 4;                    // wavefronts of a workgroup of the decode attention
constexpr int kAttnTile = 32;                    // tokens per step of a wavefront
constexpr int kAttnChunkUnit = 16 * kAttnWaves;  // a workgroup's range is a multiple of this
constexpr int kAttnRange = kAttnTile * kAttnWaves;  // list entries per workgroup as long as the device has room

// Tokens per workgroup of the matrix-core kernel for a launch of nsplit splits.
constexpr int attn_chunk(int max_sel_len, int nsplit) {
  const int even = (max_sel_len + nsplit - 1) / nsplit;
  return (even + kAttnChunkUnit - 1) / kAttnChunkUnit * kAttnChunkUnit;
}

// The splits of a request and KV head merged by all of their workgroups, which wait for each other's words
// (bounded; on giving up sel_len[b] = -1 and *fault_out = 1), in place of the last one to draw a ticket.  The words
// are zero at launch and again when the kernel ends without having given up.
struct AttnShare {
  uint64_t* words;  // [B, Hkv, split, G x 64 sums then G x parts (max, sum)], or NULL
  size_t bytes;
  int nsplit, half;          // splits; 64 entries each
  int parts, cols;           // workgroups that share a head's 64 columns of two dims, and columns of each
  uint32_t parts_magic;      // x / parts = x * parts_magic >> 16, for x below 2^8
  int absent;                // tests of the give-up: the first splits that send nothing
  uint64_t ticks;            // a wait at most (100 MHz)
  int32_t* sel_len;
  uint32_t* fault_out;
};

// What the device holds: its CUs, and the workgroups that are resident at once of the kernel with 64 entries each
// and of the one with more.
struct AttnRoom {
  int cus, half, full;
};

// Everything but the words and the waits; nsplit == 0: not shared.  They wait for each other, so that all of a launch
// must be resident: two per CU at most (more would gain nothing), and with 64 entries (16 a wavefront) where each has a
// CU to itself.  At most kAttnShareSplits, and at least one for each head of the group, whose columns they
// share.  us a layer merged by one and by all: one request of 20K, 28 heads on 4 36.1 and 32.3, 32 on 8 33.9 and 32.7
// (with 336 workgroups of 64 entries in place of 168 of 128, 33.4), 4 on 1 35.0 and 31.5; two of 8K, 28 on 4 37.9 and 35.3;
// eight, 14 splits each, 56.1 and 55.5; eight of 32 on 8, seven splits, 68.2 and 68.4: so from ten splits on.
constexpr int kAttnShareSplits = 80;
inline AttnShare plan_attn_share(int batch, int num_heads, int num_kv_heads, int max_sel_len, const AttnRoom& room) {
  AttnShare s{};
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t groups = (int64_t)batch * num_kv_heads, fine = up(max_sel_len, kAttnChunkUnit);
  const int G = num_heads / num_kv_heads;
  s.half = groups * fine <= std::min(room.cus, room.half);
  const int64_t want =
      s.half ? fine : std::min<int64_t>(up(max_sel_len, kAttnRange), std::min(room.full, 2 * room.cus) / groups);
  if (want < 2) return AttnShare{};
  s.nsplit = (int)up(max_sel_len, attn_chunk(max_sel_len, (int)want));
  if (s.nsplit < std::max(G, 10) || s.nsplit > kAttnShareSplits) return AttnShare{};
  s.parts = std::min(s.nsplit / G, 32);
  s.parts_magic = 65536u / (uint32_t)s.parts + 1u;
  s.cols = (int)up(kHeadDim / 2, s.parts);
  s.bytes = (size_t)groups * s.nsplit * G * (kHeadDim / 2 + s.parts) * 8;
  return s;
}

}  // namespace ts
