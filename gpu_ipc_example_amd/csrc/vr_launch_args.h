// Arguments of the collective kernels, packed.  The kernels, the host code that fills them in and
// a CPU test use these same functions.
//
// The runtime writes a launch's arguments to device memory and waits until they are there.  That
// costs the host 1.3 us a launch up to 112 bytes of arguments and 2.1 us from 116 on (launches in a row
// with 96, 104, 112, 116, 120, 128, 192, 296 bytes: 2.75, 2.80, 2.80, 3.47, 3.41, 3.48, 3.45, 3.52 us
// each; without any 1.45).  Eight ranks' inputs and outputs are 128 bytes as they are, 96 with 48
// bits a pointer, which is what a buffer resource takes and every device address fits: 16 are left
// for the rest.  (Tables of 16 + 16 whole pointers and 40 bytes beside them, as before: `simple` on 2 x
// 32 KiB 4.10 us a call from Python, now 3.55; `small` on 8 x 1 MiB 4.32, now 3.92.)
#pragma once

#include "vr_wire_layout.h"   // VR_HD

namespace vr {

constexpr size_t kCheapArgBytes = 112;

VR_HD uint64_t join48(uint32_t hi16, uint32_t lo) { return (uint64_t)hi16 << 32 | lo; }

// ---- direct transport (vr_direct.hip) --------------------------------------------------------
template <int N>
struct DirectArgs {
  uint32_t lo[2 * N], hi[N];  // inputs, then outputs: of the segment's first byte of chunk 0; two upper halves a word
  uint32_t pitch_lo;          // distance between chunk starts: lower 32 bits
  uint32_t seg_bytes;         // bytes of every chunk the launch covers
  uint32_t blocks_per_rank;
  // bits 0-2 log2 of the chunks dealt at a time; 3-7 waves of a work-group; 8-14 place of the first
  // output in its KiB, / 8; 15 head mask / 8; 16-19 all-gather: log2 of the tiles per XCD run;
  // 20-31 bits 32-43 of the pitch
  uint32_t shape;

  VR_HD uint64_t address(int k) const { return join48(hi[k / 2] >> 16 * (k % 2) & 0xffffu, lo[k]); }
  VR_HD uint32_t deal_log2() const { return shape & 7u; }
  // bytes one unroll step of a work-group spans, 16 a lane (from the arguments, so that nothing
  // waits for a separate load of the launch's dimensions)
  VR_HD uint32_t row() const { return (shape >> 3 & 31u) << 10; }
  VR_HD uint32_t place() const { return shape >> 5 & 1016u; }
  VR_HD uint32_t head_mask() const { return shape >> 12 & 8u; }
  VR_HD uint32_t run_log2() const { return shape >> 16 & 15u; }
  VR_HD uint64_t pitch() const { return join48(shape >> 20, pitch_lo); }
};
static_assert(sizeof(DirectArgs<8>) <= kCheapArgBytes, "a launch's arguments cost the host more beyond");

// The launch that covers [off, off + seg) of every chunk.
template <int N>
DirectArgs<N> direct_args(void *const in[], void *const out[], size_t pitch, size_t off, size_t seg, int block,
                          uint32_t blocks_per_rank, uint32_t deal_log2, uint32_t run_log2, uint32_t head_mask) {
  DirectArgs<N> a;
  for (int k = 0; k < 2 * N; k += 2) {
    const uint64_t p = (uint64_t)(uintptr_t)(k < N ? in[k] : out[k - N]) + off;
    const uint64_t q = (uint64_t)(uintptr_t)(k < N ? in[k + 1] : out[k + 1 - N]) + off;
    a.lo[k] = (uint32_t)p;
    a.lo[k + 1] = (uint32_t)q;
    a.hi[k / 2] = ((uint32_t)(p >> 32) & 0xffffu) | (uint32_t)(q >> 32) << 16;
  }
  a.pitch_lo = (uint32_t)pitch;
  a.seg_bytes = (uint32_t)seg;
  a.blocks_per_rank = blocks_per_rank;
  a.shape = deal_log2 | (uint32_t)block / 64u << 3 | (a.lo[N] >> 3 & 127u) << 8 | (head_mask ? 1u : 0u) << 15 | run_log2 << 16 |
            (uint32_t)((uint64_t)pitch >> 32) << 20;
  return a;
}

// ---- messages through LDS (vr_wire_group.hip) ----------------------------------------------------
// A rank's two pointers lie together: its wave takes all of them with two loads.
struct RankPtrs {
  uint32_t in_lo, out_lo, hi;   // hi: the input's upper half, then the output's
  VR_HD uint64_t in() const { return join48(hi & 0xffffu, in_lo); }
  VR_HD uint64_t out() const { return join48(hi >> 16, out_lo); }
};
template <int N>
struct GroupArgs {
  RankPtrs rank[N];       // of the segment's first byte of chunk 0
  uint32_t pitch_lo;      // bytes per rank-chunk (all-gather: of one slice): lower 32 bits
  uint32_t seg;           // bytes of every chunk the launch covers; bit 31: head mask / 8 (0 where
                          // every chunk starts on a line: the kernels for that take the word as it is)
  uint32_t status_lo;     // address / 256 of the time-out word, lower 32 bits
  uint32_t rest;          // bits 0-7: upper ones of that address; 8-16: of the pitch; 17-26 and 27-31: spin
                          // limit, 10 significant bits and how far they are shifted up; the all-gather,
                          // which waits for no flag, has there what run_code forms
  VR_HD uint64_t pitch() const { return join48(rest >> 8 & 511u, pitch_lo); }
  // place of the first output in its KiB, and the head mask from bit 8 on (wire_span)
  VR_HD uint32_t lines() const { return (rank[0].out_lo & 1023u) | seg >> 31 << 11; }
  static VR_HD uint64_t status_address(uint32_t rest, uint32_t status_lo) { return join48(rest & 255u, status_lo) << 8; }
  static VR_HD uint32_t spin_limit(uint32_t rest) { return (rest >> 17 & 0x3ffu) << (rest >> 27); }
  VR_HD uint32_t run_log2() const { return rest >> 17 & 7u; }
  VR_HD uint32_t run_cols() const { return (rest >> 20) << (3 + run_log2()); }
};
static_assert(sizeof(GroupArgs<8>) <= kCheapArgBytes, "a launch's arguments cost the host more beyond");

// The spin limit's bits of GroupArgs::rest: rounded up to 10 significant bits (limits below 1024,
// and the default, a power of two, stay what they are).
inline uint32_t spin_code(uint32_t limit) {
  uint32_t shift = 0;
  uint64_t m = limit;
  while (m > 0x3ffu) m = (m + 1) / 2, ++shift;
  if (m << shift > 0xffffffffull) --shift, m = 0x3ffu;   // 2^32 would not come out of the shift
  return (uint32_t)m << 17 | shift << 27;
}

// The all-gather's bits of GroupArgs::rest: log2 of the work-groups in a row on an XCD, at most 7,
// and how many groups of 8 * run work-groups a row of `cols` holds (as many as 12 bits say; the
// others stay in their order).
inline uint32_t run_code(int run, uint32_t cols) {
  uint32_t log2 = 0;
  while (log2 < 7 && (2 << log2) <= run) ++log2;
  const uint32_t groups = cols >> (3 + log2);
  return log2 << 17 | (groups < 4095u ? groups : 4095u) << 20;
}

// The launch that covers [off, off + seg) of every chunk.  `status` is the start of an allocation,
// a multiple of 256.
template <int N>
GroupArgs<N> group_args(void *const in[], void *const out[], size_t pitch, size_t off, size_t seg, uint32_t head_mask,
                        uint32_t spin_limit, const void *status) {
  GroupArgs<N> a;
  for (int k = 0; k < N; ++k) {
    const uint64_t p = (uint64_t)(uintptr_t)in[k] + off, q = (uint64_t)(uintptr_t)out[k] + off;
    a.rank[k].in_lo = (uint32_t)p;
    a.rank[k].out_lo = (uint32_t)q;
    a.rank[k].hi = ((uint32_t)(p >> 32) & 0xffffu) | (uint32_t)(q >> 32) << 16;
  }
  const uint64_t word = (uint64_t)(uintptr_t)status >> 8;
  a.pitch_lo = (uint32_t)pitch;
  a.seg = (uint32_t)seg | (head_mask ? 1u : 0u) << 31;
  a.status_lo = (uint32_t)word;
  a.rest = ((uint32_t)(word >> 32) & 255u) | ((uint32_t)((uint64_t)pitch >> 32) & 511u) << 8 | spin_code(spin_limit);
  return a;
}

}  // namespace vr
