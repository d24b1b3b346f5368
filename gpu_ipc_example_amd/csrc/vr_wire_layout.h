// Sink geometry of the wire transport: which message slot of a rank's scatter or
// gather sink a wave touches, for every flow.  The kernels (vr_wire.hip), the host
// code that sizes the scratch (vr_wire_host.cpp) and a CPU bounds test all use these
// same functions, so a sink can be proven large enough without a GPU.
//
// A sink is `slots` message slots of kSlotBytesMax bytes followed by `slots`
// 32-bit flag words (used only by the fenced flag-word format).  A rank's scratch
// is its scatter sink followed by its gather sink, the shape of the reference's
// one allocation ipcbuf0 | ipcbuf1 (main.cpp:241-243).
#pragma once

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define VR_HD __host__ __device__ constexpr
#else
#define VR_HD constexpr
#endif

namespace vr {
namespace wl {

constexpr uint32_t kSlotBytesMax = 2048;        // largest message any format stores per wave and step
constexpr uint32_t kSimplePerSection = 1024;    // messages per sender section of SimpleTransmit
                                                // (2 MiB of 2 KiB messages, simple_transmit.hpp:11)
constexpr int kSlotsFlat = 8;                   // nSlot of ParallelTransmit / BisectPTransmit
constexpr int kSlotsRing = 4;                   // nSlot of SequentialTransmit / RingTransmit

enum Flow : int { PARALLEL, SEQUENTIAL, RING, BISECT, ALLGATHER, SIMPLE, FLOW_COUNT };

// ---- slot index of a message ------------------------------------------------------------
// ParallelTransmit: sink entry (x_id + sender), ring of 8 slots per entry
// (parallel_transmit.hpp:47-58, 93).
VR_HD uint32_t parallel_slot(uint32_t x_id, int sender, uint32_t s) {
  return (x_id + (uint32_t)sender) * kSlotsFlat + s;
}
// SequentialTransmit / RingTransmit / ring all-gather: entry [peer][wire], 4 slots
// (sequential_transmit.hpp:69-77, 273-277).
VR_HD uint32_t ring_slot(uint32_t wpr, int peer, uint32_t wid, uint32_t s) {
  return ((uint32_t)peer * wpr + wid) * kSlotsRing + s;
}
// BisectPTransmit: close entries (wg + l) first, the far entries behind them
// (bisect_transmit.hpp:445-481).
VR_HD uint32_t bisect_close_slot(uint32_t wg, int l, uint32_t s) {
  return (wg + (uint32_t)l) * kSlotsFlat + s;
}
VR_HD uint32_t bisect_far_slot(uint32_t wpr, int half_ranks, uint32_t wid, uint32_t s) {
  return (wpr + (uint32_t)half_ranks + wid) * kSlotsFlat + s;
}
// SimpleTransmit: one section of kSimplePerSection messages per sender.
VR_HD uint32_t simple_slot(int section, uint32_t pos) {
  return (uint32_t)section * kSimplePerSection + pos;
}

// ---- slots a sink must hold ---------------------------------------------------------------
// `wpr` = wires (waves) per rank.  Exclusive upper bound of every slot index the
// flow's kernel forms for `nranks` ranks.
VR_HD size_t slots_needed(int flow, int nranks, uint32_t wpr) {
  switch (flow) {
    case PARALLEL: return (size_t)kSlotsFlat * wpr;
    case BISECT: return (size_t)kSlotsFlat * (2u * (size_t)wpr + (size_t)nranks / 2);
    case SIMPLE: return (size_t)nranks * kSimplePerSection;
    default: return (size_t)kSlotsRing * (size_t)nranks * wpr;
  }
}

// Largest number of wires per rank whose slot range still fits `slots` slots (the
// inverse of slots_needed; SimpleTransmit's range does not depend on the wire
// count).
VR_HD uint32_t wires_fitting(int flow, int nranks, size_t slots) {
  switch (flow) {
    case PARALLEL: return (uint32_t)(slots / kSlotsFlat);
    case BISECT: {
      const size_t entries = slots / kSlotsFlat, half = (size_t)nranks / 2;
      return entries > half ? (uint32_t)((entries - half) / 2) : 0u;
    }
    case SIMPLE: return slots >= (size_t)nranks * kSimplePerSection ? kSimplePerSection / 2 : 0u;
    default: return (uint32_t)(slots / ((size_t)kSlotsRing * (size_t)nranks));
  }
}

struct Layout {
  size_t slots;        // message slots per sink
  size_t flag_off;     // byte offset of the flag words inside a sink
  size_t sink_bytes;   // payload slots + flag words, a multiple of 256
  size_t rank_bytes;   // scatter sink + gather sink of one rank
};

// Scratch sized for every flow at up to `wpr_max` wires per rank; `with_simple`
// adds room for SimpleTransmit's sender sections.
VR_HD Layout layout_for(int nranks, uint32_t wpr_max, bool with_simple) {
  size_t slots = 0;
  for (int f = 0; f < FLOW_COUNT; ++f) {
    if (f == SIMPLE && !with_simple) continue;
    const size_t n = slots_needed(f, nranks, wpr_max);
    if (n > slots) slots = n;
  }
  const size_t flag_off = slots * kSlotBytesMax;
  const size_t sink_bytes = (flag_off + slots * sizeof(uint32_t) + 255) / 256 * 256;
  return Layout{slots, flag_off, sink_bytes, 2 * sink_bytes};
}

// ---- wires of the work-group form (vr_wire_group.hip) ------------------------------------------
// Where a lane's vectors of a wire lie in a rank's buffer.  As in the direct kernels
// (tile_start, vr_direct.hip) wires are laid on 128-byte lines of the outputs and vectors on 16
// bytes: the first wire may begin up to 112 bytes before the chunk (lanes there form offsets
// below zero, beyond the buffer's length) and its first vector may straddle the chunk's start.
// A straddling vector's upper half is what the chunk begins with; the lower half belongs to the
// chunk before, or lies ahead of the buffer.  A chunk may end inside a vector: the bounds check
// works dword by dword.
struct Span {
  size_t at;        // first byte of the buffer resource, from the start of a rank's buffer
  uint32_t bytes;   // length of the buffer resource
  uint32_t off;     // the lane's offset in it
  bool straddles;   // the vector at offset 0 begins 8 bytes below the chunk
  // Is the lane's first vector the straddling one?
  VR_HD bool half() const { return straddles && off == 0; }
  // Its load takes the 16 bytes from the chunk's start on, so that no byte outside the buffer
  // is read.  The half that counts comes, is added up (the lane does so in every rank) and is
  // stored as the lower one.  (Moved up to its place after the load instead, simple_transmit at
  // 8 x 4 MiB took 15.6 us for 14.8.)
  VR_HD uint32_t first_load() const { return half() ? 8u : off; }
};
// The chunk's bytes [base, base + seg_bytes) of each buffer; `lines` = place of the first output
// in its KiB and, as 8 << 8, whether a chunk that starts in the middle of 16 bytes does so in
// every buffer; `off` = the lane's place counted from the start of the first wire.  `lined` =
// every chunk starts on a multiple of `grain` bytes, on which wires are laid: a line, or a KiB.
VR_HD Span wire_span(bool lined, size_t base, uint32_t seg_bytes, uint32_t lines, uint32_t off, bool first_wire,
                     uint32_t grain = 128) {
  if (lined) return Span{base, seg_bytes, off, false};
  const uint32_t addr = (lines & 0x3ffu) + (uint32_t)base, head = addr & (lines >> 8 & 8u);
  return Span{base - head, seg_bytes + head, off - ((addr - head) & (grain - 16u)), first_wire && head != 0};
}

// ---- flag values ----------------------------------------------------------------------------
// May the flag values of a launch that starts at `seq` lie in the sinks already?  `next_min`
// is one more than the largest value written since they were cleared (no launch writes across
// the wrap through 0).  Receivers look for equal values, so only values above all written ones
// are safe, and above means as unsigned numbers: a counter that wrapped between two launches
// that use the sinks (in calls that use none: direct transport, messages through LDS) is far
// below, though the difference modulo 2^32 is small and positive.
VR_HD bool flags_may_repeat(uint32_t seq, uint32_t next_min) { return seq < next_min; }

}  // namespace wl
}  // namespace vr
