// CPU bounds check of the wire transport's sinks: walks every (rank, wave, peer,
// slot) combination the kernels of each flow form, with the slot functions the
// kernels themselves use (vr_wire_layout.h), and proves that every message slot
// and every flag word lies inside a sink sized by the host code's layout_for().
// Then the accesses of the work-group form to inputs and outputs, and the rule by which the host clears the sinks' flag values.
// No GPU, no library: plain g++.
#include <stdio.h>

#include <initializer_list>
#include <set>
#include <vector>

#include "vr_wire_layout.h"

using namespace vr::wl;

static int failures = 0;
#define EXPECT(cond)                                                         \
  do {                                                                       \
    if (!(cond)) {                                                           \
      if (failures < 20) printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
      ++failures;                                                            \
    }                                                                        \
  } while (0)

struct Probe {
  const Layout &l;
  size_t need;      // slots_needed() of the flow under test
  size_t max_slot = 0;
  void touch(uint32_t slot) {
    if (slot > max_slot) max_slot = slot;
    EXPECT(slot < need);
    EXPECT(slot < l.slots);
    // payload of the largest format, then the slot's flag word, both inside the sink
    EXPECT(((size_t)slot + 1) * kSlotBytesMax <= l.flag_off);
    EXPECT(l.flag_off + ((size_t)slot + 1) * sizeof(uint32_t) <= l.sink_bytes);
  }
};

static void walk(int flow, int N, uint32_t wpr, const Layout &l) {
  Probe p{l, slots_needed(flow, N, wpr)};
  const int B = N / 2;
  for (int r = 0; r < N; ++r)
    for (uint32_t wid = 0; wid < wpr; ++wid) {
      switch (flow) {
        case PARALLEL: {
          const uint32_t x_id = wid / N * N;
          for (uint32_t s = 0; s < (uint32_t)kSlotsFlat; ++s)
            for (int q = 0; q < N; ++q) p.touch(parallel_slot(x_id, q, s));   // senders and owners, all peers
          break;
        }
        case SEQUENTIAL:
        case RING:
        case ALLGATHER:
          for (uint32_t s = 0; s < (uint32_t)kSlotsRing; ++s)
            for (int peer = 0; peer < N; ++peer) p.touch(ring_slot(wpr, peer, wid, s));
          break;
        case BISECT: {
          const uint32_t wg = wid / B * B;
          for (uint32_t s = 0; s < (uint32_t)kSlotsFlat; ++s) {
            for (int l2 = 0; l2 < B; ++l2) p.touch(bisect_close_slot(wg, l2, s));
            p.touch(bisect_far_slot(wpr, B, wid, s));
          }
          break;
        }
        case SIMPLE:
          // ring position of message t * wpr + wid; a power-of-two wpr keeps each
          // position with one wave
          for (uint32_t t = 0; t < 3 * kSimplePerSection / wpr + 3; ++t) {
            const uint32_t pos = (t * wpr + wid) % kSimplePerSection;
            EXPECT(pos % wpr == wid);
            for (int section = 0; section < N; ++section) p.touch(simple_slot(section, pos));
          }
          break;
      }
    }
  // the bound is tight enough to mean something: the walk reaches its last slot
  EXPECT(p.max_slot + 1 == p.need);
}

// The work-group form's loads and stores of one rank's buffer, dword by dword, as the buffer
// resources of the kernels bound them: nothing outside the buffer is touched, every dword of it
// is stored once, from the dword that was loaded for it.  `place` = the buffer's place in its
// 128-byte line, `mask` = 8 where all buffers agree about their place in 16 bytes.
static void walk_spans(int chunks, size_t pitch, size_t seg_max, uint32_t unroll, uint32_t place, uint32_t mask) {
  const bool lined = ((place | pitch) & 127u) == 0;
  const size_t total = (size_t)chunks * pitch;
  const uint32_t lines = place | mask << 8;
  std::vector<int> stored(total / 4, 0);
  for (int c = 0; c < chunks; ++c)
    for (size_t seg_off = 0; seg_off < pitch; seg_off += seg_max) {
      const size_t seg = pitch - seg_off < seg_max ? pitch - seg_off : seg_max;
      const uint32_t wires = (uint32_t)((seg + (lined ? 0 : 120) + 1024u * unroll - 1) / (1024u * unroll));
      for (uint32_t block = 0; block < wires; ++block)
        for (uint32_t lane = 0; lane < 64; ++lane) {
          const Span s = wire_span(lined, c * pitch + seg_off, (uint32_t)seg, lines, block * (1024u * unroll) + lane * 16u, block == 0);
          for (uint32_t u = 0; u < unroll; ++u) {
            const uint32_t load = u ? s.off + u * 1024u : s.first_load(), store = s.off + u * 1024u;
            long long source[4];          // the byte of the buffer each dword came from, -1: dropped
            for (uint32_t d = 0; d < 4; ++d) {
              source[d] = -1;
              if ((uint64_t)load + 4 * d + 4 > s.bytes) continue;
              source[d] = (long long)s.at + load + 4 * d;
              EXPECT(source[d] >= 0 && source[d] + 4 <= (long long)total);
            }
            const bool half = u == 0 && s.half();
            for (uint32_t d = 0; d < (half ? 2u : 4u); ++d) {
              const uint32_t offset = (half ? 8u : store) + 4 * d;
              if ((uint64_t)(half ? 8u : store) + 4 * d + 4 > s.bytes) continue;
              const long long to = (long long)s.at + offset;
              EXPECT(to >= 0 && to + 4 <= (long long)total && source[d] == to);
              if (to >= 0 && to + 4 <= (long long)total) ++stored[to / 4];
            }
          }
        }
    }
  for (int n : stored) EXPECT(n == 1);
}

// Launches that write flags [seq, seq + used) into sinks that are cleared when
// flags_may_repeat says so, at sequence numbers that other calls move on in between (and
// callers choose): no launch meets a value that is there already.
static void walk_flags(uint32_t random) {
  const uint32_t around[] = {1, 2, 40, 0x7fffffe0u, 0x80000000u, 0x80000021u, 0xffffff00u, 0xffffffd0u, 0xfffffff0u};
  std::set<uint32_t> written;
  uint32_t next_min = 0;
  bool used = false;
  for (int launch = 0; launch < 200; ++launch) {
    random = random * 1664525u + 1013904223u;
    const uint32_t seq = around[(random >> 8) % (sizeof around / sizeof *around)] + ((random >> 16) & 7u);
    const uint32_t n = 1 + ((random >> 24) & 7u);     // (never across the wrap: the host clears there)
    if (used && flags_may_repeat(seq, next_min)) {
      written.clear();
      used = false;
    }
    for (uint32_t f = seq; f < seq + n; ++f) EXPECT(written.insert(f).second);
    used = true;
    next_min = seq + n;
  }
}

int main() {
  for (uint32_t s = 1; s <= 64; ++s) walk_flags(s * 2654435761u);
  EXPECT(!flags_may_repeat(7, 7) && !flags_may_repeat(0xffffffffu, 7) && flags_may_repeat(6, 7));
  // small values, values near the end, then small ones again after a wrap
  EXPECT(!flags_may_repeat(0xfffffff0u, 4) && flags_may_repeat(3, 0xfffffff4u));
  const int ranks[] = {2, 4, 8, 16};
  int cases = 0;
  for (size_t pitch : {8u, 16u, 24u, 112u, 120u, 128u, 136u, 1016u, 1024u, 1032u, 2040u, 2048u, 2056u, 9u * 1024u + 24u})
    for (size_t seg_max : {(size_t)1 << 30, (size_t)1024, (size_t)2048})
      for (uint32_t unroll : {1u, 2u})
        for (uint32_t place = 0; place < 128; place += 8)
          for (uint32_t mask : {0u, 8u}) {
            walk_spans(3, pitch, seg_max, unroll, place, mask);
            ++cases;
          }
  for (int N : ranks)
    for (uint32_t wpr_max = 4; wpr_max <= 2048; wpr_max *= 2)
      for (int with_simple = 0; with_simple < 2; ++with_simple) {
        const Layout l = layout_for(N, wpr_max, with_simple != 0);
        EXPECT(l.sink_bytes % 256 == 0);
        EXPECT(l.rank_bytes == 2 * l.sink_bytes);
        for (int flow = 0; flow < FLOW_COUNT; ++flow) {
          if (flow == BISECT && N < 4) continue;
          if (flow == SIMPLE && !with_simple) continue;
          const uint32_t psg = flow == PARALLEL ? N : flow == BISECT ? N / 2 : 1;
          // every wire count the host may launch: multiples of psg up to wpr_max
          // (SimpleTransmit: powers of two up to half a section)
          for (uint32_t wpr = psg; wpr <= wpr_max; wpr += psg) {
            if (flow == SIMPLE && ((wpr & (wpr - 1)) || wpr > kSimplePerSection / 2)) continue;
            if (wpr > 64 && wpr != wpr_max / psg * psg && wpr % 37) continue;   // thin out the big ones
            walk(flow, N, wpr, l);
            ++cases;
          }
        }
      }
  // wires_fitting is the inverse of slots_needed: the largest wire count whose slots fit,
  // and a walk at exactly that count stays inside the sink
  for (int N : ranks)
    for (size_t slots : {64u, 1000u, 1024u, 4096u, 12288u, 100000u}) {
      Layout l = layout_for(N, 4, false);
      l.slots = slots;
      l.flag_off = slots * kSlotBytesMax;
      l.sink_bytes = (l.flag_off + slots * sizeof(uint32_t) + 255) / 256 * 256;
      for (int flow : {PARALLEL, SEQUENTIAL, RING, BISECT, ALLGATHER}) {
        if (flow == BISECT && N < 4) continue;
        const uint32_t fit = wires_fitting(flow, N, slots);
        EXPECT(fit == 0 || slots_needed(flow, N, fit) <= slots);
        EXPECT(slots_needed(flow, N, fit + 1) > slots);
        const uint32_t psg = flow == PARALLEL ? N : flow == BISECT ? N / 2 : 1;
        const uint32_t wpr = fit / psg * psg;
        if (wpr >= psg && wpr <= 4096) {
          walk(flow, N, wpr, l);
          ++cases;
        }
      }
    }
  // the fixed region of the allocation-free entry point: 8 ranks x 32 wires, no SimpleTransmit
  const Layout fixed = layout_for(8, 32, false);
  EXPECT(8 * fixed.rank_bytes + 256 <= (34u << 20));
  printf("%d layout cases, %d failures\n", cases, failures);
  return failures ? 1 : 0;
}
