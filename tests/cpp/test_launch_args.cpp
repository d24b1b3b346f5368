// CPU check of the kernels' packed arguments (vr_launch_args.h): what the host puts in comes out
// as it was, at the ends of every field's range.  No GPU, no library: plain g++.
#include <stdio.h>

#include <initializer_list>

#include "vr_launch_args.h"

using namespace vr;

static int failures = 0;
#define EXPECT(cond)                                                         \
  do {                                                                       \
    if (!(cond)) {                                                           \
      if (failures < 20) printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
      ++failures;                                                            \
    }                                                                        \
  } while (0)

// addresses of device memory: up to 48 bits, any multiple of 8
static void *address(int k, uint64_t base) { return (void *)(uintptr_t)(base - 8ull * 0x123456789ull * (unsigned)k); }

template <int N>
static void check(uint64_t in_base, uint64_t out_base, size_t pitch, size_t off, size_t seg, uint32_t head, uint32_t spin) {
  void *in[N], *out[N];
  for (int k = 0; k < N; ++k) in[k] = address(k, in_base), out[k] = address(k, out_base);
  for (int block : {64, 1024})
    for (uint32_t run : {0u, 8u}) {
      const uint32_t deal = N == 16 ? 4u : N == 2 ? 0u : 3u;
      const DirectArgs<N> a = direct_args<N>(in, out, pitch, off, seg, block, 0xfedcba98u, deal, run, head);
      for (int k = 0; k < N; ++k) {
        EXPECT(a.address(k) == (uintptr_t)in[k] + off);
        EXPECT(a.address(N + k) == (uintptr_t)out[k] + off);
      }
      EXPECT(a.pitch() == pitch && a.seg_bytes == seg && a.blocks_per_rank == 0xfedcba98u);
      EXPECT(a.deal_log2() == deal && a.row() == (uint32_t)block * 16u && a.run_log2() == run && a.head_mask() == head);
      EXPECT(a.place() == (((uintptr_t)out[0] + off) & 1023u));
    }
  for (uint64_t status : {(uint64_t)256, (uint64_t)0xffffffffff00, (uint64_t)0x7f1234567800}) {
    const GroupArgs<N> g = group_args<N>(in, out, pitch, off, seg, head, spin, (void *)(uintptr_t)status);
    for (int k = 0; k < N; ++k) {
      EXPECT(g.rank[k].in() == (uintptr_t)in[k] + off);
      EXPECT(g.rank[k].out() == (uintptr_t)out[k] + off);
    }
    EXPECT(g.pitch() == pitch && (g.seg & 0x7fffffffu) == seg && (head || g.seg == seg));
    EXPECT(g.lines() == ((((uintptr_t)out[0] + off) & 1023u) | head << 8));
    EXPECT(g.status_address(g.rest, g.status_lo) == status);
    const uint32_t got = g.spin_limit(g.rest);
    // rounded up to 10 significant bits, at most the largest that 32 bits hold
    const uint32_t largest = 1023u << 22;
    EXPECT(spin > largest ? got == largest : got >= spin && got - spin <= (spin < 1024 ? 0 : spin / 512));
  }
}

int main() {
  const size_t one = (size_t)1;
  for (uint64_t base : {(uint64_t)0x7ffffffffff8, (uint64_t)0xfffffffff000, (uint64_t)0x900000000000})
    for (size_t pitch : {(size_t)8, (one << 32) - 8, one << 32, one << 40})
      for (size_t off : {(size_t)0, one << 30, (one << 33) + 16})
        for (size_t seg : {(size_t)8, one << 30})
          for (uint32_t head : {0u, 8u})
            for (uint32_t spin : {1u, 64u, 1023u, 1024u, 1025u, 1u << 22, (1u << 22) + 1u, 0x7fffffffu, 0xffc00000u, 0xfffffffeu}) {
              // (the largest address plus the offset stays below 2^48)
              const uint64_t b = base - (one << 34), o = b - 0x1000000008ull;
              check<2>(b, o, pitch, off, seg, head, spin);
              check<4>(b, o, pitch, off, seg, head, spin);
              check<8>(b, o, pitch, off, seg, head, spin);
              check<16>(b, o, pitch, off, seg, head, spin);
            }
  for (int run : {1, 2, 64, 128, 256})
    for (uint32_t cols : {1u, 7u, 8u, 1023u, 1024u, 1025u, 4194304u}) {
      GroupArgs<2> g = {};
      g.rest = 0x1ffffu | run_code(run, cols);
      EXPECT(1 << g.run_log2() == (run > 128 ? 128 : run));
      const uint32_t group = 8u << g.run_log2();
      EXPECT(g.run_cols() % group == 0 && g.run_cols() <= cols && (g.run_cols() + group > cols || g.run_cols() == 4095u * group));
    }
  EXPECT(sizeof(DirectArgs<8>) == kCheapArgBytes && sizeof(GroupArgs<8>) == kCheapArgBytes);
  if (failures) {
    printf("%d failures\n", failures);
    return 1;
  }
  printf("launch arguments ok\n");
  return 0;
}
