// Wire transport, launches that hold all ranks: messages through a compute unit's LDS.
//
// The waves of one wire column talk to nobody but each other: one wave per rank,
// N waves.  When a launch holds all N ranks those N waves are made ONE work-group,
// so they share a compute unit and its LDS, and the sinks of the column's ranks
// live there: message slots at work-group scope, no scratch in device memory, no
// polling across the chip, no co-residency demand on the grid.  Every wave loads its
// own rank's input only and stores its own rank's output only; between them the messages
// are scattered, added up in the protocol's order and gathered.
// Launches that hold some of the ranks keep their sinks in memory (vr_wire.hip).
//
// Two forms.  The all-to-all protocols (and, without the sums, the all-gather) are two steps
// at most that all waves of the column take together, so the work-group's barrier says that
// the messages are there.  RingTransmit's hops wait for one neighbour each, which a flag
// word per rank says.  Its polls are bounded as in vr_wire.hip: after `spin_limit`
// unsuccessful polls (or once another wave has given up) a wave records a time-out in the
// status word and runs to its end without waiting again.
//
// What bounds it: HBM, like the direct transport.  Messages through memory cost 2.75
// times the algorithmic bytes at the L2 / fabric boundary, which carries about
// 8 TB/s however much of it the memory-side cache serves; here only inputs and
// outputs cross it.  ParallelTransmit, 8 ranks in place: 256 MiB per rank 2196 us through memory,
// 670 us (6.4 TB/s); RingTransmit, 4 x 8 MB: 39.4, 10.7 us; all-gather, 8 x 1 MB: 51.6, 11.8 us.
// Small launches are bound by the chain from a wave's load to its store.  With flag words for
// every message, the owner's N - 1 additions in one wave and a copy of the sum for each peer it was
// longer: parallel, 8 x 1 MiB bfloat16 4.62 us, now 3.72, of 64 bytes less 5.51, now 3.93; 8 x 8 MiB less
// 64 28.5, now 24.7; simple_pcie, 8 x 5 MB 16.6, now 12.9; small, 8 x 1.9 MB out of place 6.8, now 6.2.
//
// One wire per work-group and no loop: the hardware starts work-groups in index
// order, so a launch sweeps the chunks front to back with all compute units close
// together (as the direct transport's one-trip grids).  A wave's message is U x 16
// bytes per lane; the host picks U and the cache policies (group_plan).

#include "vr_internal.h"

namespace vr {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Cache policies of the accesses to inputs and outputs (see vr_direct.hip).
constexpr int kStreamLoad = 2;        // nt
constexpr int kStreamStore = 2 | 16;  // nt sc1

struct Poll {
  uint32_t limit;
  __attribute__((address_space(1))) uint32_t *status;   // (device memory) non-zero once any poll gave up
  bool dead;
  // Before the first wait: the limit and the time-out word out of the arguments, not sooner than
  // here (ahead of a wave's first load, where the compiler likes to put it, it delays the load).
  template <int N>
  __device__ __forceinline__ void arm(const GroupArgs<N> &a) {
    uint32_t rest = a.rest;
    asm volatile("" : "+s"(rest));
    limit = a.spin_limit(rest);
    status = reinterpret_cast<__attribute__((address_space(1))) uint32_t *>(a.status_address(rest, a.status_lo));
    dead = false;
  }
  // Waits until `ready` holds in every lane.
  template <typename F>
  __device__ __forceinline__ void until(F &&ready) {
    if (dead) return;
    uint32_t polls = 0;
    while (!__all(ready())) {
      ++polls;
      if (polls >= limit || ((polls & 63u) == 0 &&
                             __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        dead = true;
        __hip_atomic_store(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
};

// One message: U x 16 bytes per lane.
template <int U>
struct Msg {
  u32x4 d[U];
};

// Where a chunk lies in every rank's buffer (wl::wire_span), by what chunks are known to start
// on.  GRAIN: what wires are laid on, KiBs (parallel, 8 x 8 MiB less 64 bytes on 128-byte lines 28.6 us, now
// 27.1, bisect 8 x 16 MiB less 64 56.2, 54.7) or, in the ring by columns, which would have N more wires
// then, lines (4 x 8 MB 10.9 us, on KiBs 11.0).  ON_LINES: none of the arithmetic for other starts (the extra scalar instructions of eight
// waves per 8 KiB cost 7 % at 8 x 32 MiB).  ON_VECTORS: messages of 16 bytes, no vector straddles
// a start.
enum Starts : int { ON_LINES, ON_VECTORS, ON_HALVES };
template <Starts S>
struct Span : wl::Span {};
template <Starts S, int U, int GRAIN, int N>
static __device__ __forceinline__ Span<S> span_of(const GroupArgs<N> &a, uint32_t chunk, uint32_t lane, uint32_t col = blockIdx.x) {
  return {wl::wire_span(S == ON_LINES, chunk * a.pitch(), S == ON_LINES ? a.seg : a.seg & 0x7fffffffu, S == ON_LINES ? 0 : a.lines(),
                        col * (1024u * U) + lane * 16u, col == 0, GRAIN)};
}
template <Starts S>
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *base, const Span<S> &s) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(static_cast<const char *>(base) + s.at), 0, (int)s.bytes,
                                           0x00020000);
}
// Offset of the lane's vector u, added up in a register: as an immediate of the instruction
// it would be added after the wrap of a first wire's offset below zero had been compared.
template <Starts S>
static __device__ __forceinline__ uint32_t vec_off(const Span<S> &s, int u) {
  uint32_t off = s.off + (uint32_t)u * 1024u;
  if (S != ON_LINES && u) asm("" : "+v"(off));
  return off;
}
template <int U, int LD, Starts S>
static __device__ __forceinline__ Msg<U> load(const void *base, const Span<S> &s) {
  const __amdgpu_buffer_rsrc_t rs = rsrc(base, s);
  Msg<U> m;
#pragma unroll
  for (int u = 0; u < U; ++u)
    m.d[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, S == ON_HALVES && u == 0 ? s.first_load() : vec_off(s, u), 0, LD);
  return m;
}
template <int U, int ST, Starts S>
static __device__ __forceinline__ void store(void *base, const Span<S> &s, const Msg<U> &m) {
  const __amdgpu_buffer_rsrc_t rs = rsrc(base, s);
  // (a scalar branch: only a chunk's first wire has a vector that straddles its start)
  if (S == ON_HALVES && s.straddles) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u == 0 && s.off == 0)
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{m.d[0].x, m.d[0].y}, rs, 8u, 0, ST);
      else
        __builtin_amdgcn_raw_buffer_store_b128(m.d[u], rs, vec_off(s, u), 0, ST);
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) __builtin_amdgcn_raw_buffer_store_b128(m.d[u], rs, vec_off(s, u), 0, ST);
}
// v = m + v, the received message on the left (rt64_128.hpp:947-957)
template <int DT, int U>
static __device__ __forceinline__ void add(Msg<U> &v, const Msg<U> &m) {
#pragma unroll
  for (int u = 0; u < U; ++u)
    v.d[u] = __builtin_bit_cast(u32x4, vadd<DT>(__builtin_bit_cast(h8, m.d[u]), __builtin_bit_cast(h8, v.d[u])));
}

// The sinks of a column: SLOTS message slots and FLAGS flag words in LDS.
template <int U, int SLOTS, int FLAGS>
struct Sinks {
  static constexpr uint32_t kBytes = SLOTS * U * 1024u + FLAGS * 4u;
  u32x4 *slots;
  uint32_t *flags;
  uint32_t lane;
  __device__ __forceinline__ Sinks(u32x4 *lds, uint32_t lane_) : slots(lds), lane(lane_) {
    flags = reinterpret_cast<uint32_t *>(lds + SLOTS * U * 64);
    if (threadIdx.x < (uint32_t)FLAGS) flags[threadIdx.x] = 0;   // never more than the work-group has lanes
  }
  __device__ __forceinline__ void put(int slot, const Msg<U> &m) const {
#pragma unroll
    for (int u = 0; u < U; ++u) slots[(slot * U + u) * 64 + lane] = m.d[u];
  }
  __device__ __forceinline__ Msg<U> get(int slot) const {
    Msg<U> m;
#pragma unroll
    for (int u = 0; u < U; ++u) m.d[u] = slots[(slot * U + u) * 64 + lane];
    return m;
  }
  // What was put before is in the slots once the flag can be seen.
  static __device__ __forceinline__ void publish() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
  __device__ __forceinline__ void raise(int flag, uint32_t value) const {
    if (lane == 0) __hip_atomic_store(flags + flag, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ uint32_t look(int flag) const {
    return __hip_atomic_load(flags + flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
};

#define VR_GROUP_PROLOGUE                                                                    \
  extern __shared__ u32x4 lds[];                                                              \
  const uint32_t lane = threadIdx.x & 63u;                                                    \
  const int r = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));                      \
  const char *const src = reinterpret_cast<const char *>(a.rank[r].in());                      \
  char *const dst = reinterpret_cast<char *>(a.rank[r].out());                                 \
  /* every argument arrives behind one wait */                                                \
  asm volatile("" ::"s"(src), "s"(dst), "s"(a.pitch_lo), "s"(a.seg), "s"(a.status_lo), "s"(a.rest), \
               "s"(S == ON_LINES ? 0 : a.rank[0].out_lo))

// Messages written before are in LDS for every wave of the work-group after.
static __device__ __forceinline__ void meet() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---- ParallelTransmit, SequentialTransmit, SimpleTransmit, BisectPTransmit (parallel_transmit.hpp:
// 63-131, sequential_transmit.hpp:83-207, simple_transmit.hpp:16-179, bisect_transmit.hpp:286-424) ----
// Row c of the grid sweeps chunk c.  Every wave scatters its rank's message; the owner's additions,
// N - 1 of them in a row, are shared out: each wave adds up an N-th of the message, in the
// protocol's order, into the first slot, which all waves gather from.
template <int N, int ORDER>
static __device__ __forceinline__ int operand_of(int r, int c) {   // rank r's place in chunk c's order
  if constexpr (ORDER == ORDER_ROTATED) return (r - c) & (N - 1);  // rank c, c + 1, ...
  // pairs l, l + 1, ...; in each the rank of the half's parity first, then its pair's message
  constexpr int B = N / 2;
  const int h = c / B, l = c & (B - 1);
  return 2 * (((r >> 1) - l) & (B - 1)) + ((r & 1) ^ h);
}

template <int N, int ORDER, int DT, int U, Starts S, int LD, int ST>
__global__ __launch_bounds__(64 * N) void k_group_exchange(GroupArgs<N> a) {
  VR_GROUP_PROLOGUE;
  // A wave's share of the sums: an N-th of the message, but no less than 4 bytes a lane; waves
  // without one wait.  (Shared out among all waves, 8 or 16 of 64 lanes with work to do, the
  // additions of 16 ranks bound the launch: bisect, 16 x 12 MB bfloat16 82 us, so 67.)
  constexpr int kMsg = U * 1024, kShare = kMsg / N >= 256 ? kMsg / N : 256;   // bytes
  constexpr int W = kShare >= 1024 ? 16 : kShare / 64;                         // bytes a lane adds up at once
  typedef _Float16 V __attribute__((ext_vector_type(W / 2)));
  const int c = (int)blockIdx.y;
  const auto at = span_of<S, U, 1024>(a, c, lane);
  Msg<U> v = load<U, LD>(src, at);
  u32x4 *const own = lds + operand_of<N, ORDER>(r, c) * (U * 64) + lane;
#pragma unroll
  for (int u = 0; u < U; ++u) own[u * 64] = v.d[u];
  meet();
  if (kShare * N <= kMsg || r < kMsg / kShare) {
    char *const share = reinterpret_cast<char *>(lds) + r * kShare + lane * W;
#pragma unroll
    for (int i = 0; i < kShare; i += 64 * W) {
      V x[N];
#pragma unroll
      for (int k = 0; k < N; ++k) x[k] = *reinterpret_cast<const V *>(share + i + k * kMsg);
      // the received message is the left operand (rt64_128.hpp:947-957)
      V sum;
      if constexpr (ORDER == ORDER_ROTATED) {
        sum = x[0];
#pragma unroll
        for (int k = 1; k < N; ++k) sum = vadd<DT>(x[k], sum);
      } else {
        sum = vadd<DT>(x[1], x[0]);
#pragma unroll
        for (int k = 2; k < N; k += 2) sum = vadd<DT>(vadd<DT>(x[k + 1], x[k]), sum);
      }
      *reinterpret_cast<V *>(share + i) = sum;
    }
  }
  meet();
#pragma unroll
  for (int u = 0; u < U; ++u) v.d[u] = lds[u * 64 + lane];
  store<U, ST>(dst, at, v);
}

// ---- all-gather (sequential_transmit.hpp:429-516 without the sums, its hops one) --------------------
// Row p of the grid sweeps rank p's slice: p's wave sends the message, every wave stores it.
template <int N, int U, Starts S, int LD, int ST>
__global__ __launch_bounds__(64 * N) void k_group_allgather(GroupArgs<N> a) {
  VR_GROUP_PROLOGUE;
  const int p = (int)blockIdx.y;
  // Consecutive work-groups run on consecutive XCDs, so XCD k gets every eighth KiB.  With runs, the
  // work-groups of each group of 8 * run are permuted so that it gets `run` KiB in a row (the
  // ragged last group of a slice stays as it is).
  uint32_t col = blockIdx.x;
  const uint32_t run_log2 = a.run_log2(), group = 8u << run_log2, first = col & ~(group - 1u);
  if (run_log2 && first + group <= a.run_cols()) {
    const uint32_t k = col & (group - 1u);
    col = first + ((k & 7u) << run_log2) + (k >> 3);
  }
  const auto at = span_of<S, U, 1024>(a, p, lane, col);
  // the input is one slice long: the same bytes of it as of the own slot
  const char *slot0 = src - (size_t)r * a.pitch();
  Msg<U> v;
  if (r == p) {
    v = load<U, LD>(slot0, at);
#pragma unroll
    for (int u = 0; u < U; ++u) lds[u * 64 + lane] = v.d[u];
  }
  meet();
  if (r != p) {
#pragma unroll
    for (int u = 0; u < U; ++u) v.d[u] = lds[u * 64 + lane];
  } else if (slot0 == dst) {
    return;   // the own slot needs no store when it is the input (sequential_transmit.hpp:496-497)
  }
  store<U, ST>(dst, at, v);
}

// ---- RingTransmit (sequential_transmit.hpp:429-516) --------------------------------------
// Row c of the grid sweeps chunk c.  Rank c sends its message, ranks c + 1, c + 2, ... each add theirs
// and send on; the last one's sum lies in a slot that all ranks gather from (the reference
// forwards it rank by rank).  Slot k holds what the rank of place k sent, flag k says so.
// For sizes where a launch is bound by its start or by HBM (group_plan).
template <int N, int DT, int U, Starts S, int LD, int ST>
__global__ __launch_bounds__(64 * N) void k_group_ring(GroupArgs<N> a) {
  VR_GROUP_PROLOGUE;
  Poll poll;
  const Sinks<U, N, N> sk(lds, lane);
  const int c = (int)blockIdx.y, place = operand_of<N, ORDER_ROTATED>(r, c);
  const auto at = span_of<S, U, 1024>(a, c, lane);
  Msg<U> v = load<U, LD>(src, at);
  meet();   // all flag words are zero from here on
  poll.arm(a);
  if (place > 0) {
    poll.until([&] { return sk.look(place - 1) != 0; });
    add<DT, U>(v, sk.get(place - 1));
  }
  sk.put(place, v);
  sk.publish();
  sk.raise(place, 1);
  if (place < N - 1) {
    poll.until([&] { return sk.look(N - 1) != 0; });
    v = sk.get(N - 1);
  }
  store<U, ST>(dst, at, v);
}

// The same with all N chunks of a column in one work-group: the hops of the N rings overlap.
// A rank's sink is a ring of slots fed by its predecessor; flag r counts the messages
// delivered to rank r, N - 1 of them; finished sums lie in one slot each.  With N slots a rank no
// message comes into a used slot, and the last is the sum's.  Where N slots of U KiB a rank would
// take the room of too many work-groups, two slots, and flag N + r counts the messages rank r has
// taken out, which its predecessor looks at before it reuses one: two LDS round trips more of
// three a hop (8 x 256 KiB 7.3 us with two slots, 5.9 with N; without forwarding the sums 5.5).
template <int N, int U>
struct RingSinks : Sinks<U, N * (N * U <= 8 ? N : 3), 3 * N> {
  static constexpr int kDepth = N * U <= 8 ? N : 2;
  using Sinks<U, N * (N * U <= 8 ? N : 3), 3 * N>::Sinks;
};

template <int N, int U>
struct Ring {
  static constexpr int kDepth = RingSinks<N, U>::kDepth;
  const RingSinks<N, U> &sk;
  Poll &poll;
  int r, next;
  __device__ __forceinline__ void send(int k, const Msg<U> &m) const {
    if (kDepth < N && k >= kDepth) poll.until([&] { return sk.look(N + next) >= (uint32_t)(k - kDepth + 1); });
    sk.put(next * kDepth + k % kDepth, m);
    sk.publish();
    sk.raise(next, (uint32_t)(k + 1));
  }
  __device__ __forceinline__ Msg<U> recv(int k) const {
    poll.until([&] { return sk.look(r) >= (uint32_t)(k + 1); });
    const Msg<U> m = sk.get(r * kDepth + k % kDepth);
    if constexpr (kDepth < N) {
      sk.publish();
      sk.raise(N + r, (uint32_t)(k + 1));
    }
    return m;
  }
  static __device__ __forceinline__ int sum_slot(int q) { return kDepth == N ? q * N + N - 1 : N * kDepth + q; }
  __device__ __forceinline__ void send_sum(const Msg<U> &m) const {
    sk.put(sum_slot(r), m);
    sk.publish();
    sk.raise(2 * N + r, 1);
  }
  __device__ __forceinline__ Msg<U> recv_sum(int q) const {
    poll.until([&] { return sk.look(2 * N + q) != 0; });
    return sk.get(sum_slot(q));
  }
};

template <int N, int DT, int U, Starts S, int LD, int ST>
__global__ __launch_bounds__(64 * N) void k_group_ring_columns(GroupArgs<N> a) {
  VR_GROUP_PROLOGUE;
  Poll poll;
  const RingSinks<N, U> sk(lds, lane);
  Msg<U> x[N];                                             // x[i]: chunk of rank r - i
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = load<U, LD>(src, span_of<S, U, 128>(a, (r + N - i) % N, lane));
  const Ring<N, U> ring{sk, poll, r, (r + 1) % N};
  meet();   // all waves' flag words are zero from here on
  poll.arm(a);
  ring.send(0, x[0]);
#pragma unroll
  for (int i = 1; i < N; ++i) {                            // reduce and forward; the last is the sum
    add<DT, U>(x[i], ring.recv(i - 1));
    if (i < N - 1) ring.send(i, x[i]);
  }
  ring.send_sum(x[N - 1]);
  store<U, ST>(dst, span_of<S, U, 128>(a, (r + 1) % N, lane), x[N - 1]);
#pragma unroll
  for (int i = 1; i < N; ++i)                              // the others' sums, the neighbour's first
    store<U, ST>(dst, span_of<S, U, 128>(a, (r + 1 + N - i) % N, lane), ring.recv_sum((r + N - i) % N));
}

#undef VR_GROUP_PROLOGUE

struct Pick {
  const void *fn;
  uint32_t rows, lds;   // rows of the grid, bytes of LDS the sinks take
};

template <int N, int DT, int LD, int ST, int U, bool LINED>
Pick pick_flow(WireFlow flow, bool columns) {
  constexpr Starts kWhole = LINED ? ON_LINES : ON_VECTORS, kAny = LINED ? ON_LINES : ON_HALVES;
  constexpr uint32_t kSlots = N * U * 1024u;
  if constexpr (N <= 8) {
    switch (flow) {
      case WIRE_PARALLEL:
      case WIRE_SEQUENTIAL:
      case WIRE_SIMPLE:
        if constexpr (U <= (N == 8 ? 4 : 1))
          return {reinterpret_cast<const void *>(&k_group_exchange<N, ORDER_ROTATED, DT, U, kAny, LD, ST>), N, kSlots};
        break;
      case WIRE_RING:
        if (columns) {
          if constexpr (N >= 4 && U <= (N == 8 ? 2 : 1))
            return {reinterpret_cast<const void *>(&k_group_ring_columns<N, DT, U, LINED ? ON_LINES : ON_VECTORS, LD, ST>), 1, RingSinks<N, U>::kBytes};
        } else if constexpr (U <= (N >= 4 ? 2 : 1)) {
          return {reinterpret_cast<const void *>(&k_group_ring<N, DT, U, kWhole, LD, ST>), N, kSlots + N * 4u};
        }
        break;
      case WIRE_ALLGATHER:   // no adds: one instantiation serves both element types
        return {reinterpret_cast<const void *>(&k_group_allgather<N, U, kWhole, LD, ST>), N, U * 1024u};
      default: break;
    }
  }
  if constexpr (N >= 4 && U <= (N == 8 ? 4 : N == 16 ? 2 : 1)) {
    if (flow == WIRE_BISECT)
      return {reinterpret_cast<const void *>(&k_group_exchange<N, ORDER_BISECT, DT, U, kAny, LD, ST>), N, kSlots};
  }
  return {nullptr, 0, 0};
}

template <int DT, int LD, int ST, bool LINED, int U>
Pick pick_ranks(WireFlow flow, int nranks, bool columns) {
  switch (nranks) {
    case 2: return pick_flow<2, DT, LD, ST, U, LINED>(flow, columns);
    case 4: return pick_flow<4, DT, LD, ST, U, LINED>(flow, columns);
    case 8: return pick_flow<8, DT, LD, ST, U, LINED>(flow, columns);
    case 16: return pick_flow<16, DT, LD, ST, U, LINED>(flow, columns);
    default: return {nullptr, 0, 0};
  }
}

template <int DT, int LD, int ST, bool LINED>
Pick pick_unroll(WireFlow flow, int nranks, int unroll, bool columns) {
  return unroll == 4   ? pick_ranks<DT, LD, ST, LINED, 4>(flow, nranks, columns)
         : unroll == 2 ? pick_ranks<DT, LD, ST, LINED, 2>(flow, nranks, columns)
                       : pick_ranks<DT, LD, ST, LINED, 1>(flow, nranks, columns);
}

template <int LD, int ST>
Pick pick_type(WireFlow flow, int nranks, DType dtype, int unroll, bool lined, bool columns) {
  if (lined)
    return dtype == DT_BF16 ? pick_unroll<DT_BF16, LD, ST, true>(flow, nranks, unroll, columns)
                            : pick_unroll<DT_F16, LD, ST, true>(flow, nranks, unroll, columns);
  return dtype == DT_BF16 ? pick_unroll<DT_BF16, LD, ST, false>(flow, nranks, unroll, columns)
                          : pick_unroll<DT_F16, LD, ST, false>(flow, nranks, unroll, columns);
}

}  // namespace

hipError_t launch_wire_group(hipStream_t s, const DeviceInfo &dev, WireFlow flow, int nranks, DType dtype,
                             const PtrTable &in, const PtrTable &out, size_t chunk_bytes, const GroupPlan &plan,
                             uint32_t spin_limit, uint32_t *status) {
  // what wires are laid on (span_of)
  const uint32_t grain = plan.columns ? 128u : 1024u;
  const bool lined = (((uintptr_t)out.p[0] | chunk_bytes) & (grain - 1u)) == 0;
  const Pick k =
      plan.policy == GROUP_STREAM     ? pick_type<kStreamLoad, kStreamStore>(flow, nranks, dtype, plan.unroll, lined, plan.columns)
      : plan.policy == GROUP_RESIDENT ? pick_type<0, 0>(flow, nranks, dtype, plan.unroll, lined, plan.columns)
                                      : pick_type<0, kStreamStore>(flow, nranks, dtype, plan.unroll, lined, plan.columns);
  if (!k.fn) return hipErrorInvalidValue;
  const size_t wire = 1024u * (size_t)plan.unroll;   // payload of one wave
  uint32_t lds = k.lds;
  const uint32_t cap = lds_cap_bytes(dev, plan.wgs_per_cu);
  if (cap > lds) lds = cap;
  if (hipError_t e = allow_dynamic_lds(k.fn, dev, lds); e != hipSuccess) return e;
  // (0 where every chunk starts on a line: those kernels take GroupArgs::seg as it is)
  const uint32_t head_mask =
      !lined && (flow != WIRE_RING && flow != WIRE_ALLGATHER) ? head_mask_of(nranks, in, out) : 0u;
  const size_t seg_max = plan.segment_bytes;
  for (size_t off = 0; off < chunk_bytes; off += seg_max) {
    const size_t seg = chunk_bytes - off < seg_max ? chunk_bytes - off : seg_max;
    const dim3 grid((uint32_t)((seg + (lined ? 0 : grain - 8) + wire - 1) / wire), k.rows), block(64u * (uint32_t)nranks);
    hipEvent_t ev0 = off == 0 ? tl_kernel_events.start : nullptr;
    hipEvent_t ev1 = off + seg >= chunk_bytes ? tl_kernel_events.stop : nullptr;
    hipError_t e = hipErrorInvalidValue;
    switch (nranks) {
#define VR_CASE(NN)                                                                                            \
  case NN: {                                                                                                   \
    GroupArgs<NN> a = group_args<NN>(in.p, out.p, chunk_bytes, off, seg, head_mask, spin_limit, status);       \
    if (flow == WIRE_ALLGATHER) a.rest = (a.rest & 0x1ffffu) | run_code(plan.run, grid.x);                     \
    void *kargs[] = {&a};                                                                                      \
    e = launch_kernel(k.fn, grid, block, kargs, lds, s, ev0, ev1);                                             \
    break;                                                                                                     \
  }
      VR_CASE(2)
      VR_CASE(4)
      VR_CASE(8)
      VR_CASE(16)
#undef VR_CASE
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace vr
