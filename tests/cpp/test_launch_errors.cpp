// A kernel launch that the runtime refuses is reported by the call that made it and leaves
// nothing behind: the runtime's "last error" of the thread, which the next piece of code
// that checks its own launches would take for its own, is as it was.  CPU only: the
// runtime's entry points concerned are this program's own.
#include <stdio.h>
#include <string.h>

#include "vr_internal.h"

static hipError_t g_last = hipSuccess;
static int g_launches = 0;
static bool g_refuse = true;

static hipError_t refused() {
  ++g_launches;
  if (g_refuse) g_last = hipErrorLaunchOutOfResources;
  return g_refuse ? hipErrorLaunchOutOfResources : hipSuccess;
}

extern "C" {
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return refused(); }
hipError_t hipExtLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
  return refused();
}
hipError_t hipLaunchCooperativeKernel(const void *, dim3, dim3, void **, unsigned, hipStream_t) { return refused(); }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError(void) {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
}

static int failures = 0;
#define EXPECT(cond)                                                    \
  do {                                                                  \
    if (!(cond)) {                                                      \
      printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond);            \
      ++failures;                                                       \
    }                                                                   \
  } while (0)

using namespace vr;

int main() {
  DeviceInfo dev;
  dev.cus = 256;
  dev.lds_per_cu = 160 * 1024;
  Tuning t;
  t.block = 256;
  t.unroll = 1;
  PtrTable p;
  memset(&p, 0, sizeof p);
  const GroupPlan plan = {GROUP_MIXED, 1, 0};
  WireArgs args;
  memset(&args, 0, sizeof args);
  for (int events = 0; events < 2; ++events)
    for (int which = 0; which < 5; ++which)
      for (int refuse = 0; refuse < 2; ++refuse) {
        g_refuse = refuse != 0;
        g_launches = 0;
        g_last = hipSuccess;
        hipEvent_t ev = reinterpret_cast<hipEvent_t>(&args);
        tl_kernel_events.start = tl_kernel_events.stop = events ? ev : nullptr;
        hipError_t e = hipErrorUnknown;
        switch (which) {
          case 0: e = launch_direct_allreduce(nullptr, dev, t, 2, ORDER_ROTATED, DT_F16, p, p, 64); break;
          case 1: e = launch_direct_allgather(nullptr, dev, t, 4, p, p, 64); break;
          case 2: e = launch_wire_group(nullptr, dev, WIRE_PARALLEL, 8, DT_F16, p, p, 1024, plan, 1, nullptr); break;
          default:
            e = launch_wire(nullptr, WIRE_PARALLEL, WIRE_FMT_LL, 8, 8, 8, 256, args, which == 4, DT_F16);
            break;
        }
        EXPECT(g_launches == 1);
        EXPECT(e == (refuse ? hipErrorLaunchOutOfResources : hipSuccess));
        EXPECT(g_last == hipSuccess);
      }
  printf("launch errors: %d failures\n", failures);
  return failures ? 1 : 0;
}
