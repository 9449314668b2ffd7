// Device functions of the library called by themselves, for the GPU tests
// (libpikgpu_check.so): what no output of the public entry points shows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device.h"
#include "kernels.h"

#define HAPI extern "C" __attribute__((visibility("default")))

namespace {

using pikgpu::DeviceStamps;
using pikgpu::kEndStamps;

// Wave `slow` (of workgroup slow / 4) ends some 200 us after the others (or
// after 4096 sleeps); `latest` receives the latest clock that any wave saw
// before its stamp.
__global__ void __launch_bounds__(256)
    KStampCheck(DeviceStamps* S, unsigned long long* latest, int slow,
                unsigned long long ticks) {
  const unsigned long long t0 = wall_clock64();
  if (int(blockIdx.x * 4 + threadIdx.x / 64) == slow) {
    for (int i = 0; i < 4096 && wall_clock64() - t0 < ticks; ++i) {
      __builtin_amdgcn_s_sleep(64);
    }
  }
  if (threadIdx.x % 64 == 0) {
    atomicMax(latest, static_cast<unsigned long long>(wall_clock64()));
  }
  pikgpu::StampEnd(S->end[0], blockIdx.x);
}

}  // namespace

// A launch of `groups` workgroups whose wave `slow` ends last: the latest
// clock before a stamp, and the latest stamp of the slots. HIP's error code.
HAPI int pikgpu_check_stamps(int groups, int slow, unsigned long long* before,
                             unsigned long long* stamp) {
  if (groups < 1 || slow < 0 || slow >= 4 * groups) return 1;
  struct Mem {
    DeviceStamps stamps;
    unsigned long long latest;
  };
  int khz = 100000;
  (void)hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, 0);
  Mem* d = nullptr;
  std::vector<Mem> h(1);
  hipError_t e = hipMalloc(&d, sizeof(Mem));
  if (e != hipSuccess) return e;
  if ((e = hipMemset(d, 0, sizeof(Mem))) == hipSuccess) {
    KStampCheck<<<groups, 256>>>(&d->stamps, &d->latest, slow, khz / 5);
    if ((e = hipGetLastError()) == hipSuccess) {
      e = hipMemcpy(h.data(), d, sizeof(Mem), hipMemcpyDeviceToHost);
    }
  }
  (void)hipFree(d);
  *before = h[0].latest;
  *stamp = *std::max_element(h[0].stamps.end[0],
                             h[0].stamps.end[0] + kEndStamps);
  return e;
}
