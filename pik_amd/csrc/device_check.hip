// Device functions of the library called by themselves, for the GPU tests
// (libpikgpu_check.so): what no output of the public entry points shows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device.h"
#include "kernels.h"
#include "srgb.h"

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

// Every float pattern, 256 of them per thread: how many bytes Srgb8x3 gets
// other than Srgb8Scaled's (of any of its three samples), how many the fast
// value alone would, and the largest difference of the two values.
struct SrgbCheck {
  unsigned long long wrong, fast_wrong;
  float largest;
};
__global__ void __launch_bounds__(256) KSrgbCheck(SrgbCheck* out) {
  const uint32_t first = (blockIdx.x * 256 + threadIdx.x) * 256;
  unsigned wrong = 0, fast_wrong = 0;
  float largest = 0.0f;
  for (uint32_t i = 0; i < 256; ++i) {
    const float v = __uint_as_float(first + i);
    const float exact = pikgpu::Srgb8Scaled(v), fast = pikgpu::Srgb8Fast(v);
    // one sample beside two that no edge is near
    const float r[3] = {v, 100.0f, 100.0f}, g[3] = {100.0f, v, 100.0f},
                b[3] = {100.0f, 100.0f, v};
    const uint32_t byte = uint32_t(exact);
    const uint32_t rest = uint32_t(pikgpu::Srgb8Scaled(100.0f));
    wrong += pikgpu::Srgb8x3(r) != (byte | rest << 8 | rest << 16);
    wrong += pikgpu::Srgb8x3(g) != (rest | byte << 8 | rest << 16);
    wrong += pikgpu::Srgb8x3(b) != (rest | rest << 8 | byte << 16);
    fast_wrong += uint32_t(fast) != byte;
    largest = fmaxf(largest, fabsf(fast - exact));
  }
  for (int m = 32; m >= 1; m >>= 1) {
    wrong += __shfl_xor(wrong, m, 64);
    fast_wrong += __shfl_xor(fast_wrong, m, 64);
    largest = fmaxf(largest, __shfl_xor(largest, m, 64));
  }
  if (threadIdx.x % 64 == 0) {
    if (wrong) atomicAdd(&out->wrong, wrong);
    if (fast_wrong) atomicAdd(&out->fast_wrong, fast_wrong);
    // (floats of one sign order as integers)
    atomicMax(reinterpret_cast<int*>(&out->largest),
              __float_as_int(largest));
  }
}

}  // namespace

HAPI int pikgpu_check_srgb(unsigned long long* wrong,
                           unsigned long long* fast_wrong, float* largest) {
  SrgbCheck* d = nullptr;
  SrgbCheck h = {};
  hipError_t e = hipMalloc(&d, sizeof h);
  if (e != hipSuccess) return e;
  if ((e = hipMemcpy(d, &h, sizeof h, hipMemcpyHostToDevice)) == hipSuccess) {
    KSrgbCheck<<<65536, 256>>>(d);
    if ((e = hipGetLastError()) == hipSuccess) {
      e = hipMemcpy(&h, d, sizeof h, hipMemcpyDeviceToHost);
    }
  }
  (void)hipFree(d);
  *wrong = h.wrong;
  *fast_wrong = h.fast_wrong;
  *largest = h.largest;
  return e;
}

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
