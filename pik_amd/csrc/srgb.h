// The 8-bit sRGB output's transfer function (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pikgpu {

// Linear sample in [0, 255] -> 8-bit sRGB before truncation: the sRGB
// transfer function (IEC 61966-2-1) of the [0, 1]-scaled value, clamped to
// [0, 1], times 255 and rounded as the reference's external-image conversion
// does (CastClip01 and ToExternal, pik/external_image.cc:190-197, 666-696).
__device__ inline float Srgb8Scaled(float linear255) {
  const float v = linear255 * (1.0f / 255);
  float e = v <= 0.0031308f ? 12.92f * v
                            : 1.055f * powf(v, 1.0f / 2.4f) - 0.055f;
  e = fminf(fmaxf(e, 0.0f), 1.0f);
  return e * 255.0f + 0.5f;
}
// The same by the hardware's log2 and exp2 (about 1 ulp each).
__device__ inline float Srgb8Fast(float linear255) {
  const float v = linear255 * (1.0f / 255);
  float e = v <= 0.0031308f
                ? 12.92f * v
                : 1.055f * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(v) *
                                                  (1.0f / 2.4f)) -
                      0.055f;
  e = fminf(fmaxf(e, 0.0f), 1.0f);
  return e * 255.0f + 0.5f;
}
// Three samples at once: r | g << 8 | b << 16. powf is some 100
// instructions, so it runs only where it decides: Srgb8Fast lies within
// 4.6e-5 of Srgb8Scaled, and its integer part is the byte unless it lies
// within 1/4096 of the next one (tests/test_gpu_device_check.py compares both
// over all 2^32 floats). KFinal of a 4096 x 4096 frame with this output
// alone: 180 us with powf and one store per byte, 84 us so.
__device__ inline uint32_t Srgb8x3(const float (&linear255)[3]) {
  float s[3];
  bool near_edge = false;
  for (int c = 0; c < 3; ++c) {
    s[c] = Srgb8Fast(linear255[c]);
    near_edge |= fabsf(s[c] - rintf(s[c])) < 1.0f / 4096;
  }
  if (near_edge) {
    for (int c = 0; c < 3; ++c) s[c] = Srgb8Scaled(linear255[c]);
  }
  return uint32_t(s[0]) | (uint32_t(s[1]) << 8) | (uint32_t(s[2]) << 16);
}

}  // namespace pikgpu
