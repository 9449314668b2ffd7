// Gradient quant-field search (pikgpu_search_quant_field): the kernels of
// one Adam step on the log quant field, beside the quantization with the
// forward model (KSearchForward) and the adjoint (KAdjBackward, which also
// attributes the distortion below).
//
// The reference searches the field by repeated round trips judged by
// Butteraugli (FindBestQuantization, pik/adaptive_quantization.cc:677-853);
// it has no gradient. Here every step quantizes the image with the current
// integer field, decodes it with the differentiable model and back-
// propagates the squared linear-RGB error to the dequantized coefficients
// (g = dL/dd). To first order the error the quantization of block b causes
// is D_b = 1/2 sum_k g_k e_k, with e = d - x the quantization error of each
// coefficient (x the encoder's unquantized value): for L = |J d - t|^2,
// g = 2 J^T J e, so the D_b sum to e^T J^T J e, and each block's share
// carries the decode's weighting (IDCT, colour correlation, Gaborish, the
// opsin cube) of its own coefficients. Under the quantization-noise model
// D ~ step^2 ~ qf^-2, dD_b / d log qf = -2 D_b; the rate grows with
// log qf. Each transform's log field u then follows Adam on
//   G = sum over its blocks of ( -2 w_b D_b + lambda ),
// whose stationary point equalizes the weighted distortion w_b D_b across
// blocks at the level lambda sets (w: per-block perceptual weights given by
// the caller, 1 by default).
#include "kernels.h"

namespace pikgpu {

// Block i's integer field value from its transform's log field u, rounded and
// clamped to [1, qmax]; `qfr` receives it as float for the adjoint, and the
// block's dequantisation descriptors follow it. Returns its log (the rate
// proxy).
__device__ inline float RoundField(const FrameParams& P, const FrameBuffers& B,
                                   int i, float u, int qmax, int32_t* qf,
                                   float* qfr) {
  const float v = rintf(__expf(u));
  const int q = int(fminf(fmaxf(v, 1.0f), float(qmax)));
  qf[i] = q;
  qfr[i] = float(q);
  // every block of a transform has the same value
  WriteBlockDesc(P, B, i, q, q);
  return __logf(float(q));
}
// The workgroup's sum of lq to part[wg].
__device__ inline void RatePartial(float lq, int wg, float* part) {
  __shared__ float s[4];
  for (int m = 32; m >= 1; m >>= 1) lq += __shfl_xor(lq, m, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = lq;
  __syncthreads();
  if (threadIdx.x == 0) part[wg] = (s[0] + s[1]) + (s[2] + s[3]);
}

// First block of block i's transform.
struct FirstOf {
  int x, y, size;  // first block, covered blocks per side
};
__device__ inline FirstOf FirstBlockOf(const FrameParams& P,
                                       const FrameBuffers& B, int i) {
  const uint8_t a = B.acs[i];
  FirstOf f;
  f.size = AcsCovered(a >> 4);
  const int idx = a & 15, y = i / P.bx, x = i - y * P.bx;
  f.y = y - idx / f.size;
  f.x = x - idx % f.size;
  return f;
}

// The integer field of the initial log field.
__global__ void __launch_bounds__(256)
    KSearchRound(FrameParams P, FrameBuffers B, const float* u, int qmax,
                 int32_t* qf, float* qfr, float* part) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  float lq = 0.0f;
  if (i < P.bx * P.by) {
    const FirstOf f = FirstBlockOf(P, B, i);
    lq = RoundField(P, B, i, u[f.y * P.bx + f.x], qmax, qf, qfr);
  }
  RatePartial(lq, blockIdx.x, part);
}

// One Adam step (step number t >= 1) on each transform's log field and the
// integer field of the result: gradient sum over the transform's blocks of
// -2 w D + lambda; u clamped to [ulo, uhi] and to the trust region [u0 + dlo,
// u0 + dhi] around its initial value u0. Every block of a transform computes
// its step from the old state (at the first block), so that the rounding
// needs no other block's result, and the first block keeps it; the last two
// workgroups sum the partials of the evaluation before. An update, a
// rounding and two sums of their own took 20 us in four launches, this 7 us
// (1024x1024 image); a step with the distortion in KAdjBackward and the
// forward model in KSearchForward 64 us (31 + 26 + 7) instead of 98.
__global__ void __launch_bounds__(256)
    KSearchStep(FrameParams P, FrameBuffers B, SearchArgs S, int t,
                const float* dist, const float* u0, SearchState from,
                SearchState to, int qmax, int32_t* qf, float* qfr,
                float* rate_part, SearchSums sums) {
  const int groups = int(gridDim.x) - 2;
  if (int(blockIdx.x) >= groups) {
    if (int(blockIdx.x) == groups) {
      SumPartials(sums.loss_part, sums.loss_n, sums.loss);
    } else {
      SumPartials(sums.rate_part, sums.rate_n, sums.rate);
    }
    return;
  }
  const int i = blockIdx.x * 256 + threadIdx.x;
  float lq = 0.0f;
  if (i < P.bx * P.by) {
    const FirstOf f = FirstBlockOf(P, B, i);
    const int i0 = f.y * P.bx + f.x;
    float g = 0.0f;
    for (int iy = 0; iy < f.size; ++iy) {
      for (int ix = 0; ix < f.size; ++ix) {
        const int j = (f.y + iy) * P.bx + f.x + ix;
        const float w = S.weight ? S.weight[j] : 1.0f;
        g += *S.lambda - 2.0f * w * dist[j];
      }
    }
    const float mi = S.beta1 * from.m[i0] + (1.0f - S.beta1) * g;
    const float vi = S.beta2 * from.v[i0] + (1.0f - S.beta2) * g * g;
    const float mh = mi / (1.0f - powf(S.beta1, float(t)));
    const float vh = vi / (1.0f - powf(S.beta2, float(t)));
    const float ui = from.u[i0] - S.lr * mh / (sqrtf(vh) + S.eps);
    const float lo = fmaxf(S.ulo, u0[i0] + S.dlo);
    const float hi = fminf(S.uhi, u0[i0] + S.dhi);
    const float u = fminf(fmaxf(ui, lo), hi);
    if (i == i0) {
      to.m[i] = mi;
      to.v[i] = vi;
      to.u[i] = u;
    }
    lq = RoundField(P, B, i, u, qmax, qf, qfr);
  }
  RatePartial(lq, blockIdx.x, rate_part);
}

// The rate weight: `fixed` when positive, else kappa times the mean over
// the blocks of 2 w_b D_b (one workgroup).
__global__ void __launch_bounds__(256)
    KSearchLambda(const float* dist, const float* weight, int n, float fixed,
                  float kappa, float* out) {
  __shared__ double s[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) {
    acc += 2.0 * double(weight ? weight[i] : 1.0f) * double(dist[i]);
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *out = fixed > 0.0f ? fixed : float(kappa * s[0] / double(n > 0 ? n : 1));
  }
}

// Initial state: u = u0 = log of the frame's integer field, Adam moments
// zero.
__global__ void __launch_bounds__(256)
    KSearchInit(FrameParams P, FrameBuffers B, float* u0, float* u, float* m,
                float* v) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.bx * P.by) return;
  u[i] = __logf(float(B.qf[i]));
  u0[i] = u[i];
  m[i] = 0.0f;
  v[i] = 0.0f;
}

}  // namespace pikgpu
