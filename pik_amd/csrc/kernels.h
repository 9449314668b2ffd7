// Device helpers and kernel declarations of the reconstruction (gfx950).
//
// All arithmetic that feeds an integer decision later on (the EPF guide
// bytes and sigma) keeps the reference's operation order with separate
// multiplies and adds; the library is compiled with -ffp-contract=off.
#pragma once

#include "device.h"
#include "xform.h"

namespace pikgpu {

// 3x3 symmetric convolution at p of an array that holds all its neighbours, in
// the operation order of strategy::Symmetric3 (pik/convolve.h:605-621).
__device__ inline float Conv3(const float* p, int pitch, const float (&w)[3]) {
  const float* t = p - pitch;
  const float* b = p + pitch;
  const float sum_tb = t[0] + b[0];
  const float mul0 = p[0] * w[0];
  const float sum_lr = p[-1] + p[1];
  const float x1 = sum_tb + sum_lr;
  const float mul1 = x1 * w[1] + mul0;
  const float sum_t2 = t[-1] + t[1];
  const float sum_b2 = b[-1] + b[1];
  const float x2 = sum_t2 + sum_b2;
  return x2 * w[2] + mul1;
}

// 0.145f / q for an integer q != 0 with |q| <= 32768, correctly rounded: the
// hardware's reciprocal (1 ulp), one residual step in fused arithmetic. The
// generic division takes about 11 instructions to cover every exponent; for
// these 65536 quotients this gives the same bits
// (tests/test_gpu_dequant_values.py decodes every one of them). With the
// division KBlocks spent a sixth of its VALU instructions here.
__device__ inline float BiasOver(float q) {
  const float r = __builtin_amdgcn_rcpf(q);
  const float y = 0.145f * r;
  return fmaf(fmaf(-q, y, 0.145f), r, y);
}

// AdjustQuantBias, vector form (pik/quantizer.h:61-88), of an integer q.
__device__ inline float AdjustQuantBias(int c, float q) {
  const float one_bias = c == 0 ? 0.05465007330715401f
                                : (c == 1 ? 0.07005449891748593f
                                          : 0.049935103337343655f);
  const float aq = fabsf(q);
  const float big = q - BiasOver(q);
  const float one = copysignf(1 - one_bias, q);
  return aq >= 1.5f ? big : (aq >= 0.5f ? one : q);
}

// Four consecutive floats at any 4-byte aligned address, in one load.
struct __attribute__((packed, aligned(4))) Float4U {
  float v[4];
};
__device__ inline void LoadFour(const float* p, float (&v)[4]) {
  const Float4U q = *reinterpret_cast<const Float4U*>(p);
  for (int j = 0; j < 4; ++j) v[j] = q.v[j];
}

// Per-storage-block dequantisation parameters of plane c: the dequant
// matrix row of the block's strategy, position and table, the scaled
// 1 / quant field and the colour-correlation factor
// (Dequant::DoAC, pik/compressed_image.cc:636-666).
struct BlockDq {
  const float* m;
  float scaled;
  float cc;
};

// Writes block i's two dequantisation descriptors (FrameBuffers::desc), so
// the block kernels reach the dequant matrices with one dependent load
// instead of the chain strategy -> quant field -> control field -> table
// index -> table offset. qf, qfo: the quant values of the block and of its
// transform's first block.
__device__ inline void WriteBlockDesc(const FrameParams& P,
                                      const FrameBuffers& B, int i, int qf,
                                      int qfo) {
  const int bxa = i % P.bx, bya = i / P.bx;
  const uint8_t a = B.acs[i];
  const int raw = a >> 4, idx = a & 15;
  const int s = AcsCovered(raw);
  const int kind = AcsQuantKind(raw);
  const int obxa = bxa - (idx & (s - 1)), obya = bya - (idx >> (s >> 1));
  const int qt = B.dqmap[B.dcf[(bya >> 3) * P.tx + (bxa >> 3)] * 256 + qf - 1];
  const int qto =
      B.dqmap[B.dcf[(obya >> 3) * P.tx + (obxa >> 3)] * 256 + qfo - 1];
  const uint32_t* off = B.offsets + (qt * kNumQuantKinds + kind) * 3;
  const uint32_t* offo = B.offsets + (qto * kNumQuantKinds + kind) * 3;
  B.desc[2 * i] = make_uint4(
      off[0] + idx * 64, off[1] + idx * 64, off[2] + idx * 64,
      __float_as_uint(qf == 0 ? 1E10f : P.inv_global_scale / float(qf)));
  B.desc[2 * i + 1] = make_uint4(
      offo[0] + idx * 64, offo[1] + idx * 64, offo[2] + idx * 64,
      __float_as_uint(P.inv_global_scale / float(qfo)));
}

// Coefficient k of a block from its quantized value q, in Dequant::DoAC's
// operation order.
__device__ inline float DequantWith(const BlockDq& d, int c, int16_t q, int k,
                                    float yval) {
  const float mul = d.m[k] * d.scaled;
  const float v = AdjustQuantBias(c, float(q)) * mul;
  return c == 1 ? v : d.cc * yval + v;
}

// AC plane c of pass p (0: the frame's own, then pikgpu_frame_add_pass's).
__device__ inline const int16_t* AcPlane(const FrameParams& P,
                                         const FrameBuffers& B, int p, int c) {
  const size_t plane = size_t(P.by) * P.bx * 64;
  return p == 0 ? B.ac + c * plane
                : B.ac_extra + (size_t(p - 1) * 3 + c) * plane;
}

// The launch's start (by thread 0 of its first workgroup) and its end: every
// wave's, into the latest of its workgroup's slot. What a slot holds of
// earlier launches is older, so no launch clears it.
__device__ inline void StampStart(unsigned long long* at, int wg) {
  if (wg == 0 && threadIdx.x == 0) *at = wall_clock64();
}
__device__ inline void StampEnd(unsigned long long* at, int wg) {
  if ((threadIdx.x & 63) == 0) {
    atomicMax(at + wg % kEndStamps,
              static_cast<unsigned long long>(wall_clock64()));
  }
}

// Minimum and maximum over the workgroup's 256 threads, in every thread; s
// holds 8 floats of LDS that nothing else uses meanwhile. All threads call.
__device__ inline void GroupMinMax(float* lo, float* hi, float* s) {
  for (int m = 32; m >= 1; m >>= 1) {
    *lo = fminf(*lo, __shfl_xor(*lo, m, 64));
    *hi = fmaxf(*hi, __shfl_xor(*hi, m, 64));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    s[wave] = *lo;
    s[4 + wave] = *hi;
  }
  __syncthreads();
  *lo = fminf(fminf(s[0], s[1]), fminf(s[2], s[3]));
  *hi = fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7]));
}

// Sum of n partials in double by one workgroup of 256 threads.
__device__ inline void SumPartials(const float* part, int n, double* out) {
  __shared__ double s[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += double(part[i]);
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0];
}

// ---------------------------------------------------------------------------
// Cooperative transforms of the three channels of a 32x32 tile (256
// threads). The 2-D transforms are the reference's two column passes with a
// transpose in between (pik/dct.h:370-507); each line is a 1-D butterfly of
// dct1d.h computed by one thread. Every line of every transform of every
// channel is a task, and the tasks are spread over all 256 threads: a DCT8
// block has 8 line tasks, DCT16 16, DCT32 32, DCT4X4 16 (4 lines in each
// 4x4 sub-block), DCT2X2 and IDENTITY one direct task.
//
// LDS layouts (per channel):
//  * pixels and the transpose scratch: 32 rows of kTilePitch = 33 floats;
//  * coefficients: the reference's storage order (4 block rows; block bx
//    of a row holds its 64 coefficients, a DCT16/32's F matrix runs across
//    the s blocks of its s rows), with kCoefBlock = 72 floats per block.
// With power-of-two pitches the lines that neighbouring lanes read or write
// would all sit in the same LDS bank (e.g. a DCT8 column pass writing 8
// transposed rows: an 8- to 32-way conflict); the odd pixel pitch and the
// 8-float gap between blocks give the lanes of a wave distinct banks for
// the DCT8/16/32 passes.
constexpr int kTilePitch = 33;
constexpr int kTilePlane = 32 * kTilePitch;  // 1056
constexpr int kCoefBlock = 72;
constexpr int kCoefRow = 4 * kCoefBlock;     // 288
constexpr int kCoefPlane = 4 * kCoefRow;     // 1152

// Pixel (y, x) of a tile channel.
__host__ __device__ inline int PixAt(int y, int x) {
  return y * kTilePitch + x;
}
// Coefficient at storage row `row` (0..3), column `col` (block * 64 + k).
__host__ __device__ inline int CoefAt(int row, int col) {
  return row * kCoefRow + (col >> 6) * kCoefBlock + (col & 63);
}

// The tile's transforms in task order: grouped by kind (DCT32, DCT16, DCT8,
// DCT4X4, direct: the longest lines first) over all three channels, so that
// the lanes of a wave mostly run the same line code. A kind's transforms all
// have the same number of tasks, so a task's transform follows from its kind's
// first task and a shift. (Grouped by channel first, a tile of two kinds has
// each of them in most of its waves, which then run both line codes: KBlocks 246
// us instead of 226, KEpf 831 instead of 814 on a 4096x4096 frame, KAdjForward
// 50 instead of 43 at 2048x2048.)
constexpr int kTaskKinds = 5;
// log2 of the tasks of one transform, kind k in bits 4k .. 4k + 3: 32, 16, 8,
// 16 and 1
constexpr uint32_t kTaskLog2 = 0x04345;
struct TileTasks {
  int seg[kTaskKinds + 1];   // first task of each kind; the last entry: tasks
                             // of the tile
  uint32_t kind[kTaskKinds]; // tasks per channel | first position << 16 |
                             // log2 tasks << 24
  uint16_t at[16];           // raw | tile block (by * 4 + bx) << 4 of each
                             // position
  int has_dct4;              // a DCT4X4 transform is among them
};

__device__ inline int TaskKind(int raw) {
  if (raw == kDCT32) return 0;
  if (raw == kDCT16) return 1;
  if (raw == kDCT || raw == kDCTNoHF) return 2;
  if (AcsIsDCT4(raw)) return 3;
  return 4;
}

// Wave `wave` of the workgroup fills T; `acs_t` holds the tile's 16 strategy
// bytes (0xFF outside the image). hf_only keeps only strategies with HF
// prediction. Lanes 0..15 each place one block: its position is the number
// of transforms of earlier kinds plus those of its kind at earlier blocks
// (ballots). The caller's next barrier publishes T.
__device__ inline void BuildTasksWave(const uint8_t* acs_t, bool hf_only,
                                      TileTasks* T, int wave) {
  if (int(threadIdx.x >> 6) != wave) return;
  const int b = threadIdx.x & 63;
  int raw = 0, kind = kTaskKinds;
  if (b < 16) {
    const uint8_t a = acs_t[b];
    if (a != 0xFF && (a & 15) == 0 && (!hf_only || AcsPredictHF(a >> 4))) {
      raw = a >> 4;
      kind = TaskKind(raw);
    }
  }
  int seg = 0, first = 0;  // the running kind's first task and position
#pragma unroll
  for (int k = 0; k < kTaskKinds; ++k) {
    const uint32_t m = uint32_t(__ballot(kind == k));
    const uint32_t lg = (kTaskLog2 >> (4 * k)) & 15;
    if (kind == k) {
      T->at[first + __popc(m & ((1u << b) - 1))] = uint16_t(raw | (b << 4));
    }
    if (b == 0) {
      T->seg[k] = 3 * seg;
      T->kind[k] = (uint32_t(__popc(m)) << lg) | (uint32_t(first) << 16) |
                   (lg << 24);
      if (k == 3) T->has_dct4 = m != 0;
    }
    seg += __popc(m) << lg;
    first += __popc(m);
  }
  if (b == 0) T->seg[kTaskKinds] = 3 * seg;
}
// All threads call.
__device__ inline void BuildTasks(const uint8_t* acs_t, bool hf_only,
                                  TileTasks* T) {
  BuildTasksWave(acs_t, hf_only, T, 0);
  __syncthreads();
}

// Column k of an N x N transform's F matrix (row-major, flat i * N + k)
// with origin block (oby, obx): F[i][k] sits in storage row oby + i / 8,
// column obx * 64 + (i % 8) * N + k, so its index is
//   CoefColumn(oby, obx, k) + CoefRowOffset<N>(i)
// (k < N keeps (i % 8) * N % 64 + k inside one block). With the row offset
// a compile-time constant every access of a line shares one address and
// differs only in the instruction's immediate offset.
__device__ inline unsigned CoefColumn(unsigned oby, unsigned obx, unsigned k) {
  return oby * kCoefRow + obx * kCoefBlock + k;
}
template <int N>
__host__ __device__ constexpr int CoefRowOffset(int i) {
  return (i / 8) * kCoefRow + ((i % 8) * N / 64) * kCoefBlock +
         (i % 8) * N % 64;
}

// CoefRowOffset<N>(i) + k equals the storage index of flat i * N + k
// relative to the origin block for every i, k < N.
template <int N>
constexpr bool CoefRowOffsetsMatchLayout() {
  for (int i = 0; i < N; ++i) {
    for (int k = 0; k < N; ++k) {
      const int flat = i * N + k;
      const int row = flat / (8 * N), col = flat % (8 * N);
      const int idx = row * kCoefRow + (col >> 6) * kCoefBlock + (col & 63);
      if (CoefRowOffset<N>(i) + k != idx) return false;
    }
  }
  return true;
}
static_assert(CoefRowOffsetsMatchLayout<8>() &&
                  CoefRowOffsetsMatchLayout<16>() &&
                  CoefRowOffsetsMatchLayout<32>(),
              "coefficient row offsets");

template <int N>
__device__ inline void InvLine1(const float* coef, float* tmp, int oby,
                                int obx, int c) {
  const float* col = coef + CoefColumn(oby, obx, c);
  float v[N], w[N];
  for (int r = 0; r < N; ++r) v[r] = col[CoefRowOffset<N>(r)];
  dct1d::Idct<N>(v, w);
  for (int x = 0; x < N; ++x) tmp[PixAt(oby * 8 + c, obx * 8 + x)] = w[x];
}
template <int N>
__device__ inline void InvLine2(const float* tmp, float* pix, int oby,
                                int obx, int x) {
  float v[N], w[N];
  for (int c = 0; c < N; ++c) v[c] = tmp[PixAt(oby * 8 + c, obx * 8 + x)];
  dct1d::Idct<N>(v, w);
  for (int y = 0; y < N; ++y) pix[PixAt(oby * 8 + y, obx * 8 + x)] = w[y];
}
template <int N>
__device__ inline void FwdLine1(const float* pix, float* tmp, int oby,
                                int obx, int x) {
  float v[N], w[N];
  for (int y = 0; y < N; ++y) v[y] = pix[PixAt(oby * 8 + y, obx * 8 + x)];
  dct1d::Dct<N>(v, w);
  for (int k = 0; k < N; ++k) tmp[PixAt(oby * 8 + x, obx * 8 + k)] = w[k];
}
// kAddHF: add the coefficients outside the 2s x 2s low-frequency corner
// to coef instead of storing them, or with kSubHF subtract them
// (AddBlockExceptLFAndLLFTo<true / false>, pik/ac_predictions.cc:38-70).
template <int N, bool kAddHF = false, bool kSubHF = false>
__device__ inline void FwdLine2(const float* tmp, float* coef, int oby,
                                int obx, int k) {
  constexpr int s = N / 8;
  float v[N], w[N];
  for (int x = 0; x < N; ++x) v[x] = tmp[PixAt(oby * 8 + x, obx * 8 + k)];
  dct1d::Dct<N>(v, w);
  const float scale = 1.0f / (N * N);
  float* col = coef + CoefColumn(oby, obx, k);
  for (int j = 0; j < N; ++j) {
    float& dst = col[CoefRowOffset<N>(j)];
    if (!kAddHF) {
      dst = w[j] * scale;
    } else if (!(j < 2 * s && k < 2 * s)) {
      dst = kSubHF ? dst - w[j] * scale : dst + w[j] * scale;
    }
  }
}

// One task of the inverse transform: pass 0 columns of the coefficient
// matrix into tmp, pass 1 columns of tmp into pixels (DCT4X4 per 4x4
// sub-block with the Hadamard of the four DCs, pik/ac_strategy.cc:762-790;
// DCT2X2 and IDENTITY directly in pass 1).
__device__ inline void InverseTask(int pass, int raw, int l, int oby, int obx,
                                   const float* coef, float* pix, float* tmp) {
  if (raw == kDCT || raw == kDCTNoHF) {
    if (pass == 0) InvLine1<8>(coef, tmp, oby, obx, l);
    else InvLine2<8>(tmp, pix, oby, obx, l);
  } else if (raw == kDCT16) {
    if (pass == 0) InvLine1<16>(coef, tmp, oby, obx, l);
    else InvLine2<16>(tmp, pix, oby, obx, l);
  } else if (raw == kDCT32) {
    if (pass == 0) InvLine1<32>(coef, tmp, oby, obx, l);
    else InvLine2<32>(tmp, pix, oby, obx, l);
  } else if (AcsIsDCT4(raw)) {
    const int sub = l >> 2, sy = sub >> 1, sx = sub & 1, q = l & 3;
    float v[4], w[4];
    if (pass == 0) {
      // column q of the sub-block's 4x4 matrix G, G[iy][ix] =
      // coef[(sy + 2 iy) * 8 + sx + 2 ix], G[0][0] from the DC Hadamard
      const float* cb = coef + CoefAt(oby, obx * 64);
      const float b00 = cb[0], b01 = cb[1], b10 = cb[8], b11 = cb[9];
      float dc;
      if (sub == 0) dc = b00 + b01 + b10 + b11;
      else if (sub == 1) dc = b00 + b01 - b10 - b11;
      else if (sub == 2) dc = b00 - b01 + b10 - b11;
      else dc = b00 - b01 - b10 + b11;
      for (int r = 0; r < 4; ++r) {
        v[r] = (r == 0 && q == 0) ? dc : cb[(sy + r * 2) * 8 + sx + q * 2];
      }
      dct1d::Idct<4>(v, w);
      for (int x = 0; x < 4; ++x) {
        tmp[PixAt(oby * 8 + sy * 4 + q, obx * 8 + sx * 4 + x)] = w[x];
      }
    } else {
      for (int c = 0; c < 4; ++c) {
        v[c] = tmp[PixAt(oby * 8 + sy * 4 + c, obx * 8 + sx * 4 + q)];
      }
      dct1d::Idct<4>(v, w);
      for (int y = 0; y < 4; ++y) {
        pix[PixAt(oby * 8 + sy * 4 + y, obx * 8 + sx * 4 + q)] = w[y];
      }
    }
  } else if (pass == 1) {
    DirectInverse8(raw, coef + CoefAt(oby, obx * 64),
                   pix + PixAt(oby * 8, obx * 8), kTilePitch);
  }
}

// One task of the forward transform: pass 0 columns of pixels into tmp,
// pass 1 columns of tmp into coefficients (x 1/N^2), pass 2 the DC Hadamard
// of DCT4X4 (pik/ac_strategy.cc:590-613); DCT2X2 and IDENTITY in pass 0.
// kAdjoint replaces IDENTITY's forward transform by the transpose of its
// inverse (the other strategies' transposes are scaled forward transforms).
// kAddHF adds the result outside each transform's 2s x 2s low-frequency
// corner to coef (the HF prediction; only strategies with PredictHF, so no
// DCT2X2 or IDENTITY, and the DCT4X4 DC Hadamard, which only touches that
// corner, is skipped).
template <bool kAdjoint = false, bool kAddHF = false, bool kSubHF = false>
__device__ inline void ForwardTask(int pass, int raw, int l, int oby, int obx,
                                   const float* pix, float* coef, float* tmp) {
  if (raw == kDCT || raw == kDCTNoHF) {
    if (pass == 0) FwdLine1<8>(pix, tmp, oby, obx, l);
    else if (pass == 1) FwdLine2<8, kAddHF, kSubHF>(tmp, coef, oby, obx, l);
  } else if (raw == kDCT16) {
    if (pass == 0) FwdLine1<16>(pix, tmp, oby, obx, l);
    else if (pass == 1) FwdLine2<16, kAddHF, kSubHF>(tmp, coef, oby, obx, l);
  } else if (raw == kDCT32) {
    if (pass == 0) FwdLine1<32>(pix, tmp, oby, obx, l);
    else if (pass == 1) FwdLine2<32, kAddHF, kSubHF>(tmp, coef, oby, obx, l);
  } else if (AcsIsDCT4(raw)) {
    const int sub = l >> 2, sy = sub >> 1, sx = sub & 1, q = l & 3;
    float v[4], w[4];
    float* cb = coef + CoefAt(oby, obx * 64);
    if (pass == 0) {
      for (int y = 0; y < 4; ++y) {
        v[y] = pix[PixAt(oby * 8 + sy * 4 + y, obx * 8 + sx * 4 + q)];
      }
      dct1d::Dct<4>(v, w);
      for (int k = 0; k < 4; ++k) {
        tmp[PixAt(oby * 8 + sy * 4 + q, obx * 8 + sx * 4 + k)] = w[k];
      }
    } else if (pass == 1) {
      for (int x = 0; x < 4; ++x) {
        v[x] = tmp[PixAt(oby * 8 + sy * 4 + x, obx * 8 + sx * 4 + q)];
      }
      dct1d::Dct<4>(v, w);
      for (int j = 0; j < 4; ++j) {
        float& dst = cb[(sy + j * 2) * 8 + sx + q * 2];
        if (!kAddHF) {
          dst = w[j] * (1.0f / 16);
        } else if (!(j == 0 && q == 0)) {  // outside the 2x2 corner
          dst = kSubHF ? dst - w[j] * (1.0f / 16) : dst + w[j] * (1.0f / 16);
        }
      }
    } else if (!kAddHF && l == 0) {
      const float b00 = cb[0], b01 = cb[1], b10 = cb[8], b11 = cb[9];
      cb[0] = (b00 + b01 + b10 + b11) * 0.25f;
      cb[1] = (b00 + b01 - b10 - b11) * 0.25f;
      cb[8] = (b00 - b01 + b10 - b11) * 0.25f;
      cb[9] = (b00 - b01 - b10 + b11) * 0.25f;
    }
  } else if (pass == 0) {
    if (kAdjoint && raw == kIdentity) {
      IdentityAdjoint8(pix + PixAt(oby * 8, obx * 8), kTilePitch,
                       coef + CoefAt(oby, obx * 64));
    } else {
      DirectForward8(raw, pix + PixAt(oby * 8, obx * 8), kTilePitch,
                     coef + CoefAt(oby, obx * 64));
    }
  }
}

// A thread's share of a tile's tasks, decoded once for all passes: task
// k = threadIdx.x + 256 * i in slot i (in slot 1 the waves in reverse, so that
// the wave with the longest tasks of slot 0 gets the last ones), packed as
// channel | raw << 2 | line << 6 | oby << 11 | obx << 13, and kNoTask past the
// last task. A channel has at most 16 blocks x 16 line
// tasks (DCT4X4), so three slots cover 3 x 256 tasks.
constexpr int kTaskSlots = 3;
constexpr uint32_t kNoTask = 0xFFFFFFFFu;
struct ThreadTasks {
  uint32_t t[kTaskSlots];
  bool has_dct4;  // TileTasks::has_dct4 (the same for the workgroup)
  // slot i by selects (a variable index into t would put it in scratch)
  __device__ uint32_t Slot(int i) const {
    return i == 0 ? t[0] : (i == 1 ? t[1] : t[2]);
  }
};

__device__ inline ThreadTasks AssignTasks(const TileTasks& T) {
  const int total = T.seg[kTaskKinds];
  ThreadTasks m;
  m.has_dct4 = T.has_dct4 != 0;
#pragma unroll
  for (int i = 0; i < kTaskSlots; ++i) {
    const int k = (i == 1 ? threadIdx.x ^ 192 : threadIdx.x) + 256 * i;
    m.t[i] = kNoTask;
    if (k < total) {
      const int kd = (k >= T.seg[1]) + (k >= T.seg[2]) + (k >= T.seg[3]) +
                     (k >= T.seg[4]);
      const uint32_t w = T.kind[kd];
      const int n = int(w & 0xFFFF), t = k - T.seg[kd];
      const int c = (t >= n) + (t >= 2 * n);
      const uint32_t r = uint32_t(t - c * n), lg = w >> 24;
      const uint32_t at = T.at[((w >> 16) & 0xFF) + (r >> lg)];
      const uint32_t b = at >> 4;
      m.t[i] = uint32_t(c) | ((at & 15) << 2) |
               ((r & ((1u << lg) - 1)) << 6) | ((b >> 2) << 11) |
               ((b & 3) << 13);
    }
  }
  return m;
}

// coef (3 x kCoefPlane) -> pix (3 x kTilePlane), tmp 3 x kTilePlane. All
// 256 threads must call.
__device__ __forceinline__ void TileInverse3(const ThreadTasks& m, const float* coef,
                                    float* pix, float* tmp) {
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll 1
    for (int i = 0; i < kTaskSlots; ++i) {
      const uint32_t w = m.Slot(i);
      if (w != kNoTask) {
        const int c = w & 3;
        InverseTask(pass, (w >> 2) & 15, (w >> 6) & 31, (w >> 11) & 3,
                    (w >> 13) & 3, coef + c * kCoefPlane, pix + c * kTilePlane,
                    tmp + c * kTilePlane);
      }
    }
    __syncthreads();
  }
}
__device__ __forceinline__ void TileInverse3(const TileTasks& T, const float* coef,
                                    float* pix, float* tmp) {
  TileInverse3(AssignTasks(T), coef, pix, tmp);
}

// pix (3 x kTilePlane) -> coef (3 x kCoefPlane) for the transforms in T
// (others keep their coefficient entries), tmp 3 x kTilePlane. All 256
// threads must call.
template <bool kAdjoint = false, bool kAddHF = false, bool kSubHF = false>
__device__ __forceinline__ void TileForward3(const ThreadTasks& m, const float* pix,
                                    float* coef, float* tmp) {
  // pass 2 (the DCT4X4 DC Hadamard) only when the tile has a DCT4X4
  const int passes = kAddHF ? 2 : (m.has_dct4 ? 3 : 2);
  for (int pass = 0; pass < passes; ++pass) {
#pragma unroll 1
    for (int i = 0; i < kTaskSlots; ++i) {
      const uint32_t w = m.Slot(i);
      if (w != kNoTask) {
        const int c = w & 3;
        ForwardTask<kAdjoint, kAddHF, kSubHF>(
            pass, (w >> 2) & 15, (w >> 6) & 31, (w >> 11) & 3,
            (w >> 13) & 3, pix + c * kTilePlane, coef + c * kCoefPlane,
            tmp + c * kTilePlane);
      }
    }
    __syncthreads();
  }
}
template <bool kAdjoint = false, bool kAddHF = false, bool kSubHF = false>
__device__ __forceinline__ void TileForward3(const TileTasks& T, const float* pix,
                                    float* coef, float* tmp) {
  TileForward3<kAdjoint, kAddHF, kSubHF>(AssignTasks(T), pix, coef, tmp);
}

// Coefficient ownership of a 256-thread tile pass, as in KBlocks: storage
// row crow of the tile, columns ccol..ccol+3; 16 consecutive lanes own one
// 8x8 storage block.
struct CoefSlot {
  int crow, ccol, cbx, cby;
  bool valid;
  int raw, cs, cN, lgn, cflat0, obxg, obyg;
  uint8_t acs;
};

__device__ inline CoefSlot MakeSlot(const FrameParams& P, const uint8_t* s_acs,
                                    int tbx, int tby, int gbx0, int gby0) {
  CoefSlot s;
  const int tid = threadIdx.x;
  s.crow = tid >> 6;
  s.ccol = (tid & 63) << 2;
  s.cbx = tbx + (s.ccol >> 6);
  s.cby = tby + s.crow;
  s.valid = s.cbx < P.bx && s.cby < P.by;
  s.acs = s_acs[s.crow * 4 + (s.ccol >> 6)];
  s.raw = s.acs >> 4;
  const int cidx = s.acs & 15;
  s.cs = s.acs == 0xFF ? 1 : AcsCovered(s.raw);
  const int lgs = s.cs >> 1;  // log2(cs): cs is 1, 2 or 4
  s.lgn = 3 + lgs;
  const int coby = s.crow - (cidx >> lgs), cobx = (s.ccol >> 6) - (cidx & (s.cs - 1));
  s.cflat0 = (s.crow - coby) * 64 * s.cs + (s.ccol - cobx * 64);
  s.cN = 8 * s.cs;
  s.obxg = tbx + cobx - gbx0;
  s.obyg = tby + coby - gby0;
  return s;
}

// ---------------------------------------------------------------------------
// Workgroup-to-tile order for the eight XCDs of an MI355X. Consecutive
// workgroup ids are dealt round-robin to the XCDs, each with its own L2, so
// in plain row-major order neighbouring tiles -- which read each other's
// halo rows and columns -- sit in different L2s. Here XCD k walks the
// contiguous row-major tile range [k * per, (k + 1) * per) in order.
// Launch 8 * per workgroups (per = ceil(num_tiles / 8)); ids past the last
// tile get -1 and return at once.
constexpr int kNumXcds = 8;

__host__ __device__ inline int XcdGrid(int num_tiles) {
  return kNumXcds * ((num_tiles + kNumXcds - 1) / kNumXcds);
}

__device__ inline int XcdTile(int wg, int num_tiles) {
  const int per = (num_tiles + kNumXcds - 1) / kNumXcds;
  const int tile = (wg % kNumXcds) * per + wg / kNumXcds;
  return tile < num_tiles ? tile : -1;
}

// ---------------------------------------------------------------------------
// The workgroup a kernel body works on: blockIdx / gridDim of a plain
// launch, or, in a batched launch, the frame's own grid inside one launch
// over every frame of the batch (BatchSpan).
struct VBlock {
  int x, y, z;     // workgroup index
  int nx, ny, nz;  // grid size in workgroups
};
__device__ inline VBlock PlainBlock() {
  VBlock v;
  v.x = int(blockIdx.x);
  v.y = int(blockIdx.y);
  v.z = int(blockIdx.z);
  v.nx = int(gridDim.x);
  v.ny = int(gridDim.y);
  v.nz = int(gridDim.z);
  return v;
}

// A frame of a batch in device memory: its parameters and buffers as a
// plain launch passes them.
struct BatchFrame {
  FrameParams P;
  FrameBuffers B;
};
// One frame's share of a batched launch of one phase: launch workgroups
// [first, first + count) run the frame's nx x ny x nz grid (count =
// nx * ny * nz), with the phase's per-frame integer arguments. `first` is
// a multiple of kNumXcds, so a frame's local workgroup index keeps the XCD
// of the launch's (XcdTile).
constexpr int kBatchArgs = 5;
struct BatchSpan {
  uint32_t frame, first, count;
  int nx, ny, nz;
  int arg[kBatchArgs];
};

// The span table's companion map: entry w is the index (into the launch's
// spans) of the span holding launch workgroup w, or kNoSpan for the idle
// workgroups between spans (one load instead of a search per workgroup).
typedef const BatchSpan ConstSpan;
constexpr uint32_t kNoSpan = 0xFFFFFFFFu;

__device__ inline VBlock SpanBlock(ConstSpan& s, uint32_t w) {
  const int l = int(w - s.first);
  VBlock v;
  v.nx = s.nx;
  v.ny = s.ny;
  v.nz = s.nz;
  v.x = l % s.nx;
  v.y = (l / s.nx) % s.ny;
  v.z = l / (s.nx * s.ny);
  return v;
}

// The loop of a batched kernel: workgroup blockIdx.x takes launch
// workgroups blockIdx.x, + gridDim.x, ... below `total` (one of them when
// the launch has `total` workgroups: a persistent launch has fewer), runs
// `body` with s (the BatchSpan), vb (the frame's workgroup), P and B (the
// frame's), and waits for the workgroup before the next one reuses LDS.
#define PIKGPU_BATCH_LOOP(body)                                       \
  for (uint32_t w_ = blockIdx.x; w_ < total; w_ += gridDim.x) {       \
    const uint32_t si_ = M[w_];                                       \
    if (si_ != kNoSpan) {                                             \
      ConstSpan& s = S[si_];                                          \
      const VBlock vb = SpanBlock(s, w_);                             \
      const FrameParams& P = F[s.frame].P;                            \
      const FrameBuffers& B = F[s.frame].B;                           \
      body;                                                           \
    }                                                                 \
    __syncthreads();                                                  \
  }

// One launch workgroup per frame workgroup (a launch of `total`
// workgroups), for the kernels whose registers a loop around them would
// overflow (the compiler keeps per-thread values of the body live across
// the iterations).
#define PIKGPU_BATCH_ONE(body)                                        \
  {                                                                   \
    const uint32_t w_ = blockIdx.x;                                   \
    const uint32_t si_ = w_ < total ? M[w_] : kNoSpan;                \
    if (si_ != kNoSpan) {                                             \
      ConstSpan& s = S[si_];                                          \
      const VBlock vb = SpanBlock(s, w_);                             \
      const FrameParams& P = F[s.frame].P;                            \
      const FrameBuffers& B = F[s.frame].B;                           \
      body;                                                           \
    }                                                                 \
  }

// The batched kernels' common parameters.
#define PIKGPU_BATCH_PARAMS                                             \
  const BatchFrame *__restrict__ F, const BatchSpan *__restrict__ S,    \
      const uint32_t *__restrict__ M, uint32_t total,                   \
      const DeviceConsts *K


// ---------------------------------------------------------------------------
// Small reinterpreting transforms with compile-time sizes: every array index
// is static after unrolling, so the blocks stay in registers.

// 2-point transforms in the reference's explicit form (pik/dct.h:478-504).
__device__ inline void Idct2x2(float a00, float a01, float a10, float a11,
                               float* o, int os) {
  o[0] = a00 + a01 + a10 + a11;
  o[1] = a00 + a01 - a10 - a11;
  o[os] = a00 - a01 + a10 - a11;
  o[os + 1] = a00 - a01 - a10 + a11;
}

// Index of the scale tables for size n: log2(n) - 1.
template <int N>
constexpr int ScaleIdx() {
  return N == 2 ? 0 : (N == 4 ? 1 : (N == 8 ? 2 : (N == 16 ? 3 : 4)));
}

// ReinterpretingIDCT<DCTN, LF, N> (pik/ac_strategy.cc:296-315), N >= 4:
// the LF x LF input (pitch ip) zero-padded to N x N.
template <int DCTN, int LF, int N>
__device__ inline void ReinterpIdct(const DeviceConsts* K, const float* in,
                                    int ip, float* out, int op) {
  float blk[N * N], pix[N * N];
  constexpr int ai = ScaleIdx<N>(), ti = ScaleIdx<DCTN>();
#pragma unroll
  for (int y = 0; y < N; ++y) {
#pragma unroll
    for (int x = 0; x < N; ++x) {
      float v = 0.0f;
      if (y < LF && x < LF) {
        v = (in[y * ip + x] * K->ascale[ai][y][x]) * K->tscale[ti][y][x];
      }
      blk[y * N + x] = v;
    }
  }
  dct1d::Idct2D<N>(blk, N, pix, N);
#pragma unroll
  for (int y = 0; y < N; ++y) {
#pragma unroll
    for (int x = 0; x < N; ++x) out[y * op + x] = pix[y * N + x];
  }
}

// Quantizer::QuantizeDC's factor per channel: InvMatrix(0, DCT8, c)[0] *
// (Scale() * quant_dc) (pik/quantizer.h:350-353).
struct EncDcScale {
  float scale[3];
};
// ---------------------------------------------------------------------------
// Kernels.
__global__ void KDcDequant(FrameParams P, FrameBuffers B);
__global__ void KEncForward(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                            const float* opsin, float* coef, float* dcf);
__global__ void KEncInverseTable(const float* table, int n, float* out);
__global__ void KEncDc(FrameParams P, const float* dcf, EncDcScale S,
                       int16_t* dc16);
__global__ void KEncQuant(FrameParams P, FrameBuffers B, const float* coef,
                          const float* itable, float gsf, int16_t* ac);
__global__ void KSearchForward(FrameParams P, FrameBuffers B,
                               const float* coef, const float* itable,
                               float gsf, int16_t* ac);
__global__ void KEncLf(FrameParams P, FrameBuffers B, float* coef,
                       const float* itable, float gsf, float* corner);
__global__ void KEncHfResidual(FrameParams P, FrameBuffers B, float* coef);
// KLf: workgroup size; strips of 16 block rows per group, each a workgroup
// per plane (grid: groups x strips, planes).
constexpr int kLfThreads = 1024;
constexpr int kLfStrip = 16;
constexpr int kLfStrips = kGroupDimBlocks / kLfStrip;
__global__ void KLf(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                    int border);
__global__ void KEncPred2x2Border(FrameParams P, FrameBuffers B,
                                  const DeviceConsts* K);
// KPred2x2: block rows per strip, workgroups per strip; the grid of a frame's
// groups.
constexpr int kPredRows = 4;
constexpr int kPredStrips = kGroupDimBlocks / kPredRows;
constexpr int kPredRoles = 3;
inline int PredGrid(int groups) { return groups * kPredStrips * kPredRoles; }
template <bool kEnc>
__global__ void KPred2x2(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                         const float* corner);
__global__ void KBlocks(FrameParams P, FrameBuffers B, const DeviceConsts* K);
__global__ void KAdjForward(FrameParams P, FrameBuffers B,
                            const DeviceConsts* K, AdjArgs A);
// <true>: the quant-field search's, which leaves each block's distortion (from
// the unquantized coefficients, three planes in the AC layout) instead of the
// gradients.
struct SearchDist {
  float* dist;
  const float* coef;
};
template <bool kSearch>
__global__ void KAdjBackward(FrameParams P, FrameBuffers B,
                             const DeviceConsts* K, AdjArgs A, SearchDist D);
__global__ void KAdjLoss(const float* part, int n, double* out);

// Parameters of one Adam step of the quant-field search (search.hip).
struct SearchArgs {
  const float* weight;  // per-block perceptual weight w_b, or null (1)
  const float* lambda;  // rate weight per block (device scalar)
  float lr, beta1, beta2, eps;
  float ulo, uhi;       // bounds of the log field
  float dlo, dhi;       // trust region around the initial log field
};
__global__ void KSearchRound(FrameParams P, FrameBuffers B, const float* u,
                             int qmax, int32_t* qf, float* qfr, float* part);
// The search's state at each transform's first block: log field and Adam
// moments. A step reads one copy and writes the other.
struct SearchState {
  float *u, *m, *v;
};
// The partials of the evaluation before a step, and where their sums go.
struct SearchSums {
  const float *loss_part, *rate_part;
  int loss_n, rate_n;
  double *loss, *rate;
};
__global__ void KSearchStep(FrameParams P, FrameBuffers B, SearchArgs S, int t,
                            const float* dist, const float* u0,
                            SearchState from, SearchState to, int qmax,
                            int32_t* qf, float* qfr, float* rate_part,
                            SearchSums sums);
__global__ void KSearchInit(FrameParams P, FrameBuffers B, float* u0, float* u,
                            float* m, float* v);
__global__ void KSearchLambda(const float* dist, const float* weight, int n,
                              float fixed, float kappa, float* out);

// Generic image description for the filters.
struct Img {
  const float* p;  // 3 planes
  size_t plane;    // floats per plane
  int pitch;       // floats per row
  int W, H;        // logical size (mirror borders)
  int vw, vh;      // valid source region (replicate beyond, <= W, H)
};

// Images of a frame as the filters take them: the IDCT image (full size,
// width a multiple of 8, rows 32-float aligned) and the 8-padded DC image
// (valid bx x by).
__host__ __device__ inline Img IdctImage(const FrameParams& P,
                                         const FrameBuffers& B) {
  Img ii;
  ii.p = B.idct;
  ii.plane = size_t(B.ipitch) * P.py;
  ii.pitch = B.ipitch;
  ii.W = P.px;
  ii.H = P.py;
  ii.vw = P.px;
  ii.vh = P.py;
  return ii;
}
__host__ __device__ inline Img DcImage(const FrameParams& P,
                                       const FrameBuffers& B) {
  Img dci;
  dci.p = B.dcq;
  dci.plane = size_t(P.bx) * P.by;
  dci.pitch = P.bx;
  dci.W = (P.bx + 7) / 8 * 8;
  dci.H = (P.by + 7) / 8 * 8;
  dci.vw = P.bx;
  dci.vh = P.by;
  return dci;
}

__global__ void KMinMaxPartial4(Img in, int gaborish, FrameParams P,
                                FrameBuffers B);
__global__ void KMinMaxFinal(const float* partial, int n, float* mm);
// KDcEpf: rows per workgroup of 32 columns.
constexpr int kDcEpfRows = 8;
__global__ void KDcEpf(Img in, FrameParams P, FrameBuffers B,
                       const DeviceConsts* K, int n_partial);
__global__ void KEpf(Img in, FrameParams P, FrameBuffers B,
                     const DeviceConsts* K);
__global__ void KGuide(Img in, int gaborish, FrameParams P, FrameBuffers B,
                       int n_partial);
__global__ void KDots(FrameParams P, FrameBuffers B);
// KFinal: rows per workgroup of its 256-column strips. A thread walks them
// one after the other, about 1 us each where the chip is not full, and reads
// two more: kFinalRows where that leaves four workgroups per CU (and in a
// batch, whose frames fill the chip together), else as many as do, at least 2
// (803x533: 18 us with 16 rows, 8 us with 2; one tile: 9 and 4 us).
constexpr int kFinalRows = 16;
inline int FinalRows(int px, int py) {
  const int strips = (px + 255) / 256;
  int rows = kFinalRows;
  while (rows > 2 && strips * ((py + rows - 1) / rows) < 1024) rows /= 2;
  return rows;
}
__global__ void KFinal(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                       int rows);
__global__ void KCopyPlanes(FrameBuffers B, size_t n);

// Batched forms of the reconstruction's kernels (pikgpu_batch): one launch
// per phase over every frame of a batch; see BatchSpan.
__global__ void KDcDequantBatch(PIKGPU_BATCH_PARAMS);
__global__ void KMinMaxFinalBatch(PIKGPU_BATCH_PARAMS);
__global__ void KDcEpfBatch(PIKGPU_BATCH_PARAMS);
__global__ void KLfBatch(PIKGPU_BATCH_PARAMS);
__global__ void KPred2x2Batch(PIKGPU_BATCH_PARAMS);
__global__ void KBlocksBatch(PIKGPU_BATCH_PARAMS);
__global__ void KMinMaxPartial4Batch(PIKGPU_BATCH_PARAMS);
__global__ void KGuideBatch(PIKGPU_BATCH_PARAMS);
__global__ void KEpfBatch(PIKGPU_BATCH_PARAMS);
__global__ void KCopyPlanesBatch(PIKGPU_BATCH_PARAMS);
__global__ void KDotsBatch(PIKGPU_BATCH_PARAMS);
__global__ void KFinalBatch(PIKGPU_BATCH_PARAMS);

}  // namespace pikgpu
