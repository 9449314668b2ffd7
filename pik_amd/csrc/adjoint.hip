// Forward model and adjoint of the differentiable part of the
// reconstruction, for gradient-based quant-field search (gfx950, wave64).
//
// The model is the decode with HF prediction, adaptive reconstruction and
// dots off, as a function of a real-valued quant field qf (one value per
// block; the dequantisation table stays the one the frame's integer field
// selects):
//   d_c   = AdjustQuantBias_c(q) * M_c[k] * (inv_global_scale / qf)
//           (Dequant::DoAC, pik/compressed_image.cc:586-693)
//   C'    = LLF / LF predictions + CfL(d)   (pik/ac_predictions.cc:560-620)
//   P     = TransformToPixels(C')           (pik/ac_strategy.cc:674-840)
//   G     = Gaborish(P), cropped            (pik/compressed_image.cc:1164)
//   L     = OpsinToLinear(G)                (pik/opsin_inverse.cc:39-123)
// With qf equal to the integer field, L is bit for bit the decoder's output
// for the same flags.
//
// Two kernels per evaluation, one 32x32-pixel tile per workgroup:
//   KAdjForward   dequant (real qf) + LLF/LF + CfL + IDCT -> P in HBM
//   KAdjBackward  P with a 2-pixel ring -> G, L, dL/dL (from a target or
//                 given), opsin adjoint -> dG with a 1-pixel ring (mirrored
//                 at the image edge), Gaborish transpose -> dP, transform
//                 transposes -> dC', CfL transpose -> dd, and
//                 dL/dqf = -sum_k dd . d / qf per block.
// P is written once and read once (plus ring); nothing else is stored
// between the two kernels.
#include "kernels.h"

namespace pikgpu {

namespace {

// Dequantised AC value of channel c without colour correlation, in
// DequantWith's operation order with the real-valued field's scale: m is
// the dequant matrix entry.
__device__ inline float DequantPlain(float m, float scaled, int c,
                                     int16_t q) {
  const float mul = m * scaled;
  return AdjustQuantBias(c, float(q)) * mul;
}

// What a thread needs of its four coefficients' block, loaded at the top of
// the kernel, before the first wait: the dequantisation descriptor of
// KDcDequant (or KSearchRound), the quantized values, the real-valued field
// and the colour correlation. (Through the chain strategy -> field ->
// control field -> table index -> offset, once per channel, the two kernels
// took 64 + 140 us on a 2048x2048 frame, 54 + 103 us with the descriptors, and
// 42 + 94 us now.)
struct CoefIn {
  bool valid;
  size_t at;       // index in an AC plane
  uint4 desc;
  uint2 q4[3];
  float qf, cfx, cfb;
};

__device__ inline CoefIn LoadCoefIn(const FrameParams& P,
                                    const FrameBuffers& B, const AdjArgs& A,
                                    int tbx, int tby) {
  CoefIn in;
  const int tid = threadIdx.x;
  const int ccol = (tid & 63) << 2;
  const int cbx = tbx + (ccol >> 6), cby = tby + (tid >> 6);
  in.valid = cbx < P.bx && cby < P.by;
  in.at = size_t(cby) * P.bx * 64 + size_t(cbx) * 64 + (ccol & 63);
  in.desc = make_uint4(0, 0, 0, 0);
  in.qf = 1.0f;
  in.cfx = in.cfb = 0.0f;
  for (int c = 0; c < 3; ++c) in.q4[c] = make_uint2(0, 0);
  if (in.valid) {
    const size_t plane = size_t(P.by) * P.bx * 64;
    in.desc = B.desc[2 * (cby * P.bx + cbx)];
    // four int16, 8-byte aligned (at is a multiple of 4)
    for (int c = 0; c < 3; ++c) {
      in.q4[c] = *reinterpret_cast<const uint2*>(B.ac + c * plane + in.at);
    }
    in.qf = A.qf[size_t(cby) * A.qf_pitch + cbx];
    const int ctile = (tby >> 3) * P.tx + (tbx >> 3);
    in.cfx = float(B.ytox[ctile] - 128) * 0.00390625f;
    in.cfb = float(B.ytob[ctile]) * 0.0078125f;
  }
  return in;
}
__device__ inline int16_t CoefQ(const uint2& q, int j) {
  const uint32_t w = j < 2 ? q.x : q.y;
  return int16_t((j & 1) ? w >> 16 : w & 0xFFFF);
}
__device__ inline void LoadMatrix(const FrameBuffers& B, const CoefIn& in,
                                  float (&m)[3][4]) {
  if (!in.valid) return;
  const uint32_t slot[3] = {in.desc.x, in.desc.y, in.desc.z};
  for (int c = 0; c < 3; ++c) {
    LoadFour(B.table + slot[c] + (in.at & 63), m[c]);
  }
}
__device__ inline uint8_t TileAcs(const FrameParams& P, const FrameBuffers& B,
                                  int tbx, int tby) {
  const int tid = threadIdx.x;
  if (tid >= 16) return 0xFF;
  const int bxa = tbx + (tid & 3), bya = tby + (tid >> 2);
  return (bxa < P.bx && bya < P.by) ? B.acs[bya * P.bx + bxa] : 0xFF;
}

}  // namespace

__global__ void __launch_bounds__(256, 4)
    KAdjForward(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                AdjArgs A) {
  __shared__ float s_coef[3][kCoefPlane];
  __shared__ float s_pix[3][kTilePlane];
  __shared__ float s_tmp[3][kTilePlane];
  __shared__ uint8_t s_acs[16];
  __shared__ TileTasks s_inv;

  const int tid = threadIdx.x;
  const int tiles_x = (P.bx + 3) / 4;
  const int tile = XcdTile(blockIdx.x, tiles_x * ((P.by + 3) / 4));
  if (tile < 0) return;
  const int tbx = (tile % tiles_x) * 4, tby = (tile / tiles_x) * 4;
  if (B.stamps) StampStart(&B.stamps->adj[0], blockIdx.x);
  const uint8_t a_own = TileAcs(P, B, tbx, tby);
  const CoefIn in = LoadCoefIn(P, B, A, tbx, tby);
  if (tid < 16) s_acs[tid] = a_own;
  __syncthreads();

  const int gxi = tbx / kGroupDimBlocks, gyi = tby / kGroupDimBlocks;
  const int g = gyi * P.gx + gxi;
  const CoefSlot S = MakeSlot(P, s_acs, tbx, tby, gxi * kGroupDimBlocks,
                              gyi * kGroupDimBlocks);
  // the matrix entries and the LLF / LF values load while one wave builds
  // the task table (one branch per entry for the latter; as one per entry,
  // channel and kind of value the kernel took 43 us instead of 41 on a
  // 2048x2048 frame)
  float mv[3][4] = {}, fixv[3][4];
  int fix[4];
  LoadMatrix(B, in, mv);
  for (int j = 0; j < 4; ++j) {
    const int flat = S.cflat0 + j;
    const int fi = flat >> S.lgn, fj = flat & (S.cN - 1);
    fix[j] = (fi < S.cs && fj < S.cs)
                 ? 1
                 : ((P.predict_lf && fi < 2 * S.cs && fj < 2 * S.cs) ? 2 : 0);
    fixv[0][j] = fixv[1][j] = fixv[2][j] = 0.0f;
    if (in.valid && fix[j] != 0) {
      const bool is_llf = fix[j] == 1;
      const int plane = is_llf ? kLlfPlane : kG2Plane;
      const float* p = (is_llf ? B.llf : B.lf2x2) + size_t(g) * 3 * plane +
                       (is_llf ? (S.obyg + 1 + fi) * kLlfPitch + S.obxg + 1 + fj
                               : (2 * (S.obyg + 1) + fi) * kG2Pitch +
                                     2 * (S.obxg + 1) + fj);
      for (int c = 0; c < 3; ++c) fixv[c][j] = p[c * plane];
    }
  }
  BuildTasks(s_acs, false, &s_inv);
  if (in.valid) {
    const float scaled = P.inv_global_scale / in.qf;
    const float cc[3] = {in.cfx, 0.0f, in.cfb};
    float yv[4];
    for (int ci = 0; ci < 3; ++ci) {
      const int c = ci == 0 ? 1 : (ci == 1 ? 0 : 2);
      for (int j = 0; j < 4; ++j) {
        const float v0 = DequantPlain(mv[c][j], scaled, c, CoefQ(in.q4[c], j));
        float v = c == 1 ? v0 : cc[c] * yv[j] + v0;
        if (c == 1) yv[j] = v;
        if (fix[j] == 1) {
          v = fixv[c][j];
        } else if (fix[j] == 2) {
          v += fixv[c][j];
        }
        s_coef[c][CoefAt(S.crow, S.ccol + j)] = v;
      }
    }
  }
  __syncthreads();
  TileInverse3(s_inv, &s_coef[0][0], &s_pix[0][0], &s_tmp[0][0]);
  const int pr = tid >> 3, pc0 = (tid & 7) << 2;
  const int py = tby * 8 + pr, px = tbx * 8 + pc0;
  // px and P.px are multiples of 4 and 8, the rows 128-byte aligned
  if (py < P.py && px < P.px) {
    for (int c = 0; c < 3; ++c) {
      const float* s = s_pix[c] + PixAt(pr, pc0);
      *reinterpret_cast<float4*>(B.idct + (size_t(c) * P.py + py) * B.ipitch +
                                 px) = make_float4(s[0], s[1], s[2], s[3]);
    }
  }
}

// Ring geometry of the backward tile: P at [-2, 34) and dG at [-1, 33)
// around the 32x32 tile.
constexpr int kPW = 36;
constexpr int kGW = 34;
constexpr int kGPer = (kGW * kGW + 255) / 256;  // dG positions per thread

template <bool kSearch>
__global__ void __launch_bounds__(256, 4)
    KAdjBackward(FrameParams P, FrameBuffers B, const DeviceConsts* K,
                 AdjArgs A, SearchDist D) {
  // One LDS array for the buffers of all phases, 39 KB, so that four
  // workgroups share a CU (three with a buffer each): P's ring from 0,
  // dG's ring from kDg; then dP from 0 over the dead P, the transform's
  // scratch behind it, its coefficients over the dead dG.
  constexpr int kTmp = 3 * kTilePlane, kDg = 6 * kTilePlane;
  static_assert(3 * kPW * kPW <= kDg && kCoefPlane <= kGW * kGW,
                "the rings and the transform buffers must not collide");
  __shared__ float s_buf[kDg + 3 * kGW * kGW];
  __shared__ uint8_t s_acs[16];
  __shared__ TileTasks s_fwd;
  __shared__ float s_loss[4];
  float* s_a = s_buf;
  float* s_b = s_buf + kDg;

  const int tid = threadIdx.x;
  const int tiles_x = (P.bx + 3) / 4;
  const int num_tiles = tiles_x * ((P.by + 3) / 4);
  const int tile = XcdTile(blockIdx.x, num_tiles);
  if (tile < 0) return;
  const int tbx = (tile % tiles_x) * 4, tby = (tile / tiles_x) * 4;
  const int ox = tbx * 8, oy = tby * 8;
  if (B.stamps) StampStart(&B.stamps->adj[1], blockIdx.x);
  const uint8_t a_own = TileAcs(P, B, tbx, tby);

  // 1. P ring (mirrored at the 8-padded image edge, as the Gaborish
  //    convolution reads it; positions past the mirrored row or column are
  //    clamped into the image and never used). Tiles whose columns all lie
  //    inside the image load float4s, columns -4 .. +35. The targets (or
  //    the upstream gradient) load along with it.
  const size_t iplane = size_t(P.py) * B.ipitch;
  const bool edge =
      ox == 0 || oy == 0 || ox + 32 >= P.px || oy + 32 >= P.py;
  auto row_of = [&](int y) {
    y = y < 0 ? -y - 1 : (y >= P.py ? 2 * P.py - 1 - y : y);
    return min(max(y, 0), P.py - 1);
  };
  if (ox >= 4 && ox + 36 <= P.px) {
    constexpr int kVec = 3 * kPW * 10, kPer = (kVec + 255) / 256;
    float4 wv[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = tid + u * 256;
      wv[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (k < kVec) {
        const int row = k / 10, q = k - row * 10;
        const int c = row / kPW, ly = row - c * kPW;
        wv[u] = *reinterpret_cast<const float4*>(
            B.idct + c * iplane + size_t(row_of(oy - 2 + ly)) * B.ipitch + ox -
            4 + 4 * q);
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = tid + u * 256;
      if (k < kVec) {
        const int row = k / 10, q = k - row * 10;
        // float4 q holds ring columns 4q - 2 .. 4q + 1
        float* d = s_a + row * kPW + 4 * q - 2;
        if (q > 0) {
          d[0] = wv[u].x;
          d[1] = wv[u].y;
        }
        if (q < 9) {
          d[2] = wv[u].z;
          d[3] = wv[u].w;
        }
      }
    }
  } else {
    for (int k = tid; k < kPW * kPW; k += 256) {
      int X = ox - 2 + k % kPW;
      X = X < 0 ? -X - 1 : (X >= P.px ? 2 * P.px - 1 - X : X);
      X = min(max(X, 0), P.px - 1);
      const float* src =
          B.idct + size_t(row_of(oy - 2 + k / kPW)) * B.ipitch + X;
      for (int c = 0; c < 3; ++c) s_a[c * kPW * kPW + k] = src[c * iplane];
    }
  }
  const float* const* ext = A.target[0] ? A.target : A.upstream;
  float tv[kGPer][3];
#pragma unroll
  for (int u = 0; u < kGPer; ++u) {
    const int k = tid + u * 256;
    const int Y = oy - 1 + k / kGW, X = ox - 1 + k % kGW;
    const bool ok = k < kGW * kGW && Y >= 0 && Y < P.ysize && X >= 0 &&
                    X < P.xsize;
    const size_t at = size_t(Y) * A.in_pitch + X;
    for (int c = 0; c < 3; ++c) tv[u][c] = ok ? ext[c][at] : 0.0f;
  }
  if (tid < 16) s_acs[tid] = a_own;
  __syncthreads();
  BuildTasks(s_acs, false, &s_fwd);

  // 2. G, L and dL/dG at the ring positions inside the padded image.
  const float* inv = K->opsin_inv;
  float loss = 0.0f;
#pragma unroll
  for (int u = 0; u < kGPer; ++u) {
    const int k = tid + u * 256;
    const int i = k / kGW, j = k % kGW;
    const int Y = oy - 1 + i, X = ox - 1 + j;
    if (k >= kGW * kGW || Y < 0 || Y >= P.py || X < 0 || X >= P.px) continue;
    float v[3];
    for (int c = 0; c < 3; ++c) {
      const float* pc = s_a + c * kPW * kPW + (i + 1) * kPW + j + 1;
      v[c] = P.gaborish ? Conv3(pc, kPW, P.gab_w) : pc[0];
    }
    float dv0 = 0.0f, dv1 = 0.0f, dv2 = 0.0f;
    if (Y < P.ysize && X < P.xsize) {
      // OpsinToLinear in KFinal's operation order.
      const float gamma_r = 1.0f * (v[1] + v[0]);
      const float gamma_g = 1.0f * (v[1] - v[0]);
      const float gamma_b = v[2];
      const float gamma_r2 = gamma_r * gamma_r;
      const float gamma_g2 = gamma_g * gamma_g;
      const float gamma_b2 = gamma_b * gamma_b;
      const float mixed_r = gamma_r2 * gamma_r + P.neg_bias[0];
      const float mixed_g = gamma_g2 * gamma_g + P.neg_bias[1];
      const float mixed_b = gamma_b2 * gamma_b + P.neg_bias[2];
      float lr = inv[0] * mixed_r;
      float lg = inv[3] * mixed_r;
      float lb = inv[6] * mixed_r;
      const float tr = inv[1] * mixed_g;
      const float tg = inv[4] * mixed_g;
      const float tb = inv[7] * mixed_g;
      lr = inv[2] * mixed_b + lr;
      lg = inv[5] * mixed_b + lg;
      lb = inv[8] * mixed_b + lb;
      lr = lr + tr;
      lg = lg + tg;
      lb = lb + tb;
      const bool inner = i >= 1 && i <= 32 && j >= 1 && j <= 32;
      float e0 = tv[u][0], e1 = tv[u][1], e2 = tv[u][2];
      if (A.target[0]) {
        e0 = lr - e0;
        e1 = lg - e1;
        e2 = lb - e2;
        if (inner) loss += e0 * e0 + e1 * e1 + e2 * e2;
        e0 *= 2.0f;
        e1 *= 2.0f;
        e2 *= 2.0f;
      }
      if (inner && A.linear[0]) {
        const size_t o = size_t(Y) * A.lin_pitch + X;
        A.linear[0][o] = lr;
        A.linear[1][o] = lg;
        A.linear[2][o] = lb;
      }
      // Opsin transpose: dmixed_j = sum_i inv[3i + j] dL_i; d gamma =
      // 3 gamma^2 dmixed; (r, g) = (Y + X, Y - X).
      const float dmr = inv[0] * e0 + inv[3] * e1 + inv[6] * e2;
      const float dmg = inv[1] * e0 + inv[4] * e1 + inv[7] * e2;
      const float dmb = inv[2] * e0 + inv[5] * e1 + inv[8] * e2;
      const float dgr = 3.0f * gamma_r2 * dmr;
      const float dgg = 3.0f * gamma_g2 * dmg;
      dv0 = dgr - dgg;
      dv1 = dgr + dgg;
      dv2 = 3.0f * gamma_b2 * dmb;
    }
    s_b[k] = dv0;
    s_b[kGW * kGW + k] = dv1;
    s_b[2 * kGW * kGW + k] = dv2;
  }
  // the coefficients' inputs load during the next phases
  const CoefIn in = LoadCoefIn(P, B, A, tbx, tby);
  __syncthreads();

  // 3. Ring positions outside the padded image take the value of the
  //    pixel they mirror: the transpose of the mirrored read folds the
  //    ring back onto the edge, which for the symmetric 3x3 kernel equals
  //    convolving the mirror-extended dG.
  if (edge) {
    for (int k = tid; k < kGW * kGW; k += 256) {
      const int i = k / kGW, j = k % kGW;
      const int Y = oy - 1 + i, X = ox - 1 + j;
      if (Y >= 0 && Y < P.py && X >= 0 && X < P.px) continue;
      const int si = Mirror(Y, P.py) - oy + 1, sj = Mirror(X, P.px) - ox + 1;
      const bool ok = si >= 0 && si < kGW && sj >= 0 && sj < kGW;
      for (int c = 0; c < 3; ++c) {
        s_b[c * kGW * kGW + k] = ok ? s_b[c * kGW * kGW + si * kGW + sj] : 0.0f;
      }
    }
    __syncthreads();
  }

  // 4. dP = Gaborish transpose (the same symmetric kernel) of the ring,
  //    four rows of a column per thread.
  {
    const int j = tid & 31, i0 = (tid >> 5) * 4;
    for (int c = 0; c < 3; ++c) {
      const float* g = s_b + c * kGW * kGW + (i0 + 1) * kGW + j + 1;
      for (int i = 0; i < 4; ++i) {
        s_a[c * kTilePlane + PixAt(i0 + i, j)] =
            P.gaborish ? Conv3(g + i * kGW, kGW, P.gab_w) : g[i * kGW];
      }
    }
  }
  float mv[3][4] = {}, x[3][4];
  LoadMatrix(B, in, mv);
  if (kSearch && in.valid) {
    for (int c = 0; c < 3; ++c) {
      LoadFour(D.coef + c * size_t(P.by) * P.bx * 64 + in.at, x[c]);
    }
  }
  __syncthreads();

  // 5. Transform transposes: forward transform, then the per-coefficient
  //    norm scale (IDENTITY directly).
  float* s_coef = s_b;
  TileForward3<true>(s_fwd, s_a, s_coef, s_buf + kTmp);

  // 6. CfL transpose, dL/dd and dL/dqf.
  const int gxi = tbx / kGroupDimBlocks, gyi = tby / kGroupDimBlocks;
  const CoefSlot S = MakeSlot(P, s_acs, tbx, tby, gxi * kGroupDimBlocks,
                              gyi * kGroupDimBlocks);
  float part = 0.0f;
  float dist[4] = {};
  if (in.valid) {
    const float scaled = P.inv_global_scale / in.qf;
    float out[3][4];
    for (int j = 0; j < 4; ++j) {
      const int flat = S.cflat0 + j;
      const int fi = flat >> S.lgn, fj = flat & (S.cN - 1);
      const int e = CoefAt(S.crow, S.ccol + j);
      if (fi < S.cs && fj < S.cs) {
        out[0][j] = out[1][j] = out[2][j] = 0.0f;
        continue;
      }
      const float sc = AdjointScale(K->adj_norm, S.raw, flat);
      const float gx = s_coef[e] * sc;
      const float gy = s_coef[kCoefPlane + e] * sc;
      const float gb = s_coef[2 * kCoefPlane + e] * sc;
      const float gyt = gy + in.cfx * gx + in.cfb * gb;
      const float vx = DequantPlain(mv[0][j], scaled, 0, CoefQ(in.q4[0], j));
      const float vy = DequantPlain(mv[1][j], scaled, 1, CoefQ(in.q4[1], j));
      const float vb = DequantPlain(mv[2][j], scaled, 2, CoefQ(in.q4[2], j));
      if (!kSearch) {
        part += gx * vx + gyt * vy + gb * vb;
        out[0][j] = gx;
        out[1][j] = gyt;
        out[2][j] = gb;
        continue;
      }
      // the search's distortion (search.hip): gradient times quantization
      // error in the total (after colour correlation) coefficient domain,
      // where Y's gradient is its pre-correlation one minus the factors
      // times X's and B's
      dist[j] = gx * (in.cfx * vy + vx - x[0][j]) +
                (gyt - in.cfx * gx - in.cfb * gb) * (vy - x[1][j]) +
                gb * (in.cfb * vy + vb - x[2][j]);
    }
    if (!kSearch && A.dcoef[0]) {
      for (int c = 0; c < 3; ++c) {
        float* dst = A.dcoef[c] + size_t(S.cby) * A.dc_pitch +
                     size_t(S.cbx) * 64 + (S.ccol & 63);
        if (A.dcoef_vec) {
          *reinterpret_cast<float4*>(dst) =
              make_float4(out[c][0], out[c][1], out[c][2], out[c][3]);
        } else {
          for (int j = 0; j < 4; ++j) dst[j] = out[c][j];
        }
      }
    }
  }
  if (kSearch) {
    // the block's 64 slots, pairwise over slot distances 32, 16, .. 1 (slot
    // k = 4 lane + j)
    for (int m = 8; m >= 1; m >>= 1) {
      for (int j = 0; j < 4; ++j) dist[j] += __shfl_xor(dist[j], m, 64);
    }
    const float d = (dist[0] + dist[2]) + (dist[1] + dist[3]);
    if (in.valid && (tid & 15) == 0) D.dist[S.cby * P.bx + S.cbx] = 0.5f * d;
  } else {
    // Sum over the 16 lanes of the block (all lanes take part).
    for (int m = 8; m >= 1; m >>= 1) part += __shfl_xor(part, m, 64);
    if (in.valid && (tid & 15) == 0) {
      A.dqf[size_t(S.cby) * A.dqf_pitch + S.cbx] = -part / in.qf;
    }
  }

  // 7. Tile loss partial.
  if (A.loss_part) {
    for (int m = 32; m >= 1; m >>= 1) loss += __shfl_xor(loss, m, 64);
    if ((tid & 63) == 0) s_loss[tid >> 6] = loss;
    __syncthreads();
    if (tid == 0) {
      A.loss_part[tile] = (s_loss[0] + s_loss[1]) + (s_loss[2] + s_loss[3]);
    }
  }
  if (B.stamps) StampEnd(B.stamps->end[1], blockIdx.x);
}
template __global__ void KAdjBackward<false>(FrameParams, FrameBuffers,
                                             const DeviceConsts*, AdjArgs, SearchDist);
template __global__ void KAdjBackward<true>(FrameParams, FrameBuffers,
                                            const DeviceConsts*, AdjArgs, SearchDist);

__global__ void __launch_bounds__(256)
    KAdjLoss(const float* part, int n, double* out) {
  SumPartials(part, n, out);
}

}  // namespace pikgpu
