// DC and LF-domain kernels of the reconstruction (gfx950).
//
// These run at DC resolution (1/64 of the pixels) or on the 2x-upsampled DC
// grid, per 512x512 decode group, and produce the per-group caches the block
// kernel consumes:
//   DequantDC                         pik/compressed_dc.cc:181-230
//   InitializeDecCache (DC + border)  pik/compressed_dc.cc:530-556
//   ComputeLlf                        pik/ac_predictions.cc:380-405
//   PredictLf                         pik/ac_predictions.cc:410-470
//   border of pred2x2                 pik/compressed_image.cc:980-1039
//   UpdateLfForDecoder (pred2x2)      pik/ac_predictions.cc:560-635
// The group caches have fixed pitches (device.h).
#include <float.h>
#include <stddef.h>

#include "device.h"
#include "kernels.h"

namespace pikgpu {

// DequantDC; also writes each block's dequantisation descriptors and, per
// workgroup, the minimum and maximum of the DC image over the channels (the
// DC EPF's guide has no Gaborish and its padding repeats pixels of the
// image, so its range is the image's). At most kDcGroups workgroups, each
// walking the blocks with a stride, so that every workgroup of the DC EPF
// can reduce the partials itself. With a thread per block and the min/max and
// its reduction in two kernels of their own a 4096x4096 frame took 8 + 7 + 4
// us, 14 us so; a small one 4 + 3 us and two launches more.
__device__ __forceinline__ void KDcDequantBody(
    const FrameParams& P, const FrameBuffers& B, const VBlock& vb) {
  __shared__ float s_mm[8];
  if (B.stamps) StampStart(&B.stamps->run[0], vb.x);
  const int n = P.bx * P.by;
  float lo = FLT_MAX, hi = -FLT_MAX;
  for (int i = vb.x * 256 + int(threadIdx.x); i < n; i += vb.nx * 256) {
    const uint8_t a = B.acs[i];
    const int s = AcsCovered(a >> 4), idx = a & 15;
    const int first = i - (idx >> (s >> 1)) * P.bx - (idx & (s - 1));
    WriteBlockDesc(P, B, i, B.qf[i], B.qf[first]);
    // Y first, then X/B = ytox|ytob * Y + q * mul (the portable target's
    // mul_add is a separate multiply and add).
    const float y = float(B.dc16[n + i]) * P.mul_dc[1];
    const float dqx = float(B.dc16[i]) * P.mul_dc[0];
    const float dqb = float(B.dc16[2 * n + i]) * P.mul_dc[2];
    const float x = P.ytox_dc * y + dqx;
    const float b = P.ytob_dc * y + dqb;
    B.dcq[i] = x;
    B.dcq[n + i] = y;
    B.dcq[2 * n + i] = b;
    lo = fminf(lo, fminf(fminf(x, y), b));
    hi = fmaxf(hi, fmaxf(fmaxf(x, y), b));
  }
  GroupMinMax(&lo, &hi, s_mm);
  if (threadIdx.x == 0) {
    B.mm_partial[2 * vb.x] = lo;
    B.mm_partial[2 * vb.x + 1] = hi;
  }
}
__global__ void __launch_bounds__(256)
    KDcDequant(FrameParams P, FrameBuffers B) {
  KDcDequantBody(P, B, PlainBlock());
}

// Group geometry helpers.
struct GroupGeom {
  int gbx0, gby0, gw, gh;
};
__device__ inline GroupGeom Geom(const FrameParams& P, int g) {
  GroupGeom G;
  const int gxi = g % P.gx, gyi = g / P.gx;
  G.gbx0 = gxi * kGroupDimBlocks;
  G.gby0 = gyi * kGroupDimBlocks;
  G.gw = min(kGroupDimBlocks, P.bx - G.gbx0);
  G.gh = min(kGroupDimBlocks, P.by - G.gby0);
  return G;
}

// DC of plane c of the group cache at cache coordinates (x, y): SourceCoord
// clamping (pik/compressed_dc.h:46-49) is clamp(c - 1, 0, size - 1). For a
// grayscale frame X and B come from Y (GrayXyb::YToXyb, pik/compressed_image.cc:
// 99-104, in double as there: the piece index truncates (y - sub) * mul * 16,
// the value y * slope + constant is rounded to float), as RestoreXB rebuilds
// them in the group cache before the LF predictions (:953-956).
__device__ inline float GroupDc(const FrameParams& P, const DeviceConsts* K,
                                const float* dc, int c, const GroupGeom& G,
                                int x, int y) {
  const int sx = min(max(G.gbx0 + x - 1, 0), P.bx - 1);
  const int sy = min(max(G.gby0 + y - 1, 0), P.by - 1);
  const size_t plane = size_t(P.bx) * P.by, at = size_t(sy) * P.bx + sx;
  if (!P.grayscale || c == 1) return dc[c * plane + at];
  const float yv = dc[plane + at];
  const GrayXybTable& T = K->gray;
  int i = (int)((yv - T.sub) * T.mul * kGrayPieces);
  i = min(max(0, i), kGrayPieces - 1);
  return c == 0 ? (float)(yv * T.x_slope[i] + T.x_const[i])
                : (float)(yv * T.b_slope[i] + T.b_const[i]);
}

// Strategy of cache position (x, y); border positions count as DCT8 first
// blocks (pik/ac_predictions.cc:391-399).
__device__ inline uint8_t CacheAcs(const FrameParams& P, const FrameBuffers& B,
                                   const GroupGeom& G, int x, int y) {
  if (x == 0 || y == 0 || x == G.gw + 1 || y == G.gh + 1) return 0;
  return B.acs[(G.gby0 + y - 1) * P.bx + G.gbx0 + x - 1];
}

// A border position of pred2x2 as a DCT8 block: ReinterpretingIDCT<8, 2, 2>
// of {llf, lf(0,1), lf(1,0), lf(1,1)} (pik/compressed_image.cc:980-1039).
__device__ inline void Pred2x2BorderAt(const DeviceConsts* K, float llf,
                                       float l01, float l10, float l11,
                                       float* o) {
  const float a00 = (llf * K->ascale[0][0][0]) * K->tscale[2][0][0];
  const float a01 = (l01 * K->ascale[0][0][1]) * K->tscale[2][0][1];
  const float a10 = (l10 * K->ascale[0][1][0]) * K->tscale[2][1][0];
  const float a11 = (l11 * K->ascale[0][1][1]) * K->tscale[2][1][1];
  o[0] = a00 + a01 + a10 + a11;
  o[1] = a00 + a01 - a10 - a11;
  o[kG2Pitch] = a00 - a01 + a10 - a11;
  o[kG2Pitch + 1] = a00 - a01 - a10 + a11;
}

// ---------------------------------------------------------------------------
// The LF domain of one group and plane: ComputeLlf (LowestFrequenciesFromDC,
// pik/ac_strategy.cc:850-887), then with predict_lf the steps of PredictLf
// (pik/ac_predictions.cc:410-470) -- the LLF's 2x image
// (DC2x2FromLowestFrequencies, pik/ac_strategy.cc:928-969), its 3x3 blur with
// mirrored borders (Symmetric3, pik/convolve.h:502-640), the LF coefficients
// (LowFrequenciesFromDC2x2, pik/ac_strategy.cc:1019-1064) -- and with
// `border` the border of pred2x2 (pik/compressed_image.cc:980-1039).
//
// Every step reads its neighbours' results of the one before; a strip of 16
// block rows keeps them all in LDS, with the four rows above and below
// recomputed (the blur needs the 2x row next to the strip, which may belong
// to a 32x32 transform; strips are aligned to those). The DC and the
// strategies come in once, LLF and LF go out once. As four kernels over the
// group caches in memory it took 54 us of a 4096x4096 frame and four launches
// of 3 to 5 us of a small one; one workgroup for a whole group and plane (91
// KB) 28 us and, for want of workgroups, 24 us of an 803x533 frame; strips
// 23 us and 10 us.
constexpr int kLfRows = kLfStrip + 8;  // block rows of a strip in LDS

struct LfShared {
  float g2[2 * kLfRows * kG2Pitch];  // the 2x image, then the LF coefficients
  float dc[kLfRows * kLlfPitch];     // the cache's DC, then the LLF
  float tscale[5][8][8], ascale[5][8][8];  // DeviceConsts'
  uint8_t acs[kLfRows * kLlfPitch];
};

// The strip's rows of the group cache: [lo, hi) are in LDS, [first, last)
// are its own (the group's border rows 0 and gh + 1 belong to the first and
// the last strip).
struct LfStrip {
  int lo, hi, first, last;
};

// Orders the LDS accesses of a wave's lanes around it (they run in lockstep
// and LDS accesses of a wave are in order; this keeps the compiler from
// moving them).
__device__ inline void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// One DCT16 (S = 2) or DCT32 (S = 4) transform on N = 2S lanes of a wave.
struct LfUnit {
  bool active;
  int x, y, l;  // cache column and LDS row of the first block, lane
};
// Slots of the S-aligned first-block positions of kLfRows block rows.
template <int S>
constexpr int LfSlots() {
  return kLfRows / S * (kGroupDimBlocks / S) * 2 * S;
}
// Unit `slot / N` of those in cache rows [from, to) of the strip; the first
// position at or after its first row is S-aligned.
template <int S>
__device__ inline LfUnit LfUnitAt(const LfShared& s, const GroupGeom& G,
                                  const LfStrip& R, int from, int to,
                                  int slot) {
  constexpr int N = 2 * S, kPer = kGroupDimBlocks / S;
  const int u = slot / N;
  const int x = 1 + S * (u % kPer), y = max(R.lo, 1) + S * (u / kPer);
  LfUnit f;
  f.l = slot % N;
  f.x = x;
  f.y = y - R.lo;
  f.active = x <= G.gw && y >= from && y < to && y <= G.gh &&
             s.acs[f.y * kLlfPitch + x] ==
                 uint8_t((S == 4 ? kDCT32 : kDCT16) << 4);
  return f;
}

// LLF of a unit in place of its DC and, with lf, its 2x image. Each element
// sees the operations of LowestFrequenciesFromDC and
// DC2x2FromLowestFrequencies in their order: for S = 4 the 4x4
// ReinterpretingDCT as a column pass on lanes 0..3 and a row pass after the
// transpose, for S = 2 the 2x2 Hadamard in every lane; then the column and
// row passes of Idct2D<N> over the zero-padded LLF. The transposes go
// through the unit's own region of the 2x image. Every lane of the wave
// calls.
template <int S>
__device__ inline void LlfUnit(const LfUnit& f, bool lf, LfShared* s) {
  constexpr int N = 2 * S;
  constexpr int ai = ScaleIdx<N>(), ti = ScaleIdx<8 * S>();
  const int l = f.l;
  float* t = s->g2 + 2 * f.y * kG2Pitch + 2 * f.x;  // rows of kG2Pitch
  float* dc = s->dc + f.y * kLlfPitch + f.x;
  float col[S];  // LLF column l (lanes l < S)
  if (S == 4) {
    float v[4], w[4];
    if (f.active && l < 4) {
#pragma unroll
      for (int iy = 0; iy < 4; ++iy) v[iy] = dc[iy * kLlfPitch + l];
      dct1d::Dct<4>(v, w);
#pragma unroll
      for (int k = 0; k < 4; ++k) t[l * kG2Pitch + k] = w[k];
    }
    WaveSync();
    if (f.active && l < 4) {
#pragma unroll
      for (int xx = 0; xx < 4; ++xx) v[xx] = t[xx * kG2Pitch + l];
      dct1d::Dct<4>(v, w);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float cf = w[j] * (1.0f / 16);
        const float u = cf * s->tscale[1][j][l];
        col[j] = u * s->ascale[4][j][l];
        dc[j * kLlfPitch + l] = col[j];
      }
    }
  } else {
    float d[4];
    if (f.active) {
      const float a00 = dc[0], a01 = dc[1];
      const float a10 = dc[kLlfPitch], a11 = dc[kLlfPitch + 1];
      d[0] = (a00 + a01 + a10 + a11) * 0.25f;
      d[1] = (a00 + a01 - a10 - a11) * 0.25f;
      d[2] = (a00 - a01 + a10 - a11) * 0.25f;
      d[3] = (a00 - a01 - a10 + a11) * 0.25f;
    }
    WaveSync();
    if (f.active && l < 2) {
#pragma unroll
      for (int iy = 0; iy < 2; ++iy) {
        const float v = (l == 0 ? d[iy * 2] : d[iy * 2 + 1]) *
                        s->tscale[0][iy][l];
        col[iy] = v * s->ascale[3][iy][l];
        dc[iy * kLlfPitch + l] = col[iy];
      }
    }
  }
  if (!lf) return;
  WaveSync();
  float v[N], w[N];
  if (f.active) {
#pragma unroll
    for (int r = 0; r < N; ++r) {
      v[r] = (r < S && l < S) ? (col[r < S ? r : 0] * s->ascale[ai][r][l]) *
                                    s->tscale[ti][r][l]
                              : 0.0f;
    }
    dct1d::Idct<N>(v, w);
#pragma unroll
    for (int k = 0; k < N; ++k) t[l * kG2Pitch + k] = w[k];
  }
  WaveSync();
  if (f.active) {
#pragma unroll
    for (int cc = 0; cc < N; ++cc) v[cc] = t[cc * kG2Pitch + l];
    dct1d::Idct<N>(v, w);
  }
  WaveSync();
  if (f.active) {
#pragma unroll
    for (int yy = 0; yy < N; ++yy) t[yy * kG2Pitch + l] = w[yy];
  }
}

// LowFrequenciesFromDC2x2 of a unit, in place: ReinterpretingDCT<8S, 2S, 2S>
// (pik/ac_strategy.cc:272-293) as a column pass, the transpose and a row pass.
template <int S>
__device__ inline void LfCoefUnit(const LfUnit& f, LfShared* s) {
  constexpr int N = 2 * S;
  constexpr int ti = ScaleIdx<N>(), ai = ScaleIdx<8 * S>();
  const int l = f.l;
  float* t = s->g2 + 2 * f.y * kG2Pitch + 2 * f.x;
  float v[N], w[N];
  if (f.active) {
#pragma unroll
    for (int y = 0; y < N; ++y) v[y] = t[y * kG2Pitch + l];
    dct1d::Dct<N>(v, w);
  }
  WaveSync();
  if (f.active) {
#pragma unroll
    for (int k = 0; k < N; ++k) t[l * kG2Pitch + k] = w[k];
  }
  WaveSync();
  if (f.active) {
#pragma unroll
    for (int x = 0; x < N; ++x) v[x] = t[x * kG2Pitch + l];
    dct1d::Dct<N>(v, w);
  }
  WaveSync();
  if (f.active) {
    const float scale = 1.0f / (N * N);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float cf = w[j] * scale;
      const float u = cf * s->tscale[ti][j][l];
      t[j * kG2Pitch + l] = u * s->ascale[ai][j][l];
    }
  }
}

// Copies `floats` (a multiple of 4) from LDS to memory, both 16-byte aligned.
__device__ inline void StoreRows(const float* from, float* to, int floats) {
  for (int i = threadIdx.x; 4 * i < floats; i += kLfThreads) {
    reinterpret_cast<float4*>(to)[i] =
        reinterpret_cast<const float4*>(from)[i];
  }
}

// The strip of workgroup (group, strip); false when the group has no such
// strip.
__device__ inline bool LfStripAt(const GroupGeom& G, int k, LfStrip* R) {
  if (k * kLfStrip >= G.gh) return false;
  const int H = G.gh + 2;
  R->first = k == 0 ? 0 : 1 + k * kLfStrip;
  R->last = (k + 1) * kLfStrip >= G.gh ? H : 1 + (k + 1) * kLfStrip;
  R->lo = max(R->first - 4, 0);
  R->hi = min(R->last + 4, H);
  return true;
}

__device__ __forceinline__ void KLfBody(const FrameParams& P,
                                        const FrameBuffers& B,
                                        const DeviceConsts* K, int border,
                                        const VBlock& vb) {
  __shared__ __attribute__((aligned(16))) LfShared s;
  const int tid = threadIdx.x;
  const int g = vb.x / kLfStrips, k = vb.x % kLfStrips, c = vb.y;
  const GroupGeom G = Geom(P, g);
  if (B.stamps) StampStart(&B.stamps->run[1], vb.x + c);
  LfStrip R;
  if (!LfStripAt(G, k, &R)) return;
  const int W = G.gw + 2, H = G.gh + 2;
  const bool lf = P.predict_lf != 0;
  // Positions of the strip's rows, kLfThreads apart: the quotient and
  // remainder of the step are the same for all.
  const int y0 = tid / W, x0 = tid - y0 * W;
  const int dy = kLfThreads / W, dx = kLfThreads - dy * W;
  auto next = [&](int* x, int* y) {
    *x += dx;
    *y += dy;
    if (*x >= W) {
      *x -= W;
      *y += 1;
    }
  };
  // the DC, the strategies and the scale tables, every load issued before
  // the first store
  {
    constexpr int kPos =
        (kLfRows * kLlfPitch + kLfThreads - 1) / kLfThreads;
    float v[kPos];
    uint8_t a[kPos];
    int at[kPos];
    float sc = 0.0f;
    constexpr int kScales = 2 * 5 * 8 * 8;
    static_assert(kScales <= kLfThreads && offsetof(DeviceConsts, ascale) ==
                                               5 * 8 * 8 * sizeof(float) &&
                      offsetof(LfShared, ascale) - offsetof(LfShared, tscale) ==
                          5 * 8 * 8 * sizeof(float),
                  "one scale per thread");
    if (tid < kScales) sc = (&K->tscale[0][0][0])[tid];
    int x = x0, y = R.lo + y0;
#pragma unroll
    for (int u = 0; u < kPos; ++u) {
      at[u] = -1;
      v[u] = 0.0f;
      a[u] = 0;
      if (y < R.hi) {
        at[u] = (y - R.lo) * kLlfPitch + x;
        v[u] = GroupDc(P, K, B.dc, c, G, x, y);
        a[u] = CacheAcs(P, B, G, x, y);
      }
      next(&x, &y);
    }
    if (tid < kScales) (&s.tscale[0][0][0])[tid] = sc;
#pragma unroll
    for (int u = 0; u < kPos; ++u) {
      if (at[u] >= 0) {
        s.dc[at[u]] = v[u];
        s.acs[at[u]] = a[u];
      }
    }
  }
  __syncthreads();
  const size_t gc = size_t(g) * 3 + c;
  float* pred = B.pred2x2 + gc * kG2Plane;
  // LLF and the 2x image: the strategies of one DC value (whose LLF is that
  // value), then the lane units
  {
    int x = x0, y = R.lo + y0;
#pragma unroll 1
    for (; y < R.hi; next(&x, &y)) {
      const int yl = y - R.lo;
      const uint8_t a = s.acs[yl * kLlfPitch + x];
      const int raw = a >> 4;
      if ((a & 15) != 0 || raw == kDCT16 || raw == kDCT32) continue;
      float v = s.dc[yl * kLlfPitch + x];
      if (raw == kDCT || raw == kDCTNoHF || raw == kLines) {
        // ReinterpretingIDCT<8, 1, 2>: one coefficient, 2-point IDCT of it.
        v = (v * s.ascale[0][0][0]) * s.tscale[2][0][0];
      }
      if (lf) {
        float* o = s.g2 + 2 * yl * kG2Pitch + 2 * x;
        o[0] = v;
        o[1] = v;
        o[kG2Pitch] = v;
        o[kG2Pitch + 1] = v;
      } else if (border && y >= R.first && y < R.last &&
                 (x == 0 || y == 0 || x == W - 1 || y == H - 1)) {
        float* o = pred + 2 * y * kG2Pitch + 2 * x;
        o[0] = v;
        o[1] = v;
        o[kG2Pitch] = v;
        o[kG2Pitch + 1] = v;
      }
    }
  }
#pragma unroll 1
  for (int slot = tid; slot - tid < LfSlots<4>(); slot += kLfThreads) {
    const LfUnit f = LfUnitAt<4>(s, G, R, R.lo, R.hi, slot);
    if (__ballot(f.active)) LlfUnit<4>(f, lf, &s);
  }
#pragma unroll 1
  for (int slot = tid; slot - tid < LfSlots<2>(); slot += kLfThreads) {
    const LfUnit f = LfUnitAt<2>(s, G, R, R.lo, R.hi, slot);
    if (__ballot(f.active)) LlfUnit<2>(f, lf, &s);
  }
  __syncthreads();
  {
    float* llf = B.llf + gc * kLlfPlane;
    for (int i = R.first * kLlfPitch + tid; i < R.last * kLlfPitch;
         i += kLfThreads) {
      llf[i] = s.dc[i - R.lo * kLlfPitch];
    }
  }
  if (!lf) return;
  // the blur of the strip's own rows, whose results wait in registers until
  // every window is read
  {
    const int W2 = 2 * W, H2 = 2 * H;
    const int per = kLfThreads / W2;  // rows per pass
    constexpr int kOwn = 2 * (kLfStrip + 2);
    constexpr int kPer = kLfThreads / kG2Pitch;
    constexpr int kRows = (kOwn + kPer - 1) / kPer;
    const int r0 = tid / W2, x = tid - r0 * W2;
    const int xm = max(x - 1, 0), xp = min(x + 1, W2 - 1);
    const float* g2 = s.g2 - 2 * R.lo * kG2Pitch;
    float o[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int y = 2 * R.first + r0 + u * per;
      o[u] = 0.0f;
      if (r0 < per && y < 2 * R.last) {
        // Symmetric3's operation order; one mirrored step past an edge is
        // the edge itself
        const float* rt = g2 + max(y - 1, 0) * kG2Pitch;
        const float* rm = g2 + y * kG2Pitch;
        const float* rb = g2 + min(y + 1, H2 - 1) * kG2Pitch;
        const float sum_tb = rt[x] + rb[x];
        const float mul0 = rm[x] * P.lfblur_w[0];
        const float sum_lr = rm[xm] + rm[xp];
        const float x1 = sum_tb + sum_lr;
        const float mul1 = x1 * P.lfblur_w[1] + mul0;
        const float sum_t2 = rt[xm] + rt[xp];
        const float sum_b2 = rb[xm] + rb[xp];
        const float x2 = sum_t2 + sum_b2;
        o[u] = x2 * P.lfblur_w[2] + mul1;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int y = 2 * R.first + r0 + u * per;
      if (r0 < per && y < 2 * R.last) {
        s.g2[(y - 2 * R.lo) * kG2Pitch + x] = o[u];
      }
    }
  }
  __syncthreads();
  // LF coefficients of the own rows in place, and the border of pred2x2
  {
    int x = x0, y = R.first + y0;
#pragma unroll 1
    for (; y < R.last; next(&x, &y)) {
      const int yl = y - R.lo;
      const uint8_t a = s.acs[yl * kLlfPitch + x];
      const int raw = a >> 4;
      if ((a & 15) != 0 || raw == kDCT16 || raw == kDCT32) continue;
      float* p = s.g2 + 2 * yl * kG2Pitch + 2 * x;
      const float b00 = p[0], b01 = p[1];
      const float b10 = p[kG2Pitch], b11 = p[kG2Pitch + 1];
      float d[4] = {(b00 + b01 + b10 + b11) * 0.25f,
                    (b00 + b01 - b10 - b11) * 0.25f,
                    (b00 - b01 + b10 - b11) * 0.25f,
                    (b00 - b01 - b10 + b11) * 0.25f};
      if (raw == kDCT || raw == kDCTNoHF || raw == kLines) {
        // ReinterpretingDCT<8, 2, 2>
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = d[i] * s.tscale[0][i >> 1][i & 1];
          d[i] = v * s.ascale[2][i >> 1][i & 1];
        }
      }
      p[0] = d[0];
      p[1] = d[1];
      p[kG2Pitch] = d[2];
      p[kG2Pitch + 1] = d[3];
      if (border && (x == 0 || y == 0 || x == W - 1 || y == H - 1)) {
        Pred2x2BorderAt(K, s.dc[yl * kLlfPitch + x], d[1], d[2], d[3],
                        pred + 2 * y * kG2Pitch + 2 * x);
      }
    }
  }
#pragma unroll 1
  for (int slot = tid; slot - tid < LfSlots<4>(); slot += kLfThreads) {
    const LfUnit f = LfUnitAt<4>(s, G, R, R.first, R.last, slot);
    if (__ballot(f.active)) LfCoefUnit<4>(f, &s);
  }
#pragma unroll 1
  for (int slot = tid; slot - tid < LfSlots<2>(); slot += kLfThreads) {
    const LfUnit f = LfUnitAt<2>(s, G, R, R.first, R.last, slot);
    if (__ballot(f.active)) LfCoefUnit<2>(f, &s);
  }
  __syncthreads();
  static_assert(kG2Plane % 4 == 0 && 2 * kG2Pitch % 4 == 0, "float4 rows");
  StoreRows(s.g2 + 2 * (R.first - R.lo) * kG2Pitch,
            B.lf2x2 + gc * kG2Plane + 2 * R.first * kG2Pitch,
            2 * (R.last - R.first) * kG2Pitch);
}
__global__ void __launch_bounds__(kLfThreads)
    KLf(FrameParams P, FrameBuffers B, const DeviceConsts* K, int border) {
  KLfBody(P, B, K, border, PlainBlock());
}

// The interior of pred2x2: per first block, the decoder-side LF coefficients
// (dequantised + LLF + LF prediction) reinterpreted as a 2x upsampled DC
// block (DC2x2FromLowFrequencies, pik/ac_strategy.cc:971-1017, as called by
// UpdateLfForDecoder, pik/ac_predictions.cc:621-633).
//
// kEnc: the encoder's side (ComputeDecoderBlockAnd2x2DC, pik/ac_predictions.
// cc:136-199): the corner's values were formed by KEncLf and wait in
// `corner` (coefficient layout).
//
// Three workgroups per four block rows of a group -- the 8x8 strategies, the
// DCT32 and the DCT16 transforms, which wait for their loads at the same time
// instead of one after the other -- each for all three planes: X and B take
// the dequantised Y of their colour correlation from the same thread.
// Bound by the scattered corners' memory sectors: for some 20 MB of corners
// of a 4096x4096 frame the L2 fetches 80 MB (twice that by a streaming copy's
// scale) and 21 MB are written. One thread per block and plane, from a list of
// the blocks by class that the host built at every upload (0.4 ms at that
// size), took 40 us; inside KLf, whose large workgroups wait for these loads
// together, 70 us; in one workgroup for the three kinds of a strip 40 us; 37 us
// so. (Another frame of that size: 46 us from the list, 45 us so.)

// The three planes' corner value of F-matrix row i, column j of the transform
// of S x S blocks at frame block (bxa, bya), group block (bxg, byg).
template <int S, bool kEnc>
__device__ inline void Corner3(const FrameParams& P, const FrameBuffers& B,
                               int g, int bxa, int bya, int bxg, int byg,
                               int i, int j, float ccx, float ccb,
                               const float* corner, float (&v)[3]) {
  const int flat = i * 8 * S + j, sb = flat >> 6, k = flat & 63;
  const size_t at = size_t(bya) * P.bx * 64 + size_t(bxa) * 64 + flat;
  if (kEnc) {
    for (int c = 0; c < 3; ++c) {
      v[c] = corner[size_t(c) * P.by * P.bx * 64 + at];
    }
    return;
  }
  if (i < S && j < S) {
    for (int c = 0; c < 3; ++c) {
      v[c] = B.llf[(size_t(g) * 3 + c) * kLlfPlane +
                   (byg + 1 + i) * kLlfPitch + bxg + 1 + j];
    }
    return;
  }
  const uint4 d = B.desc[2 * (bya * P.bx + bxa + sb)];
  const float scaled = __uint_as_float(d.w);
  const BlockDq dq[3] = {{B.table + d.x, scaled, ccx},
                         {B.table + d.y, scaled, 0.0f},
                         {B.table + d.z, scaled, ccb}};
  for (int p = 0; p < P.num_passes; ++p) {
    // each later pass adds its own value, with its own colour correlation
    // (Dequant<false>::DoAC, pik/compressed_image.cc:695-703)
    const float y = DequantWith(dq[1], 1, AcPlane(P, B, p, 1)[at], k, 0.0f);
    const float x = DequantWith(dq[0], 0, AcPlane(P, B, p, 0)[at], k, y);
    const float b = DequantWith(dq[2], 2, AcPlane(P, B, p, 2)[at], k, y);
    v[0] = p == 0 ? x : x + v[0];
    v[1] = p == 0 ? y : y + v[1];
    v[2] = p == 0 ? b : b + v[2];
  }
  if (P.predict_lf) {
    for (int c = 0; c < 3; ++c) {
      v[c] += B.lf2x2[(size_t(g) * 3 + c) * kG2Plane +
                      (2 * (byg + 1) + i) * kG2Pitch + 2 * (bxg + 1) + j];
    }
  }
}

// The DCT16 (S = 2) and DCT32 (S = 4) transforms of the workgroup's rows on
// N = 2S lanes each: lane l builds column l of the corner and runs the column
// pass of Idct2D, then the row pass after the transpose through the unit's
// N x N floats at t. Every thread calls.
template <int S, bool kEnc>
__device__ inline void PredUnits(const FrameParams& P, const FrameBuffers& B,
                                 const DeviceConsts* K, const GroupGeom& G,
                                 int g, int byg0, float ccx, float ccb,
                                 const float* corner, float* s_t) {
  constexpr int N = 2 * S, kPer = kGroupDimBlocks / S;
  constexpr int ai = ScaleIdx<N>(), ti = ScaleIdx<8 * S>();
  const int unit = int(threadIdx.x) / N, l = int(threadIdx.x) % N;
  const int bxg = S * (unit % kPer), byg = byg0 + S * (unit / kPer);
  const bool inside =
      byg < byg0 + kPredRows && bxg < G.gw && byg < G.gh;
  const int bxa = G.gbx0 + bxg, bya = G.gby0 + byg;
  const bool active =
      inside && B.acs[bya * P.bx + bxa] ==
                    uint8_t((S == 4 ? kDCT32 : kDCT16) << 4);
  if (__ballot(active) == 0) return;  // the same for the wave
  float* t = s_t + unit * N * (N + 1);
  float v[3][N], w[N];
  if (active) {
#pragma unroll
    for (int y = 0; y < N; ++y) {
      float q[3];
      Corner3<S, kEnc>(P, B, g, bxa, bya, bxg, byg, y, l, ccx, ccb, corner, q);
      // ReinterpretingIDCT<8S, 2S, 2S>'s scaling
      for (int c = 0; c < 3; ++c) {
        v[c][y] = (q[c] * K->ascale[ai][y][l]) * K->tscale[ti][y][l];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (active) {
      dct1d::Idct<N>(v[c], w);
#pragma unroll
      for (int x = 0; x < N; ++x) t[l * (N + 1) + x] = w[x];
    }
    WaveSync();
    if (active) {
#pragma unroll
      for (int cc = 0; cc < N; ++cc) v[c][cc] = t[cc * (N + 1) + l];
      dct1d::Idct<N>(v[c], w);
      float* o = B.pred2x2 + (size_t(g) * 3 + c) * kG2Plane +
                 2 * (byg + 1) * kG2Pitch + 2 * (bxg + 1);
#pragma unroll
      for (int y = 0; y < N; ++y) o[y * kG2Pitch + l] = w[y];
    }
    WaveSync();
  }
}

template <bool kEnc>
__device__ __forceinline__ void KPred2x2Body(const FrameParams& P,
                                             const FrameBuffers& B,
                                             const DeviceConsts* K,
                                             const float* corner,
                                             const VBlock& vb) {
  // the transposes: 16 DCT32 units of 8 x 9 or 64 DCT16 units of 4 x 5
  __shared__ float s_t[64 * 4 * 5];
  const int role = vb.x % kPredRoles, strip = vb.x / kPredRoles;
  const int g = strip / kPredStrips, byg0 = strip % kPredStrips * kPredRows;
  const GroupGeom G = Geom(P, g);
  if (byg0 >= G.gh) return;
  const auto cfl = [&](int bxg, float* ccx, float* ccb) {
    const int tile = ((G.gby0 + byg0) >> 3) * P.tx + ((G.gbx0 + bxg) >> 3);
    *ccx = float(B.ytox[tile] - 128) * 0.00390625f;
    *ccb = float(B.ytob[tile]) * 0.0078125f;
  };
  float ccx = 0.0f, ccb = 0.0f;
  if (role == 1) {
    const int bxg = int(threadIdx.x) / 8 % 16 * 4;
    if (!kEnc && bxg < G.gw) cfl(bxg, &ccx, &ccb);
    PredUnits<4, kEnc>(P, B, K, G, g, byg0, ccx, ccb, corner, s_t);
    return;
  }
  if (role == 2) {
    const int bxg = int(threadIdx.x) / 4 % 32 * 2;
    if (!kEnc && bxg < G.gw) cfl(bxg, &ccx, &ccb);
    PredUnits<2, kEnc>(P, B, K, G, g, byg0, ccx, ccb, corner, s_t);
    return;
  }
  // one block of the rows per thread
  const int bxg = threadIdx.x & 63, byg = byg0 + int(threadIdx.x >> 6);
  if (bxg < G.gw && byg < G.gh) {
    const int bxa = G.gbx0 + bxg, bya = G.gby0 + byg;
    const uint8_t a = B.acs[bya * P.bx + bxa];
    const int raw = a >> 4;
    if ((a & 15) == 0 && raw != kDCT16 && raw != kDCT32) {
      if (!kEnc) cfl(bxg, &ccx, &ccb);
      float F[4][3];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Corner3<1, kEnc>(P, B, g, bxa, bya, bxg, byg, i >> 1, i & 1, ccx, ccb,
                         corner, F[i]);
      }
      const bool dct = raw == kDCT || raw == kDCTNoHF || raw == kLines;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // ReinterpretingIDCT<8, 2, 2>'s scaling; the others (DCT2X2,
          // DCT4X4(_NOHF), IDENTITY) take the 2x2 Hadamard as it is
          f[i] = dct ? (F[i][c] * K->ascale[0][i >> 1][i & 1]) *
                           K->tscale[2][i >> 1][i & 1]
                     : F[i][c];
        }
        Idct2x2(f[0], f[1], f[2], f[3],
                B.pred2x2 + (size_t(g) * 3 + c) * kG2Plane +
                    2 * (byg + 1) * kG2Pitch + 2 * (bxg + 1),
                kG2Pitch);
      }
    }
  }
}
template <bool kEnc>
__global__ void __launch_bounds__(256)
    KPred2x2(FrameParams P, FrameBuffers B, const DeviceConsts* K,
             const float* corner) {
  KPred2x2Body<kEnc>(P, B, K, corner, PlainBlock());
}
template __global__ void KPred2x2<false>(FrameParams, FrameBuffers,
                                         const DeviceConsts*, const float*);
template __global__ void KPred2x2<true>(FrameParams, FrameBuffers,
                                        const DeviceConsts*, const float*);

// The border of pred2x2 as the encoder without LF prediction forms it: zeros
// in place of the LF values (pik/ac_predictions.cc:187-198; everyone else's
// border is KLf's).
__global__ void __launch_bounds__(256)
    KEncPred2x2Border(FrameParams P, FrameBuffers B, const DeviceConsts* K) {
  const int pos = blockIdx.x * 256 + threadIdx.x;
  const int g = blockIdx.y, c = blockIdx.z;
  const GroupGeom G = Geom(P, g);
  const int W = G.gw + 2, H = G.gh + 2;
  if (pos >= W * H) return;
  const int x = pos % W, y = pos / W;
  if (!(x == 0 || y == 0 || x == W - 1 || y == H - 1)) return;
  const size_t gc = size_t(g) * 3 + c;
  Pred2x2BorderAt(K, B.llf[gc * kLlfPlane + y * kLlfPitch + x], 0.0f, 0.0f,
                  0.0f, B.pred2x2 + gc * kG2Plane + 2 * y * kG2Pitch + 2 * x);
}

// ---------------------------------------------------------------------------
// Batched forms: one launch over every frame of a batch, each frame's part
// of the launch running the plain kernel's grid (BatchSpan, with the
// plain launch's integer arguments in arg[]).
__global__ void __launch_bounds__(256) KDcDequantBatch(PIKGPU_BATCH_PARAMS) {
  PIKGPU_BATCH_LOOP(KDcDequantBody(P, B, vb));
}
__global__ void __launch_bounds__(256) KPred2x2Batch(PIKGPU_BATCH_PARAMS) {
  PIKGPU_BATCH_ONE(KPred2x2Body<false>(P, B, K, nullptr, vb));
}
__global__ void __launch_bounds__(kLfThreads) KLfBatch(PIKGPU_BATCH_PARAMS) {
  PIKGPU_BATCH_ONE(KLfBody(P, B, K, s.arg[0], vb));
}

}  // namespace pikgpu
