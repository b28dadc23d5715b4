// Spatial-mode building blocks (multi-radius hillshade, slope and curvature):
// the NaN-aware Gaussian of a symmetrically padded window, the padded copy,
// the corner-aligned upsampling to a shape, the bilinear sample of a global
// coarse response at a window's raster positions, and the weighted combine of
// per-radius fields.
//
// The reference runs a spatial-mode tile through Dask as one chunk
// (algorithms/tile/dask_bridge.py:395-405): map_overlap with boundary
// 'reflect' pads the window symmetrically ([d c b a | a b c d | d c b a],
// dask.array.overlap.reflect), the block function smooths the padded block
// (_smooth_for_radius, _nan_utils.py:527-552) and runs the local block
// function on it, and the result is trimmed.  Large radii come from one
// global overview (coarse_large_radius_response, _nan_utils.py:328-427).
#include <algorithm>
#include <cmath>
#include <vector>

#include "fsg_common.hpp"

namespace fsg {

constexpr int GN_MAX_R = 160;   // Gaussian taps per side (sigma <= 40 at truncate 4)

struct GaussW {
  int r;
  double g[GN_MAX_R + 1];      // centre, then distance 1 .. r
};

// symmetric ("reflect" in dask) index of i in [0, n), for |excess| <= n
__device__ __forceinline__ int sym(int i, int n) {
  return i < 0 ? -1 - i : (i >= n ? 2 * n - 1 - i : i);
}

// Value of the virtually padded window at padded coordinates, 'nearest'
// beyond the padded extent [0, n + 2 pad).
struct PadSrc {
  const float* p;
  int64_t ld;
  int h, w, pad;
  __device__ __forceinline__ float at(int pr, int pc) const {
    const int hp = h + 2 * pad, wp = w + 2 * pad;
    pr = min(max(pr, 0), hp - 1);
    pc = min(max(pc, 0), wp - 1);
    return p[(int64_t)sym(pr - pad, h) * ld + sym(pc - pad, w)];
  }
};

// The NaN-aware Gaussian runs as two LDS-tiled passes over output tiles of 128 along
// the filter axis and 64 across it, each a product with a band matrix in float64 on
// the matrix cores (v_mfma_f64_16x16x4_f64: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and,
// in entry e, D[l / 16 + 4 e][l % 16]): T[y][k] = g[|k - y - r|] over the 16 + 2 r
// samples that 16 outputs reach, zero outside the band, so the LDS span past a
// window of taps must be finite.  Sums stay float64; only their order is the
// matrix cores', not scipy's, which the float32 rounding after each axis hides
// but for near-ties.  A tile whose span holds an infinity takes gn_slow, scipy's
// order tap by tap: zero weights must not meet it.
// Bound: float64 MFMA issue, (16 + 2 r) / 4 instructions of 64 cycles per 16 x 16
// outputs, for the wide filters (r = 64: 144 of 129 taps); memory for r <= 16.
// As VALU sums (3 operations per pair of taps) the passes took 147 and 164 us on
// average over an 8192^2 hillshade job's 17 windows; now 97 and 98.
// A wave owns 32 outputs along the axis as two groups of 16: the second group's
// band is the first's 16 samples later, so a sample's LDS read and conversion
// serve eight products.
constexpr int GN_T = 64;   // tile extent across the filter axis
constexpr int GN_L = 128;  // ... along it
typedef double d4 __attribute__((ext_vector_type(4)));

// sample as the accumulation sees it: 0 plain, 1 NaN -> 0, 2 validity (0 / 1)
template <int MODE>
__device__ __forceinline__ double gn_val(float f) {
  if constexpr (MODE == 0) return (double)f;
  else if constexpr (MODE == 1) return isnan(f) ? 0.0 : (double)f;
  else return isnan(f) ? 0.0 : 1.0;
}

// The band's weights: T[t] = g[|t - 15 - r|] (0 past r), so that output y and
// sample k take T[k - y + 15].  n <= 512 entries, two per thread: the loads are
// issued (gn_band) ahead of the tile's and stored (put) after them.
struct GnBand {
  double v[2];
  __device__ __forceinline__ void get(const GaussW& G) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int d = abs((int)threadIdx.x + 256 * u - 15 - G.r);
      v[u] = d <= G.r ? G.g[min(d, GN_MAX_R)] : 0.0;
    }
  }
  __device__ __forceinline__ void put(double* T, int n) const {
    if ((int)threadIdx.x < n) T[threadIdx.x] = v[0];
    if ((int)threadIdx.x + 256 < n) T[threadIdx.x + 256] = v[1];
  }
};

// One output in scipy's symmetric order: the centre, then acc + (x[-d] + x[+d]) *
// g[d] for d = r .. 1, each operation rounded on its own.  T: the band.
template <int MODE>
__device__ __forceinline__ double gn_slow(const float* s, int st, const double* T, int r) {
  const double* g = T + 15 + r;
  double acc = gn_val<MODE>(s[0]) * g[0];
#pragma unroll 1
  for (int d = r; d >= 1; d--)
    acc = acc + (gn_val<MODE>(s[-d * st]) + gn_val<MODE>(s[d * st])) * g[d];
  return acc;
}

__host__ __device__ inline int gn_ksteps(int r, int step) { return (16 + 2 * r + step - 1) / step; }

// Pass 0 (axis 0) over the padded extent: tv = f32(sum g * where(nan, 0, x)),
// tw = f32(sum g * valid).  A tile whose input span holds no NaN has tw =
// f32(wsum) everywhere, wsum being the same accumulation over all-valid samples
// (on the host): it writes no tw but the mark -1 at its first pixel.
// LDS: the band, then 112 + 4 n_ks rows of 64 columns.  A lane's sample of the four
// column tiles is one 16-byte read: tile n has the columns 4 j + n, so a lane
// holds four consecutive outputs of a row.
template <int MODE>
__device__ __forceinline__ void gn_rows_mma(const float* s, const double* T, int n_ks, int lane,
                                            d4 (&acc)[2][4]) {
  const int k = lane >> 4, j = lane & 15;
#pragma unroll
  for (int n = 0; n < 4; n++) acc[0][n] = acc[1][n] = d4{0.0, 0.0, 0.0, 0.0};
  const float* p = s + k * GN_T + 4 * j;
  const double* tp = T + k - j + 15;
  auto step = [&](int ks, bool g0, bool g1) {
    const float4 v = *(const float4*)(p + 4 * ks * GN_T);
    const double x[4] = {gn_val<MODE>(v.x), gn_val<MODE>(v.y), gn_val<MODE>(v.z),
                         gn_val<MODE>(v.w)};
    if (g0) {
      const double a = tp[4 * ks];
#pragma unroll
      for (int n = 0; n < 4; n++)
        acc[0][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[n], acc[0][n], 0, 0, 0);
    }
    if (g1) {
      const double a = tp[4 * ks - 16];
#pragma unroll
      for (int n = 0; n < 4; n++)
        acc[1][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[n], acc[1][n], 0, 0, 0);
    }
  };
#pragma unroll 2
  for (int ks = 0; ks < 4; ks++) step(ks, true, false);
#pragma unroll 2
  for (int ks = 4; ks < n_ks; ks++) step(ks, true, true);
#pragma unroll 2
  for (int ks = n_ks; ks < n_ks + 4; ks++) step(ks, false, true);
}

__global__ __launch_bounds__(256, 2) void k_gauss_nan_rows(PadSrc S, GaussW G, int n_ks,
                                                        float* __restrict__ tv,
                                                        float* __restrict__ tw, int64_t ldt) {
  extern __shared__ __attribute__((aligned(16))) double gband[];
  const int n_band = (4 * n_ks + 16 + 1) & ~1;
  float* const gl = (float*)(gband + n_band);
  const int lane = threadIdx.x & 63;
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hp = S.h + 2 * S.pad, wp = S.w + 2 * S.pad;
  const int tx0 = blockIdx.x * GN_T, ty0 = blockIdx.y * GN_L;
  const int nrow = GN_L + 2 * G.r, npad = 112 + 4 * n_ks;
  GnBand B;
  B.get(G);
  bool nan = false, inf = false;
  // staging in batches of 32 rows per wave: with two blocks a CU, what a batch
  // waits for memory is hidden by little else
  const int wr0 = ty0 - G.r - S.pad, wc0 = tx0 - S.pad;   // window row and column of (0, 0)
  const bool inside = wr0 >= 0 && wr0 + nrow <= S.h && wc0 >= 0 && wc0 + GN_T <= S.w;
  const int pc = min(tx0 + lane, wp - 1);
  const float* const base = inside ? S.p + (int64_t)wr0 * S.ld + wc0 : S.p;
  const int wc = inside ? lane : sym(pc - S.pad, S.w);
  constexpr int GN_B = 32;
  for (int i0 = q; i0 < npad; i0 += 4 * GN_B) {
    float v[GN_B];
#pragma unroll
    for (int u = 0; u < GN_B; u++) {
      const int i = min(i0 + 4 * u, nrow - 1);
      const int row = inside ? i : sym(min(max(ty0 - G.r + i, 0), hp - 1) - S.pad, S.h);
      v[u] = (base + (int64_t)row * S.ld)[wc];
    }
#pragma unroll
    for (int u = 0; u < GN_B; u++) {
      const int i = i0 + 4 * u;
      if (i >= npad) break;
      const float x = i < nrow ? v[u] : 0.0f;
      gl[i * GN_T + lane] = x;
      nan |= isnan(x);
      inf |= isinf(x);
    }
  }
  B.put(gband, n_band);
  const bool any_nan = __syncthreads_or(nan);
  const bool any_inf = __syncthreads_or(inf);
  const int j = lane & 15;
  // entry e of the lane's groups: row y0 + 4 e, columns x .. x + 3
  const int x = tx0 + 4 * j, y0 = ty0 + q * 32 + (lane >> 4);
  auto store = [&](float* dst, const d4 (&acc)[2][4]) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int y = y0 + 4 * e;
      if (y >= hp) break;
      const d4 (&a)[4] = acc[e >> 2];
      const float v[4] = {(float)a[0][e & 3], (float)a[1][e & 3], (float)a[2][e & 3],
                          (float)a[3][e & 3]};
      float* o = dst + (int64_t)y * ldt + x;
      if (x + 3 < wp) {
        __builtin_memcpy(o, v, 16);
      } else {
#pragma unroll
        for (int n = 0; n < 3; n++)
          if (x + n < wp) o[n] = v[n];
      }
    }
  };
  if (any_inf) {
#pragma unroll 1
    for (int m = 0; m < 32; m++) {
      const int y = ty0 + q * 32 + m;
      if (y >= hp || tx0 + lane >= wp) break;
      const float* s = gl + (q * 32 + m + G.r) * GN_T + lane;
      const int64_t o = (int64_t)y * ldt + tx0 + lane;
      tv[o] = (float)gn_slow<1>(s, GN_T, gband, G.r);
      tw[o] = (float)gn_slow<2>(s, GN_T, gband, G.r);
    }
    return;
  }
  const float* s = gl + q * 32 * GN_T;
  d4 acc[2][4];
  if (!any_nan) {
    gn_rows_mma<0>(s, gband, n_ks, lane, acc);
    store(tv, acc);
    if (threadIdx.x == 0) tw[(int64_t)ty0 * ldt + tx0] = -1.0f;
    return;
  }
  gn_rows_mma<1>(s, gband, n_ks, lane, acc);
  store(tv, acc);
  gn_rows_mma<2>(s, gband, n_ks, lane, acc);
  store(tw, acc);
}

// Pass 1 (axis 1, 'nearest' along the padded rows) and where(sw > 0, sv / sw,
// 0) in float32.  Where every tile of the span is marked as without NaN, sw is
// the constant f32 of that accumulation (wdiv, from the host).
// LDS: the band, then 64 rows of P floats (P = 4 mod 64: the 16 rows of a 16-byte
// read spread over the banks) for the 112 + 16 n_ks samples, those past 128 + 2 r
// zero.  A step takes 16 samples: lane group k = l / 16 reads samples 4 k .. 4 k +
// 3 of its row at once, and MFMA t of the step takes sample 4 k + t.
__device__ __forceinline__ void gn_cols_mma(const float* s, int P, const double* T, int n_ks,
                                            int lane, d4 (&acc)[2][4]) {
  const int k = lane >> 4, j = lane & 15;
#pragma unroll
  for (int m = 0; m < 4; m++) acc[0][m] = acc[1][m] = d4{0.0, 0.0, 0.0, 0.0};
  const float* p = s + j * P + 4 * k;
  const double* tp = T + 4 * k - j + 15;
  double b[4] = {0.0, 0.0, 0.0, 0.0};   // the band of the step, which is the second
                                        // group's in the step after
  auto step = [&](int ks, bool g0, bool g1) {
    double c[4];
#pragma unroll
    for (int t = 0; t < 4; t++) c[t] = g0 ? tp[16 * ks + t] : 0.0;
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const float4 v = *(const float4*)(p + 16 * m * P + 16 * ks);
      const double x[4] = {(double)v.x, (double)v.y, (double)v.z, (double)v.w};
#pragma unroll
      for (int t = 0; t < 4; t++) {
        if (g0) acc[0][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], c[t], acc[0][m], 0, 0, 0);
        if (g1) acc[1][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], b[t], acc[1][m], 0, 0, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) b[t] = c[t];
  };
  step(0, true, false);
#pragma unroll 1
  for (int ks = 1; ks < n_ks; ks++) step(ks, true, true);
  step(n_ks, false, true);
}

__global__ __launch_bounds__(256, 2) void k_gauss_nan_cols(const float* __restrict__ tv,
                                                        const float* __restrict__ tw, int64_t ldt,
                                                        int hp, int wp, GaussW G, int n_ks, int P,
                                                        float* __restrict__ out, int64_t ldo,
                                                        float wconst, float wdiv) {
  extern __shared__ __attribute__((aligned(16))) double gband[];
  const int n_band = (16 * n_ks + 16 + 1) & ~1;
  float* const gl = (float*)(gband + n_band);
  const int lane = threadIdx.x & 63;
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tx0 = blockIdx.x * GN_L, ty0 = blockIdx.y * GN_T;
  const int ncol = GN_L + 2 * G.r, npad = 112 + 16 * n_ks;
  const float* const mark = tw + (int64_t)(ty0 / GN_L * GN_L) * ldt;   // of this row of tiles
  GnBand B;
  B.get(G);
  // the marks of the tiles that the span touches
  const int t_lo = max(tx0 - G.r, 0) / GN_T, t_hi = min(tx0 + GN_L - 1 + G.r, wp - 1) / GN_T;
  bool varied = false;
  for (int t = t_lo; t <= t_hi; t++) varied |= mark[t * GN_T] != -1.0f;
  // staging: two 64-column pieces of a wave's 16 rows in flight; weights: a marked
  // tile's tw is wconst
  auto stage = [&](const float* src, bool weights) {
    bool odd = false;
    for (int c = 0; c < npad; c += 128) {
      float v[2][16];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int col = min(max(tx0 - G.r + c + 64 * h + lane, 0), wp - 1);
#pragma unroll
        for (int u = 0; u < 16; u++)
          v[h][u] = (src + (int64_t)min(ty0 + q + 4 * u, hp - 1) * ldt)[col];
      }
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int j = c + 64 * h + lane;
        const int col = min(max(tx0 - G.r + j, 0), wp - 1);
        const bool marked = weights && mark[col / GN_T * GN_T] == -1.0f;
        if (j >= npad) continue;
#pragma unroll
        for (int u = 0; u < 16; u++) {
          const float x = j >= ncol ? 0.0f : marked ? wconst : v[h][u];
          gl[(q + 4 * u) * P + j] = x;
          odd |= !isfinite(x);
        }
      }
    }
    return odd;
  };
  // entry e of acc[g][m]: row ty0 + 16 m + l / 16 + 4 e, column tx0 + 32 q + 16 g + l % 16
  const float* s = gl + q * 32;
  d4 acc[2][4];
  float fw[2][4][4];
  B.put(gband, n_band);
  if (varied) {
    stage(tw, true);
    __syncthreads();
    gn_cols_mma(s, P, gband, n_ks, lane, acc);
    __syncthreads();
  }
#pragma unroll
  for (int g = 0; g < 2; g++)
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int e = 0; e < 4; e++) fw[g][m][e] = varied ? (float)acc[g][m][e] : wdiv;
  const bool odd = __syncthreads_or(stage(tv, false));
  if (!odd) gn_cols_mma(s, P, gband, n_ks, lane, acc);
#pragma unroll
  for (int g = 0; g < 2; g++)
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i = 16 * m + (lane >> 4) + 4 * e, c = 32 * q + 16 * g + (lane & 15);
        float v;
        if (odd)
          v = (float)gn_slow<0>(gl + i * P + c + G.r, 1, gband, G.r);
        else
          v = (float)acc[g][m][e];
        const float f = fw[g][m][e];
        if (tx0 + c < wp && ty0 + i < hp)
          out[(int64_t)(ty0 + i) * ldo + tx0 + c] = f > 0.0f ? v / f : 0.0f;
      }
}

// ---------------------------------------- the same passes on the vector units
//
// Small extents: the products' tiles of 128 x 64 leave most CUs idle there, and a
// tile's chain (twice the staging, a band and marks to read) is longer.  64 x 64
// tiles; each of the 4 waves of a block owns GN_M consecutive outputs along the
// filter axis for 64 lines across it, so one sample loaded from LDS into a
// register serves GN_M outputs: the pair (x[-d], x[+d]) of output m at distance d
// is x[m - d], x[m + d], and a block of GN_M distances reads two register windows
// of 2 GN_M - 1 samples that slide by GN_M per block.  Sums in scipy's symmetric
// order, as gn_slow's.
constexpr int GN_M = 16;   // outputs per lane along the filter axis (4 waves x 16 = 64)

// acc[m] = sum_k g[|k|] v(s[(m + k) ST]), k in [-r, r], in the order above.
// s points at the lane's first output; the LDS line holds r samples before
// it and r + GN_M - 1 after it.
template <int MODE, int ST>
__device__ __forceinline__ void gn_line(const float* s, const GaussW& G, double (&acc)[GN_M]) {
  const double g0 = G.g[0];
#pragma unroll
  for (int m = 0; m < GN_M; m++) acc[m] = gn_val<MODE>(s[m * ST]) * g0;
  int d = G.r;
  for (; d % GN_M != 0; d--) {   // the top r mod GN_M distances one at a time
    const double g = G.g[d];
#pragma unroll
    for (int m = 0; m < GN_M; m++)
      acc[m] = acc[m] + (gn_val<MODE>(s[(m - d) * ST]) + gn_val<MODE>(s[(m + d) * ST])) * g;
  }
  if (d == 0) return;
  // distances d .. d - GN_M + 1: L[k] = x[k - d], R[k] = x[k + d - GN_M + 1]
  double L[2 * GN_M - 1], R[2 * GN_M - 1];
#pragma unroll
  for (int k = 0; k < 2 * GN_M - 1; k++) {
    L[k] = gn_val<MODE>(s[(k - d) * ST]);
    R[k] = gn_val<MODE>(s[(k + d - (GN_M - 1)) * ST]);
  }
  for (;;) {
#pragma unroll
    for (int dd = 0; dd < GN_M; dd++) {
      const double g = G.g[d - dd];
#pragma unroll
      for (int m = 0; m < GN_M; m++) acc[m] = acc[m] + (L[m + dd] + R[m - dd + GN_M - 1]) * g;
    }
    d -= GN_M;
    if (d == 0) break;
#pragma unroll
    for (int k = 0; k < GN_M - 1; k++) L[k] = L[k + GN_M];
#pragma unroll
    for (int k = GN_M - 1; k < 2 * GN_M - 1; k++) L[k] = gn_val<MODE>(s[(k - d) * ST]);
#pragma unroll
    for (int k = 2 * GN_M - 2; k >= GN_M; k--) R[k] = R[k - GN_M];
#pragma unroll
    for (int k = 0; k < GN_M; k++) R[k] = gn_val<MODE>(s[(k + d - (GN_M - 1)) * ST]);
  }
}

// Pass 0: tv and tw as k_gauss_nan_rows forms them, tw written everywhere (f32(wsum)
// in a tile without NaN).  LDS: (64 + 2r) rows x 64 columns.
__global__ __launch_bounds__(256, 2) void k_gauss_tap_rows(PadSrc S, GaussW G,
                                                           float* __restrict__ tv,
                                                           float* __restrict__ tw, int64_t ldt,
                                                           float wconst) {
  extern __shared__ __attribute__((aligned(16))) float gl[];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int hp = S.h + 2 * S.pad, wp = S.w + 2 * S.pad;
  const int tx0 = blockIdx.x * GN_T, ty0 = blockIdx.y * GN_T;
  const int nrow = GN_T + 2 * G.r;
  const int pc = min(tx0 + lane, wp - 1);
  bool nan = false;
  // staging in batches of 8 rows per wave (8 loads in flight per lane)
  for (int i0 = q; i0 < nrow; i0 += 32) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + 4 * u;
      v[u] = i < nrow ? S.at(ty0 - G.r + i, pc) : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + 4 * u;
      if (i < nrow) {
        gl[i * GN_T + lane] = v[u];
        nan |= isnan(v[u]);
      }
    }
  }
  const bool any_nan = __syncthreads_or(nan);
  const float* s = gl + (q * GN_M + G.r) * GN_T + lane;
  const int x = tx0 + lane;
  const int y0 = ty0 + q * GN_M;
  const int nm = x < wp ? min(GN_M, hp - y0) : 0;   // rows this lane stores
  double acc[GN_M];
  if (any_nan) gn_line<1, GN_T>(s, G, acc);
  else gn_line<0, GN_T>(s, G, acc);
#pragma unroll
  for (int m = 0; m < GN_M; m++)
    if (m < nm) tv[(int64_t)(y0 + m) * ldt + x] = (float)acc[m];
  if (!any_nan) {
#pragma unroll
    for (int m = 0; m < GN_M; m++)
      if (m < nm) tw[(int64_t)(y0 + m) * ldt + x] = wconst;
    return;
  }
  gn_line<2, GN_T>(s, G, acc);
#pragma unroll
  for (int m = 0; m < GN_M; m++)
    if (m < nm) tw[(int64_t)(y0 + m) * ldt + x] = (float)acc[m];
}

// Pass 1.  A tile whose tw span is all f32(wsum) divides by the constant wdiv.  LDS:
// 64 rows x (64 + 2r + 1) columns (odd pitch: lanes walk rows without bank
// conflicts), reused for tw, tv and the transposed output tile.
__global__ __launch_bounds__(256, 2) void k_gauss_tap_cols(const float* __restrict__ tv,
                                                        const float* __restrict__ tw, int64_t ldt,
                                                        int hp, int wp, GaussW G,
                                                        float* __restrict__ out, int64_t ldo,
                                                        float wconst, float wdiv) {
  extern __shared__ __attribute__((aligned(16))) float gl[];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int tx0 = blockIdx.x * GN_T, ty0 = blockIdx.y * GN_T;
  const int ncol = GN_T + 2 * G.r, P = ncol + 1;
  // staging: column chunks of 64, each in batches of 8 rows per wave (8 loads in flight)
  auto stage = [&](const float* src) {
    bool off = false;
    for (int c = 0; c < ncol; c += 64) {
      const int j = c + lane;
      const bool jok = j < ncol;
      const int col = min(max(tx0 - G.r + j, 0), wp - 1);
#pragma unroll
      for (int k0 = 0; k0 < GN_T / 4; k0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int i = q + 4 * (k0 + u);
          v[u] = jok ? src[(int64_t)min(ty0 + i, hp - 1) * ldt + col] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int i = q + 4 * (k0 + u);
          if (jok) {
            gl[i * P + j] = v[u];
            off |= __float_as_uint(v[u]) != __float_as_uint(wconst);
          }
        }
      }
    }
    return off;
  };
  const float* s = gl + lane * P + q * GN_M + G.r;
  double acc[GN_M];
  float fw[GN_M], fo[GN_M];
  const bool varied = __syncthreads_or(stage(tw));
  if (varied) {
    gn_line<0, 1>(s, G, acc);
#pragma unroll
    for (int m = 0; m < GN_M; m++) fw[m] = (float)acc[m];
  } else {
#pragma unroll
    for (int m = 0; m < GN_M; m++) fw[m] = wdiv;
  }
  __syncthreads();
  stage(tv);
  __syncthreads();
  gn_line<0, 1>(s, G, acc);
#pragma unroll
  for (int m = 0; m < GN_M; m++) {
    const float v = (float)acc[m];
    fo[m] = fw[m] > 0.0f ? v / fw[m] : 0.0f;
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < GN_M; m++) gl[lane * (GN_T + 1) + q * GN_M + m] = fo[m];
  __syncthreads();
  const int x = tx0 + lane;
  if (x >= wp) return;
  for (int i = q; i < GN_T; i += 4) {
    const int y = ty0 + i;
    if (y < hp) out[(int64_t)y * ldo + x] = gl[i * (GN_T + 1) + lane];
  }
}

// The extents that take the vector units, by their 64 x 64 tiles.  Both passes in us,
// vector / products, without NaN and with 1 % of discs: r = 2 at 1024 tiles 40 / 42
// and 42 / 48, at 1444 53 / 49 and 54 / 55; r = 8 (its distances all one at a time)
// at 529 39 / 39 and 40 / 44, at 1024 49 / 44 and 58 / 50; r = 16 at 729 42 / 43 and
// 47 / 54, at 1089 60 / 57 and 63 / 71, at 1444 67 / 57 and 71 / 69; r = 32 at 729
// 53 / 51 and 62 / 69, at 1024 63 / 56 and 77 / 74; r = 64 at 529 75 / 69 and 82 / 97,
// at 729 77 / 68 and 108 / 99; r = 160 (one block a CU) at 256 76 / 81 and 111 / 130,
// at 289 132 / 80 and 170 / 131.
static bool gauss_vector(int hp, int wp, int r) {
  const int64_t tiles = (((int64_t)hp + GN_T - 1) / GN_T) * (((int64_t)wp + GN_T - 1) / GN_T);
  const int most = r <= 4 ? 1300 : r < 16 ? 700 : r <= 20 ? 1300 : r <= 32 ? 1000
                   : r <= 128 ? 600 : 256;
  return tiles <= most;
}

// The copies and interpolations below give a wave 256 columns, four per lane 64
// apart (each access 256 contiguous bytes), and `walk` rows of them: what a
// column or a pair of source rows determines is computed once per walk.  One
// pixel per thread redid it (and, for the interpolations, eight float64
// conversions and two lerps) for every output.
constexpr int ROW_WALK = 16;

struct Strip {
  int x, y0, rows;   // this lane's first column, the wave's rows
};
__device__ __forceinline__ Strip row_strip(int h, int walk) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Strip p;
  p.x = blockIdx.x * 256 + (threadIdx.x & 63);
  p.y0 = (blockIdx.y * 4 + wave) * walk;
  p.rows = min(walk, h - p.y0);
  return p;
}
// The rows of a wave: ROW_WALK, fewer where that would leave the launch less than
// WALK_WAVES waves (a walk is one wave's chain: 1024^2 overview samples 13.3 us in
// walks of 16 rows, 7.4 of 1, 7.2 one pixel per thread; 2048^2 15.5, 9.0 of 4,
// 11.9; upsampling 2048^2 9.3 of 4 rows, 10.9 of 2, 13.7 of 1), more where the
// grid's 65535 block rows would not cover the extent.
constexpr int64_t WALK_WAVES = 4096;
static int strip_walk(int w, int h) {
  constexpr int64_t max_rows = 4 * 65535;
  const int64_t rows = ((int64_t)w + 255) / 256 * h / WALK_WAVES;
  return (int)std::max(std::min<int64_t>(ROW_WALK, std::max<int64_t>(1, rows)),
                       (h + max_rows - 1) / max_rows);
}
static dim3 strip_grid(int w, int h, int walk) {
  const int64_t rows = 4 * (int64_t)walk;
  return dim3((unsigned)(((int64_t)w + 255) / 256), (unsigned)((h + rows - 1) / rows));
}

// 4096^2 padded by 32: 31 us, now 22.
__global__ void __launch_bounds__(256) k_pad_sym(PadSrc S, float* __restrict__ out, int64_t ldo,
                                                 int walk) {
  const int hp = S.h + 2 * S.pad, wp = S.w + 2 * S.pad;
  const Strip p = row_strip(hp, walk);
  int col[4];
#pragma unroll
  for (int m = 0; m < 4; m++) col[m] = sym(min(p.x + 64 * m, wp - 1) - S.pad, S.w);
  for (int y = 0; y < p.rows; y += 4) {
    float v[4][4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float* row =
          S.p + (int64_t)sym(p.y0 + min(y + k, p.rows - 1) - S.pad, S.h) * S.ld;
#pragma unroll
      for (int m = 0; m < 4; m++) v[k][m] = row[col[m]];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (y + k >= p.rows) break;
      float* o = out + (int64_t)(p.y0 + y + k) * ldo + p.x;
#pragma unroll
      for (int m = 0; m < 4; m++)
        if (p.x + 64 * m < wp) o[64 * m] = v[k][m];
    }
  }
}

// upsample_to_shape (_nan_utils.py:671-698): scipy zoom order 1, corner
// aligned (in = out * (n_in - 1) / (n_out - 1)), of where(nan, 0, x) and of
// valid, num / max(den, 1e-6) where den > 1e-3 else NaN; the zoom output
// shape round(n_in * (N / n_in)) is edge-padded (or cropped) to N.  A
// NaN-free source gives den = 1 and the plain zoom bit for bit.
// 1024^2 to 4096^2: 65 us, now 22.
__global__ void __launch_bounds__(256)
k_upsample_shape(const float* __restrict__ src, int64_t lds, int hs, int ws, int zh, int zw,
                 float* __restrict__ out, int64_t ldo, int h, int w, int walk) {
  const Strip p = row_strip(h, walk);
  if (p.rows <= 0) return;
  const double zx = zw > 1 ? (double)(ws - 1) / (double)(zw - 1) : 0.0;
  const double zy = zh > 1 ? (double)(hs - 1) / (double)(zh - 1) : 0.0;
  int x0[4], x1[4];
  double tx[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const int jj = min(p.x + 64 * m, zw - 1);   // edge padding past the zoom output
    const double cx = fmin(fmax((double)jj * zx, 0.0), (double)(ws - 1));
    x0[m] = (int)floor(cx);
    x1[m] = min(x0[m] + 1, ws - 1);
    tx[m] = cx - (double)x0[m];
  }
  auto fz = [](float v) { return isnan(v) ? 0.0 : (double)v; };
  auto vz = [](float v) { return isnan(v) ? 0.0 : 1.0; };
  // the two source rows of the walk, interpolated at the lane's columns
  double na[4], nb[4], da[4], db[4];
  int cur = -1;
  for (int y = 0; y < p.rows; y++) {
    const int ii = min(p.y0 + y, zh - 1);
    const double cy = fmin(fmax((double)ii * zy, 0.0), (double)(hs - 1));
    const int y0 = __builtin_amdgcn_readfirstlane((int)floor(cy)), y1 = min(y0 + 1, hs - 1);
    const double ty = cy - (double)y0, my = 1.0 - ty;
    if (y0 != cur) {
      cur = y0;
      const float* ra = src + (int64_t)y0 * lds;
      const float* rb = src + (int64_t)y1 * lds;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const float a = ra[x0[m]], b = ra[x1[m]], c = rb[x0[m]], d = rb[x1[m]];
        const double mx = 1.0 - tx[m];
        na[m] = fz(a) * mx + fz(b) * tx[m];
        nb[m] = fz(c) * mx + fz(d) * tx[m];
        da[m] = vz(a) * mx + vz(b) * tx[m];
        db[m] = vz(c) * mx + vz(d) * tx[m];
      }
    }
    float* o = out + (int64_t)(p.y0 + y) * ldo + p.x;
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const float fn = (float)(na[m] * my + nb[m] * ty), fd = (float)(da[m] * my + db[m] * ty);
      float v = fn;
      if (fd != 1.0f) v = fd > 1e-3f ? fn / fmaxf(fd, 1e-6f) : __builtin_nanf("");
      if (p.x + 64 * m < w) o[64 * m] = v;
    }
  }
}

// _bilinear_sample_coarse (_nan_utils.py:255-281): map_coordinates order 1,
// mode 'nearest', at float32 coordinates (g + 0.5) * f32(n_c / N) - 0.5 of the
// window's raster rows r0 + i and columns c0 + j; NaN where the window is NaN.
// 1024^2 overview, 4096^2 window: 42 us, now 30.
__global__ void __launch_bounds__(256)
k_sample_coarse(const float* __restrict__ coarse, int64_t ldc, int hc, int wc, int r0, int c0,
                float fy, float fx, const float* __restrict__ win, int64_t ldw,
                float* __restrict__ out, int64_t ldo, int h, int w, int walk) {
  const Strip p = row_strip(h, walk);
  if (p.rows <= 0) return;
  int x0[4], x1[4];
  double tx[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const float fxc = ((float)(c0 + min(p.x + 64 * m, w - 1)) + 0.5f) * fx - 0.5f;
    const double cx = fmin(fmax((double)fxc, 0.0), (double)(wc - 1));
    x0[m] = (int)floor(cx);
    x1[m] = min(x0[m] + 1, wc - 1);
    tx[m] = cx - (double)x0[m];
  }
  double top[4], bot[4];
  int cur = -1;
  for (int y = 0; y < p.rows; y++) {
    const int i = p.y0 + y;
    const float fyc = ((float)(r0 + i) + 0.5f) * fy - 0.5f;
    const double cy = fmin(fmax((double)fyc, 0.0), (double)(hc - 1));
    const int y0 = __builtin_amdgcn_readfirstlane((int)floor(cy)), y1 = min(y0 + 1, hc - 1);
    const double ty = cy - (double)y0, my = 1.0 - ty;
    float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (win) {
#pragma unroll
      for (int m = 0; m < 4; m++) z[m] = (win + (int64_t)i * ldw)[min(p.x + 64 * m, w - 1)];
    }
    if (y0 != cur) {
      cur = y0;
      const float* ra = coarse + (int64_t)y0 * ldc;
      const float* rb = coarse + (int64_t)y1 * ldc;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const double mx = 1.0 - tx[m];
        top[m] = (double)ra[x0[m]] * mx + (double)ra[x1[m]] * tx[m];
        bot[m] = (double)rb[x0[m]] * mx + (double)rb[x1[m]] * tx[m];
      }
    }
    float* o = out + (int64_t)i * ldo + p.x;
#pragma unroll
    for (int m = 0; m < 4; m++) {
      float v = (float)(top[m] * my + bot[m] * ty);
      if (isnan(z[m])) v = __builtin_nanf("");
      if (p.x + 64 * m < w) o[64 * m] = v;
    }
  }
}

constexpr int CMB_MAX = 16;
struct CombineArgs {
  const float* f[CMB_MAX];
  int64_t ld;
  int n, agg;           // FSG_AGG_*
  float w[CMB_MAX];
  int h, w_;
};

// _combine_multiscale_dask (_nan_utils.py:182-213) and hillshade's inline
// variant: weighted sum out = f0 * w0 (+ f_i * w_i in order), or the float32
// mean / min / max / sum over the fields; then the output epilogue.
// Bound: memory, (n + 1) x 4 bytes a pixel; four consecutive columns per lane (16-byte
// accesses, dword-aligned) and the agg chosen once.  4096^2, five fields: 170 us, now 110.
template <int AGG>
__device__ __forceinline__ void combine_rows(const CombineArgs& A, const OutDev& o) {
  const int j = blockIdx.x * 256 + (threadIdx.x & 63) * 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (j >= A.w_) return;
  const PostK pp = load_post(o);
  const int n4 = min(4, A.w_ - j);
  for (int i = blockIdx.y * 4 + wave; i < A.h; i += gridDim.y * 4) {
    const int64_t e = (int64_t)i * A.ld + j;
    float v[4];
    for (int k = 0; k < A.n; k++) {
      float x[4];
      if (n4 == 4) {
        __builtin_memcpy(x, A.f[k] + e, 16);
      } else {
#pragma unroll
        for (int m = 0; m < 4; m++) x[m] = A.f[k][e + min(m, n4 - 1)];
      }
      const float w = A.w[k];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        if (AGG == FSG_AGG_WEIGHTED) x[m] = x[m] * w;
        if (k == 0) {
          v[m] = x[m];
        } else if (AGG == FSG_AGG_MAX || AGG == FSG_AGG_MIN) {
          v[m] = (isnan(v[m]) || isnan(x[m])) ? __builtin_nanf("")
                 : AGG == FSG_AGG_MAX ? fmaxf(v[m], x[m]) : fminf(v[m], x[m]);
        } else {
          v[m] = v[m] + x[m];
        }
      }
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
      if (AGG == FSG_AGG_MEAN) v[m] = v[m] / (float)A.n;
      v[m] = post_value(pp, v[m]);
    }
    store_out4(o, i, j, v, 0, n4, n4 == 4);
  }
}

__global__ void __launch_bounds__(256) k_combine(CombineArgs A, OutDev o) {
  switch (A.agg) {
    case FSG_AGG_WEIGHTED: combine_rows<FSG_AGG_WEIGHTED>(A, o); break;
    case FSG_AGG_MEAN: combine_rows<FSG_AGG_MEAN>(A, o); break;
    case FSG_AGG_SUM: combine_rows<FSG_AGG_SUM>(A, o); break;
    case FSG_AGG_MAX: combine_rows<FSG_AGG_MAX>(A, o); break;
    default: combine_rows<FSG_AGG_MIN>(A, o); break;
  }
}

static dim3 grid2(int w, int h) {
  return dim3((unsigned)((w + 255) / 256), (unsigned)std::min(h, 16384));
}

}  // namespace fsg

using namespace fsg;

extern "C" size_t fsg_gaussian_nan_workspace_size(int32_t h, int32_t w, int32_t pad) {
  if (h <= 0 || w <= 0 || pad < 0) return 0;
  return 2 * ((sizeof(float) * (size_t)(h + 2 * pad) * (w + 2 * pad) + 255) & ~(size_t)255);
}

extern "C" int fsg_gaussian_nan(const fsg_window* src, int32_t pad, double sigma, float* out,
                                int64_t ldo, void* workspace, size_t workspace_bytes,
                                void* stream) {
  int rc = validate_window(src, "fsg_gaussian_nan");
  if (rc) return rc;
  if (src->h <= 0 || src->w <= 0 || pad < 0 || pad > std::min(src->h, src->w) || !out ||
      !(sigma > 0.0))
    return fail(FSG_E_INVALID, "fsg_gaussian_nan: bad arguments (pad must be <= the window)");
  const int hp = src->h + 2 * pad, wp = src->w + 2 * pad;
  if (ldo < wp) return fail(FSG_E_INVALID, "fsg_gaussian_nan: ldo smaller than the padded width");
  const size_t need = fsg_gaussian_nan_workspace_size(src->h, src->w, pad);
  if (!workspace || workspace_bytes < need)
    return fail(FSG_E_WORKSPACE, "fsg_gaussian_nan: workspace too small");
  GaussW G{};
  G.r = (int)(4.0 * sigma + 0.5);   // scipy truncate = 4.0
  if (G.r > GN_MAX_R) return fail(FSG_E_UNSUPPORTED, "fsg_gaussian_nan: sigma above 40");
  std::vector<double> full(2 * G.r + 1);
  gaussian_weights(sigma, G.r, full.data());
  for (int d = 0; d <= G.r; d++) G.g[d] = full[G.r + d];
  // the all-valid accumulations: pass 0 over validity 1, pass 1 over f32 of that
  double w0 = 1.0 * G.g[0];
  for (int d = G.r; d >= 1; d--) w0 = w0 + (1.0 + 1.0) * G.g[d];
  const float wconst = (float)w0;
  double w1 = (double)wconst * G.g[0];
  for (int d = G.r; d >= 1; d--) w1 = w1 + ((double)wconst + (double)wconst) * G.g[d];
  const float wdiv = (float)w1;
  float* tv = (float*)workspace;
  float* tw = (float*)((char*)workspace + need / 2);
  hipStream_t s = as_stream(stream);
  PadSrc S{src->data, src->ld, src->h, src->w, pad};
  TimedScope ts("k_gauss_nan", s);
  if (gauss_vector(hp, wp, G.r)) {
    const dim3 grid((wp + GN_T - 1) / GN_T, (hp + GN_T - 1) / GN_T);
    const size_t lds_r = sizeof(float) * (GN_T + 2 * G.r) * GN_T;
    const size_t lds_c = sizeof(float) * GN_T * (GN_T + 2 * G.r + 1);
    hipLaunchKernelGGL(k_gauss_tap_rows, grid, dim3(256), lds_r, s, S, G, tv, tw, (int64_t)wp,
                       wconst);
    FSG_CHECK_LAUNCH("k_gauss_tap_rows");
    hipLaunchKernelGGL(k_gauss_tap_cols, grid, dim3(256), lds_c, s, tv, tw, (int64_t)wp, hp, wp,
                       G, out, ldo, wconst, wdiv);
    FSG_CHECK_LAUNCH("k_gauss_tap_cols");
    return FSG_OK;
  }
  const dim3 grid_r((wp + GN_T - 1) / GN_T, (hp + GN_L - 1) / GN_L);
  const dim3 grid_c((wp + GN_L - 1) / GN_L, (hp + GN_T - 1) / GN_T);
  const int ks_r = gn_ksteps(G.r, 4), ks_c = gn_ksteps(G.r, 16);
  const int P = (112 + 16 * ks_c + 63) / 64 * 64 + 4;
  const size_t lds_r =
      sizeof(double) * ((4 * ks_r + 17) & ~1) + sizeof(float) * (112 + 4 * ks_r) * GN_T;
  const size_t lds_c = sizeof(double) * ((16 * ks_c + 17) & ~1) + sizeof(float) * GN_T * P;
  hipLaunchKernelGGL(k_gauss_nan_rows, grid_r, dim3(256), lds_r, s, S, G, ks_r, tv, tw,
                     (int64_t)wp);
  FSG_CHECK_LAUNCH("k_gauss_nan_rows");
  hipLaunchKernelGGL(k_gauss_nan_cols, grid_c, dim3(256), lds_c, s, tv, tw, (int64_t)wp, hp, wp, G,
                     ks_c, P, out, ldo, wconst, wdiv);
  FSG_CHECK_LAUNCH("k_gauss_nan_cols");
  return FSG_OK;
}

extern "C" int fsg_pad_symmetric(const fsg_window* src, int32_t pad, float* out, int64_t ldo,
                                 void* stream) {
  int rc = validate_window(src, "fsg_pad_symmetric");
  if (rc) return rc;
  if (src->h <= 0 || src->w <= 0 || pad < 0 || pad > std::min(src->h, src->w) || !out ||
      ldo < src->w + 2 * pad)
    return fail(FSG_E_INVALID, "fsg_pad_symmetric: bad arguments (pad must be <= the window)");
  const int hp = src->h + 2 * pad, wp = src->w + 2 * pad;
  PadSrc S{src->data, src->ld, src->h, src->w, pad};
  const int walk = strip_walk(wp, hp);
  hipLaunchKernelGGL(k_pad_sym, strip_grid(wp, hp, walk), dim3(256), 0, as_stream(stream), S, out,
                     ldo, walk);
  FSG_CHECK_LAUNCH("k_pad_sym");
  return FSG_OK;
}

// dask map_overlap boundary='reflect' at the raster edges of a window: each
// side padded by its own amount with numpy's 'symmetric' rule
__global__ void k_pad_sides(const float* __restrict__ src, int64_t lds, int h, int w, int top,
                            int left, float* __restrict__ out, int64_t ldo, int ho, int wo) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= wo) return;
  const int sc = sym(c - left, w);
  for (int r = blockIdx.y; r < ho; r += gridDim.y)
    out[(int64_t)r * ldo + c] = src[(int64_t)sym(r - top, h) * lds + sc];
}

extern "C" int fsg_pad_reflect(const fsg_window* src, int32_t top, int32_t bottom, int32_t left,
                               int32_t right, float* out, int64_t ldo, void* stream) {
  int rc = validate_window(src, "fsg_pad_reflect");
  if (rc) return rc;
  if (src->h <= 0 || src->w <= 0 || !out || top < 0 || bottom < 0 || left < 0 || right < 0 ||
      std::max(top, bottom) > src->h || std::max(left, right) > src->w ||
      ldo < (int64_t)src->w + left + right)
    return fail(FSG_E_INVALID,
                "fsg_pad_reflect: bad arguments (each pad at most the window extent)");
  const int ho = src->h + top + bottom, wo = src->w + left + right;
  hipLaunchKernelGGL(k_pad_sides, grid2(wo, ho), dim3(256), 0, as_stream(stream), src->data,
                     src->ld, src->h, src->w, top, left, out, ldo, ho, wo);
  FSG_CHECK_LAUNCH("k_pad_sides");
  return FSG_OK;
}

extern "C" int fsg_upsample_to_shape(const float* src, int64_t lds, int32_t hs, int32_t ws,
                                     float* out, int64_t ldo, int32_t h, int32_t w,
                                     void* stream) {
  if (!src || !out || hs <= 0 || ws <= 0 || h <= 0 || w <= 0 || lds < ws || ldo < w)
    return fail(FSG_E_INVALID, "fsg_upsample_to_shape: bad arguments");
  // scipy zoom output shape: round(n_in * (N / n_in))
  const int zh = (int)std::nearbyint((double)hs * ((double)h / (double)hs));
  const int zw = (int)std::nearbyint((double)ws * ((double)w / (double)ws));
  const int walk = strip_walk(w, h);
  hipLaunchKernelGGL(k_upsample_shape, strip_grid(w, h, walk), dim3(256), 0, as_stream(stream), src,
                     lds, hs, ws, std::max(1, zh), std::max(1, zw), out, ldo, h, w, walk);
  FSG_CHECK_LAUNCH("k_upsample_shape");
  return FSG_OK;
}

extern "C" int fsg_sample_coarse(const float* coarse, int64_t ldc, int32_t hc, int32_t wc,
                                 int32_t r0, int32_t c0, int32_t full_h, int32_t full_w,
                                 const float* nan_src, int64_t ld_nan, float* out, int64_t ldo,
                                 int32_t h, int32_t w, void* stream) {
  if (!coarse || !out || hc <= 0 || wc <= 0 || full_h <= 0 || full_w <= 0 || h <= 0 || w <= 0 ||
      ldc < wc || ldo < w || (nan_src && ld_nan < w))
    return fail(FSG_E_INVALID, "fsg_sample_coarse: bad arguments");
  const float fy = (float)((double)hc / (double)full_h), fx = (float)((double)wc / (double)full_w);
  const int walk = strip_walk(w, h);
  hipLaunchKernelGGL(k_sample_coarse, strip_grid(w, h, walk), dim3(256), 0, as_stream(stream),
                     coarse, ldc, hc, wc, r0, c0, fy, fx, nan_src, ld_nan, out, ldo, h, w, walk);
  FSG_CHECK_LAUNCH("k_sample_coarse");
  return FSG_OK;
}

extern "C" int fsg_combine_fields(const float* const* fields, int32_t n, int64_t ld,
                                  const float* weights, int32_t agg, int32_t h, int32_t w,
                                  const fsg_output* out, void* stream) {
  if (!fields || n <= 0 || n > CMB_MAX || h <= 0 || w <= 0 || ld < w || !out ||
      agg < FSG_AGG_WEIGHTED || agg > FSG_AGG_MIN || (agg == FSG_AGG_WEIGHTED && !weights))
    return fail(FSG_E_INVALID, "fsg_combine_fields: bad arguments");
  fsg_region reg{0, 0, h, w};
  int rc = validate_output(out, &reg, "fsg_combine_fields");
  if (rc) return rc;
  CombineArgs A{};
  for (int k = 0; k < n; k++) {
    if (!fields[k]) return fail(FSG_E_INVALID, "fsg_combine_fields: field NULL");
    A.f[k] = fields[k];
    A.w[k] = weights ? weights[k] : 0.0f;
  }
  A.ld = ld;
  A.n = n;
  A.agg = agg;
  A.h = h;
  A.w_ = w;
  hipLaunchKernelGGL(k_combine,
                     dim3((unsigned)((w + 255) / 256), (unsigned)std::min((h + 3) / 4, 4096)),
                     dim3(256), 0, as_stream(stream), A, make_out(out));
  FSG_CHECK_LAUNCH("k_combine");
  return FSG_OK;
}
