// Ray marches: sparse Yokoyama openness and stylised ambient occlusion.
//
// Openness (compute_openness_vectorized, _impl_openness.py:31-132): per
// direction the horizon extreme of atan((z_s - z) / d) over the valid
// in-window samples.  atan is monotone, so the kernel takes the extreme of the
// slope ratio and evaluates one atanf per direction instead of one per sample
// (AngleSum).
// The ratio uses f32(1/phys) multiplication (within 1.5 ulp of the reference's
// division by f32(phys)).
//
// Ambient occlusion (compute_ambient_occlusion_block,
// _impl_ambient_occlusion.py:32-121): edge-padded samples, clamp(atan,0,pi/4),
// ring weighting, mean over valid samples, then a sigma=1 'nearest' Gaussian
// (scipy two-pass order) of where(nan, 1, ao), gamma, NaN restored.
#include <algorithm>
#include <cmath>

#include <string>

#include "rays.hpp"

namespace fsg {

// Block order of the ray kernels on a 1-D grid.  With at least 8 block columns
// the region is cut into 8 column panels, one per XCD (workgroup b runs on XCD
// b mod 8), walked row by row inside the panel: the rows an XCD's resident
// blocks sample (their own plus the rays' vertical reach) then span one panel's
// width, not the whole region's, and stay in that XCD's L2.  Narrower regions
// keep the plain row-major order.
struct RayGrid {
  int nbx, nby;   // block columns and rows of the region
  int pw;         // blocks per panel row (0: row-major)
};

inline RayGrid ray_grid(int h, int w, int bh, int bw) {
  RayGrid G;
  G.nbx = (w + bw - 1) / bw;
  G.nby = (h + bh - 1) / bh;
  G.pw = G.nbx >= 8 ? (G.nbx + 7) / 8 : 0;
  return G;
}

inline int64_t ray_grid_blocks(const RayGrid& G) {
  return G.pw ? (int64_t)8 * G.pw * G.nby : (int64_t)G.nbx * G.nby;
}

// (bx, by) of block b; false for the padding blocks of the last panel
__device__ __forceinline__ bool ray_block(const RayGrid& G, int b, int& bx, int& by) {
  if (G.pw == 0) {
    by = b / G.nbx;
    bx = b - by * G.nbx;
    return true;
  }
  const int xcd = b & 7, k = b >> 3;
  by = k / G.pw;
  bx = xcd * G.pw + (k - by * G.pw);
  return bx < G.nbx && by < G.nby;
}

// ND: the table's distances per direction when it is 1 .. 10 (fixed-length
// rows: wide scalar table loads, no guards), 0 for any other count.
template <int ND>
__global__ void __launch_bounds__(256)
k_openness(WinDevR W, int r0, int c0, int rh, int rw, OpenTab T, OutDev out, RayGrid G) {
  int bx, by;
  if (!ray_block(G, blockIdx.x, bx, by)) return;
  const int c = bx * 64 + threadIdx.x;
  const int r = by * 4 + threadIdx.y;
  // block-uniform: do all samples of the block's pixels stay inside the window?
  const int bi0 = r0 + by * 4, bj0 = c0 + bx * 64;
  const bool interior = openness_interior(W, T, bi0, bi0 + 3, bj0, bj0 + 63);
  if (c >= rw || r >= rh) return;
  const int i = r0 + r, j = c0 + c;
  const PostK pp = load_post(out);
  const float z = W.p[(int64_t)i * W.ld + j];
  if (isnan(z)) {
    store_out(out, r, c, apply_post(pp, __builtin_nanf("")));
    return;
  }
  float a;
  if constexpr (ND > 0)
    a = !interior ? openness_angle_u<ND, true>(W, i, j, z, T)
        : open_off32(W, T) ? openness_angle_u<ND, false, true>(W, i, j, z, T)
                        : openness_angle_u<ND, false>(W, i, j, z, T);
  else
    a = openness_angle_at(W, i, j, z, T, interior);
  store_out(out, r, c, apply_post(pp, openness_value(T, a)));
}

// ------------------------------------------------ tiles staged in LDS
//
// Sampling straight from memory costs about 10 cycles of a CU's L1 per wave and
// sample: a ray's samples start at any column, so a wave's 256 bytes straddle
// its lines, and the 64 to 160 samples of a pixel are what the launch spends
// its time on (16-byte loads of four pixels were three times slower still:
// 8736 against 2739 us at 8192^2, 16 directions).  An LDS read takes 2 at any
// alignment.  So a workgroup of 16 waves stages its tile of RT_W columns with
// the rays' reach around it, once, and samples that: address = the lane's +
// one scalar per sample.  Samples outside the window are staged as the caller's
// rule has them (NaN for openness, the edge for AO): no interior test.  What
// bounds it now is VALU issue: a difference, a product and an extreme per sample, and
// an atanf per direction.  8192^2 from memory / staged, in us: 16 directions of 50
// pixels 2737 / 1591, 8 of 64 1496 / 1231, 16 of 8 2248 / 1097.
constexpr int RT_W = 128;             // tile columns: two per lane, 64 apart
constexpr int RT_LDS = 160 * 1024;    // a CU's LDS
constexpr int RT_LDS_HALF = 80 * 1024;
constexpr int RT_PIECES = 5;          // 64-column pieces of a staged row
constexpr int64_t RT_MIN_PX = 9 << 14;
constexpr int64_t RT_MIN_PX_NEAR = (1 << 18) + 1;   // openness, a reach of 16 or less

struct RayTile {
  RayGrid G;
  int th;            // tile rows
  int dy, dx;        // reach on each axis
  int pitch;         // floats per staged row (RT_W + 2 dx)
  int lds;           // bytes
};

// The tile of a region, or th = 0 where the reach leaves LDS no 16 rows (beyond
// 68 pixels) or the region has fewer than min_px pixels, where too few tiles share
// the staging.  From memory / staged, in us: openness at 384^2, 16 directions of 50
// pixels 25 / 17, 8 of 64 14.2 / 12.2, 8 of 24 11.9 / 10.1, but 16 of 16 13.6 / 15.1
// and 8 of 8 8.1 / 9.3 (rays that stay in a few rows hit L1), at 512^2 14.0 / 15.0
// and 8.5 / 9.3, at 576^2 24 / 17 and 13.4 / 11.3; at 300^2 8 of 64 11.4 / 12.1.  AO
// with its smoothing at 384^2, 16 samples a ring of radius 10 30.5 / 25.6, 8 of 64
// 23.8 / 24.2.  Two tiles a CU where 48 rows or more fit half the LDS (one computes
// while the other stages), else one of what fits; then the rows of the fewest full
// rounds of tiles, spread evenly (regions of one round: down to 8 rows).
inline RayTile ray_tile(int h, int w, int dy, int dx, int64_t min_px = RT_MIN_PX) {
  RayTile R{};
  R.dy = dy;
  R.dx = dx;
  R.pitch = RT_W + 2 * dx;
  if (R.pitch > 64 * RT_PIECES || w < 64 || (int64_t)h * w < min_px) return R;
  const int half = RT_LDS_HALF / 4 / R.pitch - 2 * dy, full = RT_LDS / 4 / R.pitch - 2 * dy;
  const int th = half >= 48 ? half : full, slots = half >= 48 ? 512 : 256;
  if (th < 16) return R;
  const int64_t nbx = (w + RT_W - 1) / RT_W;
  const int64_t rounds = (nbx * ((h + th - 1) / th) + slots - 1) / slots;
  const int64_t nby = std::max<int64_t>((h + th - 1) / th, rounds * slots / nbx);
  R.th = std::min(th, std::max(8, (int)((h + nby - 1) / nby)));
  R.G = ray_grid(h, w, R.th, RT_W);
  R.lds = (R.th + 2 * dy) * R.pitch * 4;
  return R;
}

// rows [i0, i0 + rows) x columns [j0, j0 + pitch) of the window into LDS; EDGE:
// clamped to the window, else NaN outside it.  A wave takes every 16th row; four
// rows' loads (up to five 64-column pieces each) are in flight together.  The
// staged values are several times the tile's, so a tile inside the window takes
// a path without per-value arithmetic.
template <bool EDGE, bool INSIDE>
__device__ __forceinline__ void stage_rows(const WinDevR& W, int i0, int rows, int j0, int pitch,
                                           float* lds) {
  const unsigned lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int jc[RT_PIECES];
#pragma unroll
  for (int q = 0; q < RT_PIECES; q++) jc[q] = INSIDE ? 0 : clampi(j0 + (int)lane + 64 * q, W.w);
  for (int k0 = wave; k0 < rows; k0 += 64) {
    float v[4][RT_PIECES];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int i = i0 + min(k0 + 16 * u, rows - 1);
      const float* row = W.p + (int64_t)(INSIDE ? i : clampi(i, W.h)) * W.ld;
#pragma unroll
      for (int q = 0; q < RT_PIECES; q++) {
        if (64 * q >= pitch) break;
        if (INSIDE) {
          if (64 * q + 64 <= pitch || (int)lane + 64 * q < pitch)
            v[u][q] = (row + j0 + 64 * q)[lane];
        } else {
          v[u][q] = row[jc[q]];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int k = k0 + 16 * u;
      if (k >= rows) break;
      const bool iok = INSIDE || (i0 + k >= 0 && i0 + k < W.h);
      float* d = lds + k * pitch + lane;
#pragma unroll
      for (int q = 0; q < RT_PIECES; q++) {
        if (64 * q >= pitch) break;
        const float x = INSIDE || EDGE || (iok && j0 + (int)lane + 64 * q == jc[q])
                            ? v[u][q] : __builtin_nanf("");
        if (64 * q + 64 <= pitch || (int)lane + 64 * q < pitch) d[64 * q] = x;
      }
    }
  }
}

template <bool EDGE>
__device__ __forceinline__ void stage_tile(const WinDevR& W, int i0, int rows, int j0, int pitch,
                                           float* lds) {
  if (i0 >= 0 && i0 + rows <= W.h && j0 >= 0 && j0 + pitch <= W.w)
    stage_rows<EDGE, true>(W, i0, rows, j0, pitch, lds);
  else
    stage_rows<EDGE, false>(W, i0, rows, j0, pitch, lds);
}

// The tile kernels' tables hold each sample's LDS byte offset in place of its
// (dx, dy): kernel arguments of both would pass 4 KB.
inline short2 lds_offset(short2 o, const RayTile& R) {
  return __builtin_bit_cast(short2, (o.y * R.pitch + o.x) * 4);
}
__device__ __forceinline__ const float* lds_sample(const char* at, short2 off) {
  return (const float*)(at + __builtin_bit_cast(int, off));
}

// Openness of a staged tile: same ratios, extremes and AngleSum as
// openness_angle_s, so the same bits.
template <int ND, bool NEG>
__device__ __forceinline__ void openness_pair(const char* at, const float z[2], const OpenTab& T,
                                              float out[2]) {
  AngleSum S[2];
  for (int d = 0; d < T.n_dirs; d++) {
    float v[ND][2];
#pragma unroll
    for (int k = 0; k < ND; k++) {
      const float* p = lds_sample(at, T.off[d * ND + k]);
      v[k][0] = p[0];
      v[k][1] = p[64];
    }
    float ext[2] = {__builtin_nanf(""), __builtin_nanf("")};
#pragma unroll
    for (int k = 0; k < ND; k++) {
      const float inv = T.inv[d * ND + k];
#pragma unroll
      for (int m = 0; m < 2; m++) {
        const float q = (v[k][m] - z[m]) * inv;
        ext[m] = NEG ? fminf(ext[m], q) : fmaxf(ext[m], q);
      }
    }
    // a direction without a valid sample is rare: one vote for the wave
    if (__builtin_amdgcn_ballot_w64(__builtin_isunordered(ext[0], ext[1])) == 0) {
      S[0].add<NEG>(ext[0]);
      S[1].add<NEG>(ext[1]);
    } else {
#pragma unroll
      for (int m = 0; m < 2; m++)
        if (!isnan(ext[m])) S[m].add<NEG>(ext[m]);
    }
  }
  out[0] = S[0].mean();
  out[1] = S[1].mean();
}

template <int ND>
__global__ void __launch_bounds__(1024)
k_openness_tile(WinDevR W, int r0, int c0, int rh, int rw, OpenTab T, RayTile R,
                OutDev out) {
  extern __shared__ __attribute__((aligned(16))) float rt[];
  int bx, by;
  if (!ray_block(R.G, blockIdx.x, bx, by)) return;
  const int y0 = by * R.th, rows = min(R.th, rh - y0), x0 = bx * RT_W;
  stage_tile<false>(W, r0 + y0 - R.dy, rows + 2 * R.dy, c0 + x0 - R.dx, R.pitch, rt);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const PostK pp = load_post(out);
  for (int y = wave; y < rows; y += 16) {
    const float* at = rt + (y + R.dy) * R.pitch + R.dx + lane;
    const float z[2] = {at[0], at[64]};
    // a NaN pixel's ratios would all be NaN (and its columns past the window too)
    const float zv[2] = {isnan(z[0]) ? 0.0f : z[0], isnan(z[1]) ? 0.0f : z[1]};
    float a[2];
    if (T.negative)
      openness_pair<ND, true>((const char*)at, zv, T, a);
    else
      openness_pair<ND, false>((const char*)at, zv, T, a);
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const int c = x0 + lane + 64 * m;
      if (c < rw)
        store_out(out, y0 + y, c, apply_post(pp, isnan(z[m]) ? z[m] : openness_value(T, a[m])));
    }
  }
}

// The same at a list of window pixels (row, col), float32 out[n].
__global__ void __launch_bounds__(256)
k_openness_points(WinDevR W, const int2* __restrict__ pts, int n, OpenTab T,
                  float* __restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int2 q = pts[e];
  // a point outside the window reads nothing and gets NaN
  if (q.x < 0 || q.x >= W.h || q.y < 0 || q.y >= W.w) {
    out[e] = __builtin_nanf("");
    return;
  }
  const float z = W.p[(int64_t)q.x * W.ld + q.y];
  out[e] = isnan(z) ? __builtin_nanf("")
                    : openness_value(T, openness_angle_at(W, q.x, q.y, z, T, false));
}

// Sampled exact check of an approximate openness-angle raster (the learned
// surrogate's judge; no reference counterpart).  The window is cut into
// tile_h x tile_w tiles (ragged at the far edges); tile t (row-major) gets
// n_t = max(1, ceil(frac * th * tw / L)) segments of L pixels along one row,
// segment k at
//   h = splitmix64(splitmix64(seed ^ splitmix64(t)) + k),
//   row = y0 + (h >> 32) % th,  col0 = x0 + (h & 0xffffffff) % (tw - L + 1).
// One wave per segment, lane = pixel, so the ray gathers coalesce as in the
// dense kernel.  Block (t, split) takes segments split*4 + wave, +
// JUDGE_SPLIT*4, ... and writes the sum and count of |exact - approx| over
// pixels where both are numbers; the reduction order is fixed, so the result
// is deterministic.
constexpr int JUDGE_SPLIT = 64;

__host__ __device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

struct JudgeGeo {
  int tile_h, tile_w, n_tx, L;
  double frac;
  uint64_t seed;
};

__device__ __forceinline__ int judge_count(const JudgeGeo& G, int th, int tw) {
  return max(1, (int)ceil(G.frac * (double)th * (double)tw / (double)G.L));
}

__global__ void __launch_bounds__(256)
k_openness_judge(WinDevR W, OpenTab T, const float* __restrict__ approx, int64_t lda, JudgeGeo G,
                 double* __restrict__ part) {
  const int tile = blockIdx.x / JUDGE_SPLIT, split = blockIdx.x % JUDGE_SPLIT;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int y0 = (tile / G.n_tx) * G.tile_h, x0 = (tile % G.n_tx) * G.tile_w;
  const int th = min(G.tile_h, W.h - y0), tw = min(G.tile_w, W.w - x0);
  const int n_seg = judge_count(G, th, tw);
  const uint64_t key = splitmix64(G.seed ^ splitmix64((uint64_t)tile));
  float sum = 0.0f, cnt = 0.0f;
  for (int s = split * 4 + wave; s < n_seg; s += JUDGE_SPLIT * 4) {
    const uint64_t h = splitmix64(key + (uint64_t)s);
    const int i = y0 + (int)((h >> 32) % (uint64_t)th);
    const int jseg = x0 + (int)((h & 0xffffffffull) % (uint64_t)(tw - G.L + 1));
    const int j = jseg + lane;
    const bool interior = openness_interior(W, T, i, i, jseg, jseg + G.L - 1);
    if (lane < G.L) {
      const float z = W.p[(int64_t)i * W.ld + j];
      const float a = approx[(int64_t)i * lda + j];
      if (!isnan(z) && !isnan(a)) {
        const float v = openness_value(T, openness_angle_at(W, i, j, z, T, interior));
        sum += fabsf(v - a);
        cnt += 1.0f;
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    sum += __shfl_down(sum, o);
    cnt += __shfl_down(cnt, o);
  }
  __shared__ double red[4][2];
  if (lane == 0) {
    red[wave][0] = sum;
    red[wave][1] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double ps = 0.0, pc = 0.0;
    for (int w = 0; w < 4; w++) {
      ps += red[w][0];
      pc += red[w][1];
    }
    part[(int64_t)blockIdx.x * 2] = ps;
    part[(int64_t)blockIdx.x * 2 + 1] = pc;
  }
}

// mean absolute error per tile (NaN for a tile without a valid sample)
__global__ void k_openness_judge_finish(const double* __restrict__ part, int n_tiles,
                                        float* __restrict__ tile_mae) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tiles) return;
  double s = 0.0, c = 0.0;
  for (int k = 0; k < JUDGE_SPLIT; k++) {
    s += part[((int64_t)t * JUDGE_SPLIT + k) * 2];
    c += part[((int64_t)t * JUDGE_SPLIT + k) * 2 + 1];
  }
  tile_mae[t] = c > 0.0 ? (float)(s / c) : __builtin_nanf("");
}

constexpr int AO_MAX = 256;
constexpr int AO_GROUP = 4;
constexpr int AO_RUN = 16;      // |1 + i ratio| <= sqrt 2: a run's product stays below 2^32
constexpr int AO_LAST = 0x80;   // in AoTab::len: the last group of its run

// Samples in table order without the skipped ones, cut into groups of at most
// AO_GROUP consecutive samples of one distance factor, and the groups into runs
// of one distance factor (a ring) of at most AO_RUN groups.
struct AoTab {
  int n, n_groups;
  float intensity;  // f32(intensity)
  int dmax_y, dmax_x;  // largest |offset| on each axis (interior test)
  short2 off[AO_MAX];
  float inv[AO_MAX];
  float scale[AO_MAX];           // per group: distance factor / (pi / 4)
  unsigned char len[AO_MAX];     // per group: samples, AO_LAST
};

// The angles of a run of samples.  A sample's angle is atan of its ratio clamped
// to [0, 1] (so within [0, pi/4]; 0 for a NaN sample), the argument of 1 + i
// ratio, and arguments add under multiplication.  A group's product has its
// argument within [0, pi]; the running product is kept in the upper half plane
// with the half turns counted, so a run of any length takes one
// atan: two FMAs and an eighth of a complex product more a sample in place of
// an atanf, a division and a mask.
struct AoRun {
  float x = 1.0f, y = 0.0f;   // y: its sign is not part of the value
  unsigned signs = 0;         // one bit per group of the run
  __device__ __forceinline__ void add(const float v[AO_GROUP], const float inv[AO_GROUP],
                                      float z) {
    float a[AO_GROUP];
#pragma unroll
    for (int k = 0; k < AO_GROUP; k++)
      a[k] = __builtin_amdgcn_fmed3f((v[k] - z) * inv[k], 0.0f, 1.0f);
    const float x0 = __builtin_fmaf(-a[0], a[1], 1.0f), y0 = a[0] + a[1];
    const float x1 = __builtin_fmaf(-a[2], a[3], 1.0f), y1 = a[2] + a[3];
    const float gx = __builtin_fmaf(x0, x1, -(y0 * y1)), gy = __builtin_fmaf(x0, y1, y0 * x1);
    const float ay = fabsf(y);
    const float nx = __builtin_fmaf(x, gx, -(ay * gy)), ny = __builtin_fmaf(x, gy, ay * gx);
    x = __uint_as_float(__float_as_uint(nx) ^ (__float_as_uint(ny) & 0x80000000u));
    y = ny;
    signs = __builtin_amdgcn_alignbit(signs, __float_as_uint(ny), 31);
  }
  // total + scale * the run's angle; the next run starts
  __device__ __forceinline__ float flush(float scale, float total) {
    const float t = __builtin_fmaf((float)__popc(signs), 3.14159274f, arg_upper(x, fabsf(y)));
    x = 1.0f;
    y = 0.0f;
    signs = 0;
    return __builtin_fmaf(t, scale, total);
  }
};

// AO of a pixel before the Gaussian, from its occlusion sum and valid samples
__device__ __forceinline__ float ao_value(const AoTab& T, float z, float total, float count) {
  const float mean = total / fmaxf(count, 1.0f);
  const float ao = 1.0f - mean * T.intensity;
  return isnan(z) ? 1.0f : fminf(fmaxf(ao, 0.0f), 1.0f);
}

// Pass 1: AO before the Gaussian on the expanded region, stored as
// where(isnan(z), 1, ao) -- the array the reference smooths.  Absent samples of
// a short group repeat the group's first one with a ratio of 0.
__global__ void __launch_bounds__(256)
k_ao_raw(WinDevR W, int er0, int ec0, int eh, int ew, AoTab T, float* __restrict__ dst,
         RayGrid G) {
  int bx, by;
  if (!ray_block(G, blockIdx.x, bx, by)) return;
  const int c = bx * 64 + threadIdx.x, r = by * 4 + threadIdx.y;
  if (c >= ew || r >= eh) return;
  const int i = er0 + r, j = ec0 + c;
  // block-uniform: do all samples of the block's pixels stay inside the window?
  const int bi0 = er0 + by * 4, bj0 = ec0 + bx * 64;
  const bool interior = bi0 - T.dmax_y >= 0 && bi0 + 3 + T.dmax_y < W.h &&
                        bj0 - T.dmax_x >= 0 && bj0 + 63 + T.dmax_x < W.w;
  const float* pc = W.p + (int64_t)i * W.ld + j;
  const float z = *pc, zv = isnan(z) ? 0.0f : z;
  float total = 0.0f;
  int count = 0, e0 = 0;
  AoRun A;
  for (int g = 0; g < T.n_groups; g++) {
    const int len = T.len[g] & (AO_LAST - 1);
    float v[AO_GROUP], inv[AO_GROUP];
#pragma unroll
    for (int k = 0; k < AO_GROUP; k++) {
      const int e = k < len ? e0 + k : e0;
      const short2 o = T.off[e];
      inv[k] = k < len ? T.inv[e] : 0.0f;
      v[k] = interior ? pc[(int64_t)o.y * W.ld + o.x]
                      : W.p[(int64_t)clampi(i + o.y, W.h) * W.ld + clampi(j + o.x, W.w)];
    }
#pragma unroll
    for (int k = 0; k < AO_GROUP; k++) count += k < len && !isnan(v[k]);
    A.add(v, inv, zv);
    if (T.len[g] & AO_LAST) total = A.flush(T.scale[g], total);
    e0 += len;
  }
  dst[(int64_t)r * ew + c] = ao_value(T, z, total, (float)count);
}

// The same from a tile staged in LDS: same groups, same operations, same bits.
// The valid samples are counted only where the running sum of the samples is
// NaN (one is, or two infinities met).
__global__ void __launch_bounds__(1024)
k_ao_raw_tile(WinDevR W, int er0, int ec0, int eh, int ew, AoTab T, RayTile R,
              float* __restrict__ dst) {
  extern __shared__ __attribute__((aligned(16))) float rt[];
  int bx, by;
  if (!ray_block(R.G, blockIdx.x, bx, by)) return;
  const int y0 = by * R.th, rows = min(R.th, eh - y0), x0 = bx * RT_W;
  stage_tile<true>(W, er0 + y0 - R.dy, rows + 2 * R.dy, ec0 + x0 - R.dx, R.pitch, rt);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int y = wave; y < rows; y += 16) {
    const char* at = (const char*)(rt + (y + R.dy) * R.pitch + R.dx + lane);
    float z[2], zv[2], total[2] = {0.0f, 0.0f}, chk[2] = {0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 2; m++) {
      z[m] = ((const float*)at)[64 * m];
      zv[m] = isnan(z[m]) ? 0.0f : z[m];
    }
    int e0 = 0;
    AoRun A[2];
#pragma unroll 2
    for (int g = 0; g < T.n_groups; g++) {
      const int len = T.len[g] & (AO_LAST - 1);
      float v[2][AO_GROUP], inv[AO_GROUP];
#pragma unroll
      for (int k = 0; k < AO_GROUP; k++) {
        const int e = k < len ? e0 + k : e0;
        const float* p = lds_sample(at, T.off[e]);
        v[0][k] = p[0];
        v[1][k] = p[64];
        inv[k] = k < len ? T.inv[e] : 0.0f;
      }
#pragma unroll
      for (int m = 0; m < 2; m++) {
        chk[m] += (v[m][0] + v[m][1]) + (v[m][2] + v[m][3]);
        A[m].add(v[m], inv, zv[m]);
      }
      if (T.len[g] & AO_LAST) {
        const float sc = T.scale[g];
        total[0] = A[0].flush(sc, total[0]);
        total[1] = A[1].flush(sc, total[1]);
      }
      e0 += len;
    }
    int count[2] = {T.n, T.n};
    if (__builtin_amdgcn_ballot_w64(__builtin_isunordered(chk[0], chk[1])) != 0) {
      count[0] = count[1] = 0;
      for (int e = 0; e < T.n; e++) {
        const float* p = lds_sample(at, T.off[e]);
        count[0] += !isnan(p[0]);
        count[1] += !isnan(p[64]);
      }
    }
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const int c = x0 + lane + 64 * m;
      if (c < ew)
        dst[(int64_t)(y0 + y) * ew + c] = ao_value(T, z[m], total[m], (float)count[m]);
    }
  }
}

// The values of pixels j .. j + 3 of row i (j + 3 possibly past the window's
// last column: absent pixels repeat the last one).
__device__ __forceinline__ void load4_clamped(const WinDevR& W, int i, int j, float z[4]) {
  const float* row = W.p + (int64_t)i * W.ld;
  if (j + 3 < W.w) {
    float4 q;
    __builtin_memcpy(&q, row + j, sizeof(q));
    z[0] = q.x; z[1] = q.y; z[2] = q.z; z[3] = q.w;
  } else {
#pragma unroll
    for (int m = 0; m < 4; m++) z[m] = row[min(j + m, W.w - 1)];
  }
}

// Pass 2: sigma=1 Gaussian ('nearest' at the window edge, scipy's two passes
// with float32 between them), gamma, NaN restore.  A wave walks SH rows down a
// strip of 256 columns, four per lane, with the nine rows of the axis-0 pass in
// registers as float64, so each row is read and converted once; the axis-1 pass
// takes its neighbours from the adjacent lanes, so lanes 1 .. 62 write.  Each
// pixel read its 81 neighbours from memory before: 147 us on average over the
// launches of a 5003 x 6007 spatial job, now 25.
constexpr int AO_SC = 248;   // output columns of a strip

struct AoSmooth {
  WinDevR W;
  int r0, c0, rh, rw;          // region in window coordinates
  int er0, ec0, eh, ew;        // extent of src, likewise
  const float* src;
  int SH, n_strips;
};

__device__ __forceinline__ float lane_left(float v) {    // of lane - 1
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_right(float v) {   // of lane + 1
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false));
}

// sum of g[|k|] x[k], k = -4 .. 4: the centre, then pairs from the outside in
__device__ __forceinline__ double gauss9(const double* x, const Gauss9& G) {
  double s = x[4] * G.g[0];
#pragma unroll
  for (int d = 4; d >= 1; d--) s = __builtin_fma(x[4 - d] + x[4 + d], G.g[d], s);
  return s;
}

__global__ void __launch_bounds__(256)
k_ao_smooth(AoSmooth A, Gauss9 G, OutDev out) {
  const int lane = threadIdx.x & 63;
  const int unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int strip = unit % A.n_strips, y0 = unit / A.n_strips * A.SH;
  if (y0 >= A.rh) return;
  const int rows = min(A.SH, A.rh - y0);
  const int c = strip * AO_SC + 4 * lane - 4;      // this lane's first region column
  const int j = A.c0 + c;                          // ... and window column
  const WinDevR& W = A.W;
  // where every column of the strip lies inside src: one 16-byte load per row
  const int js = A.c0 + strip * AO_SC - 4;
  const bool inner = js >= A.ec0 && js + 255 < A.ec0 + A.ew;
  auto load = [&](int i, float v[4]) {
    const float* p = A.src + (int64_t)(clampi(i, W.h) - A.er0) * A.ew - A.ec0;
    if (inner) {
      __builtin_memcpy(v, p + j, 16);
    } else {
      // columns past what a lane's outputs need are clamped into src as well
#pragma unroll
      for (int m = 0; m < 4; m++)
        v[m] = p[min(max(clampi(j + m, W.w), A.ec0), A.ec0 + A.ew - 1)];
    }
  };
  const PostK pp = load_post(out);
  const bool writes = lane >= 1 && lane <= 62 && c < A.rw;
  const int n = min(4, A.rw - c);
  // the rows come in batches of AO_SB: their loads are issued together
  constexpr int AO_SB = 4;
  double x[4][8 + AO_SB];   // per column: rows y - 4 .. y + 3 + AO_SB around the batch at y
#pragma unroll
  for (int k = 0; k < 8; k++) {
    float v[4];
    load(A.r0 + y0 - 4 + k, v);
#pragma unroll
    for (int m = 0; m < 4; m++) x[m][k] = (double)v[m];
  }
  for (int yb = 0; yb < rows; yb += AO_SB) {
    float f[AO_SB][4], zz[AO_SB][4];
#pragma unroll
    for (int k = 0; k < AO_SB; k++) load(A.r0 + y0 + min(yb + k, rows - 1) + 4, f[k]);
#pragma unroll
    for (int k = 0; k < AO_SB; k++)
      if (writes) load4_clamped(W, A.r0 + y0 + min(yb + k, rows - 1), j, zz[k]);
#pragma unroll
    for (int k = 0; k < AO_SB; k++)
#pragma unroll
      for (int m = 0; m < 4; m++) x[m][8 + k] = (double)f[k][m];
#pragma unroll
    for (int k = 0; k < AO_SB; k++) {
      const int y = yb + k;
      if (y >= rows) break;
      // axis 0, then the neighbours' columns
      double t[12];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const float v = (float)gauss9(x[m] + k, G);
        t[m] = (double)lane_left(v);
        t[4 + m] = (double)v;
        t[8 + m] = (double)lane_right(v);
      }
      float res[4];
#pragma unroll
      for (int m = 0; m < 4; m++) res[m] = (float)gauss9(t + m, G);
      if (writes) {
#pragma unroll
        for (int m = 0; m < 4; m++)
          res[m] = post_value(pp, isnan(zz[k][m]) ? zz[k][m] : gamma_pow(res[m]));
        if (n == 4)
          store_out4(out, y0 + y, c, res, 0, 4, true);
        else
          store_out4(out, y0 + y, c, res, 0, n, false);
      }
    }
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int k = 0; k < 8; k++) x[m][k] = x[m][k + AO_SB];
  }
}

static void expanded(const fsg_window* win, const fsg_region* reg, int* er0, int* ec0, int* eh,
                     int* ew) {
  *er0 = std::max(0, reg->r0 - 4);
  *ec0 = std::max(0, reg->c0 - 4);
  const int er1 = std::min(win->h, reg->r0 + reg->h + 4);
  const int ec1 = std::min(win->w, reg->c0 + reg->w + 4);
  *eh = er1 - *er0;
  *ew = ec1 - *ec0;
}

}  // namespace fsg

using namespace fsg;

extern "C" int fsg_openness(const fsg_window* win, const fsg_region* reg,
                            const fsg_openness_params* p, const fsg_output* out, void* stream) {
  int rc = validate_window(win, "fsg_openness");
  if (rc) return rc;
  rc = validate_region(win, reg, "fsg_openness");
  if (rc) return rc;
  if (!out) return fail(FSG_E_INVALID, "fsg_openness: output NULL");
  if ((rc = validate_output(out, reg, "fsg_openness"))) return rc;
  OpenTab T;
  if ((rc = openness_table(p, T, "fsg_openness"))) return rc;
  if (reg->h == 0 || reg->w == 0) return FSG_OK;
  WinDevR W{win->data, win->ld, win->h, win->w};
  const RayTile R = T.n_dist >= 1 && T.n_dist <= OPEN_UNROLL
                        ? ray_tile(reg->h, reg->w, T.dmax_y, T.dmax_x,
                                   std::max(T.dmax_y, T.dmax_x) <= 16 ? RT_MIN_PX_NEAR : RT_MIN_PX)
                        : RayTile{};
  if (R.th)
    for (int e = 0; e < T.n_dirs * T.n_dist; e++) T.off[e] = lds_offset(T.off[e], R);
  const RayGrid G = R.th ? R.G : ray_grid(reg->h, reg->w, 4, 64);
  if (ray_grid_blocks(G) > INT32_MAX)
    return fail(FSG_E_UNSUPPORTED, "fsg_openness: region too large for one launch");
  dim3 blk(64, 4), grd((unsigned)ray_grid_blocks(G));
  TimedScope ts("k_openness", as_stream(stream));
  const OutDev od = make_out(out);
  hipStream_t s = as_stream(stream);
  switch (T.n_dist) {
#define FSG_OPEN_ND(N)                                                                       \
  case N:                                                                                    \
    if (R.th)                                                                                \
      hipLaunchKernelGGL(k_openness_tile<N>, grd, dim3(1024), R.lds, s, W, reg->r0, reg->c0, \
                         reg->h, reg->w, T, R, od);                                          \
    else                                                                                     \
      hipLaunchKernelGGL(k_openness<N>, grd, blk, 0, s, W, reg->r0, reg->c0, reg->h, reg->w, \
                         T, od, G);                                                          \
    break;
    FSG_OPEN_ND(1) FSG_OPEN_ND(2) FSG_OPEN_ND(3) FSG_OPEN_ND(4) FSG_OPEN_ND(5)
    FSG_OPEN_ND(6) FSG_OPEN_ND(7) FSG_OPEN_ND(8) FSG_OPEN_ND(9) FSG_OPEN_ND(10)
#undef FSG_OPEN_ND
    default:
      hipLaunchKernelGGL(k_openness<0>, grd, blk, 0, s, W, reg->r0, reg->c0, reg->h, reg->w, T,
                         od, G);
  }
  FSG_CHECK_LAUNCH("k_openness");
  return FSG_OK;
}

extern "C" int fsg_openness_points(const fsg_window* win, const int32_t* points, int32_t n,
                                   const fsg_openness_params* p, float* out, void* stream) {
  int rc = validate_window(win, "fsg_openness_points");
  if (rc) return rc;
  if (n < 0 || (n > 0 && (!points || !out)))
    return fail(FSG_E_INVALID, "fsg_openness_points: bad point list");
  OpenTab T;
  if ((rc = openness_table(p, T, "fsg_openness_points"))) return rc;
  if (n == 0) return FSG_OK;
  WinDevR W{win->data, win->ld, win->h, win->w};
  TimedScope ts("k_openness_points", as_stream(stream));
  hipLaunchKernelGGL(k_openness_points, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream),
                     W, (const int2*)points, n, T, out);
  FSG_CHECK_LAUNCH("k_openness_points");
  return FSG_OK;
}

extern "C" size_t fsg_openness_judge_workspace_size(const fsg_window* win, int32_t tile_h,
                                                    int32_t tile_w) {
  if (!win || win->h <= 0 || win->w <= 0 || tile_h <= 0 || tile_w <= 0) return 0;
  const size_t n_tiles = (size_t)((win->h + tile_h - 1) / tile_h) * ((win->w + tile_w - 1) / tile_w);
  return sizeof(double) * 2 * JUDGE_SPLIT * n_tiles;
}

extern "C" int fsg_openness_judge(const fsg_window* win, const fsg_openness_params* p,
                                  const float* approx, int64_t lda, int32_t tile_h,
                                  int32_t tile_w, double sample_frac, uint64_t seed,
                                  int32_t seg_len, float* tile_mae, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  int rc = validate_window(win, "fsg_openness_judge");
  if (rc) return rc;
  if (win->h == 0 || win->w == 0 || !approx || lda < win->w || !tile_mae || tile_h <= 0 ||
      tile_w <= 0 || !(sample_frac > 0.0) || sample_frac > 1.0)
    return fail(FSG_E_INVALID, "fsg_openness_judge: bad arguments");
  const int n_ty = (win->h + tile_h - 1) / tile_h, n_tx = (win->w + tile_w - 1) / tile_w;
  const int min_tw = std::min(tile_w, win->w - (n_tx - 1) * tile_w);
  if (seg_len < 1 || seg_len > 64 || seg_len > min_tw)
    return fail(FSG_E_INVALID, "fsg_openness_judge: seg_len must be 1..64 and fit every tile");
  const int64_t n_tiles = (int64_t)n_ty * n_tx;
  if (n_tiles * JUDGE_SPLIT > 0x7fffffff)
    return fail(FSG_E_INVALID, "fsg_openness_judge: too many tiles");
  if (!workspace || workspace_bytes < fsg_openness_judge_workspace_size(win, tile_h, tile_w))
    return fail(FSG_E_WORKSPACE, "fsg_openness_judge: workspace too small");
  OpenTab T;
  if ((rc = openness_table(p, T, "fsg_openness_judge"))) return rc;
  WinDevR W{win->data, win->ld, win->h, win->w};
  JudgeGeo G{tile_h, tile_w, n_tx, seg_len, sample_frac, seed};
  hipStream_t s = as_stream(stream);
  TimedScope ts("k_openness_judge", s);
  hipLaunchKernelGGL(k_openness_judge, dim3((unsigned)(n_tiles * JUDGE_SPLIT)), dim3(256), 0, s,
                     W, T, approx, lda, G, (double*)workspace);
  FSG_CHECK_LAUNCH("k_openness_judge");
  hipLaunchKernelGGL(k_openness_judge_finish, dim3((unsigned)((n_tiles + 255) / 256)), dim3(256),
                     0, s, (const double*)workspace, (int)n_tiles, tile_mae);
  FSG_CHECK_LAUNCH("k_openness_judge_finish");
  return FSG_OK;
}

extern "C" size_t fsg_ambient_occlusion_workspace_size(const fsg_window* win,
                                                       const fsg_region* reg) {
  if (!win || !reg) return 0;
  int er0, ec0, eh, ew;
  expanded(win, reg, &er0, &ec0, &eh, &ew);
  if (eh <= 0 || ew <= 0) return 0;
  return sizeof(float) * (size_t)eh * (size_t)ew;
}

extern "C" int fsg_ambient_occlusion(const fsg_window* win, const fsg_region* reg,
                                     const fsg_ao_params* p, const fsg_output* out,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  int rc = validate_window(win, "fsg_ambient_occlusion");
  if (rc) return rc;
  rc = validate_region(win, reg, "fsg_ambient_occlusion");
  if (rc) return rc;
  if (!p || !out) return fail(FSG_E_INVALID, "fsg_ambient_occlusion: params/output NULL");
  if ((rc = validate_output(out, reg, "fsg_ambient_occlusion"))) return rc;
  if (p->n_samples < 0 || (p->n_samples > 0 && !p->samples))
    return fail(FSG_E_INVALID, "fsg_ambient_occlusion: bad sample table");
  if (p->n_samples > AO_MAX)
    return fail(FSG_E_UNSUPPORTED, "fsg_ambient_occlusion: more than 256 samples");
  if (reg->h == 0 || reg->w == 0) return FSG_OK;
  const size_t need = fsg_ambient_occlusion_workspace_size(win, reg);
  if (!workspace || workspace_bytes < need)
    return fail(FSG_E_WORKSPACE, "fsg_ambient_occlusion: workspace too small");
  AoTab T{};
  T.intensity = (float)p->intensity;
  float df = 0.0f;   // of the open group
  int run = 0;       // groups of the open run
  for (int e = 0; e < p->n_samples; e++) {
    const fsg_ao_sample& s = p->samples[e];
    if (s.skip || (s.dx == 0 && s.dy == 0)) continue;
    if (std::abs(s.dx) > 32767 || std::abs(s.dy) > 32767)
      return fail(FSG_E_UNSUPPORTED, "fsg_ambient_occlusion: offset beyond int16");
    T.off[T.n] = make_short2((short)s.dx, (short)s.dy);
    T.inv[T.n] = 1.0f / (float)s.phys;
    T.dmax_y = std::max(T.dmax_y, std::abs(s.dy));
    T.dmax_x = std::max(T.dmax_x, std::abs(s.dx));
    const bool new_run = T.n_groups == 0 || df != (float)s.dist_factor;
    if (new_run || T.len[T.n_groups - 1] == AO_GROUP) {
      df = (float)s.dist_factor;
      run = new_run || run == AO_RUN ? 1 : run + 1;
      if (run == 1 && T.n_groups) T.len[T.n_groups - 1] |= AO_LAST;
      T.scale[T.n_groups] = (float)((double)df * (4.0 / M_PI));
      T.len[T.n_groups++] = 0;
    }
    T.len[T.n_groups - 1]++;
    T.n++;
  }
  if (T.n_groups) T.len[T.n_groups - 1] |= AO_LAST;
  int er0, ec0, eh, ew;
  expanded(win, reg, &er0, &ec0, &eh, &ew);
  WinDevR W{win->data, win->ld, win->h, win->w};
  hipStream_t s = as_stream(stream);
  float* raw = (float*)workspace;
  {
    const RayTile R = ray_tile(eh, ew, T.dmax_y, T.dmax_x);
    if (R.th)
      for (int e = 0; e < T.n; e++) T.off[e] = lds_offset(T.off[e], R);
    const RayGrid RG = R.th ? R.G : ray_grid(eh, ew, 4, 64);
    if (ray_grid_blocks(RG) > INT32_MAX)
      return fail(FSG_E_UNSUPPORTED, "fsg_ambient_occlusion: region too large for one launch");
    const dim3 grd((unsigned)ray_grid_blocks(RG));
    TimedScope ts("k_ao_raw", s);
    if (R.th)
      hipLaunchKernelGGL(k_ao_raw_tile, grd, dim3(1024), R.lds, s, W, er0, ec0, eh, ew, T, R,
                         raw);
    else
      hipLaunchKernelGGL(k_ao_raw, grd, dim3(64, 4), 0, s, W, er0, ec0, eh, ew, T, raw, RG);
    FSG_CHECK_LAUNCH("k_ao_raw");
  }
  {
    AoSmooth A{W, reg->r0, reg->c0, reg->h, reg->w, er0, ec0, eh, ew, raw, 0, 0};
    A.n_strips = (reg->w + AO_SC - 1) / AO_SC;
    // rows per wave: at least 8192 waves, 8 to 64 rows (a wave's first 8 rows
    // are start-up loads)
    A.SH = (int)std::min<int64_t>(
        64, std::max<int64_t>(8, (int64_t)reg->h * A.n_strips / 8192 / 4 * 4));
    const int64_t units = (int64_t)A.n_strips * ((reg->h + A.SH - 1) / A.SH);
    if ((units + 3) / 4 > INT32_MAX)
      return fail(FSG_E_UNSUPPORTED, "fsg_ambient_occlusion: region too large for one launch");
    hipLaunchKernelGGL(k_ao_smooth, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, A,
                       make_gauss9(), make_out(out));
    FSG_CHECK_LAUNCH("k_ao_smooth");
  }
  return FSG_OK;
}
