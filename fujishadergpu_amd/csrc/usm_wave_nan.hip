// TopoUSM main pass, the blocks of a window that met a NaN (see usm_wave.hpp).
#include <algorithm>

#include "usm_wave.hpp"

namespace fsg {

// Blocks in x take k_usm_wave's tile of that number, blocks in y `sub` of its
// rows each; unmarked tiles are done.
template <int NR, int NS, int KR>
__global__ void __launch_bounds__(64) k_usm_wave_nan(WaveArgs A, int sub) {
  __shared__ double P[4 * WAVE_PB];
  __shared__ double Hc[(NS > 0 ? NS : 1) * 2 * WAVE_NC];
  const int b = blockIdx.x;
  const int tile = (b & 7) * A.per_xcd + (b >> 3);
  if (tile >= A.n_blocks || !A.flags[tile]) return;
  const int t0 = (tile / A.n_strips) * A.SH;
  const int y0 = t0 + blockIdx.y * sub;
  const int rows = min(min(sub, t0 + A.SH - y0), A.rh - y0);
  if (rows <= 0) return;
  wave_rect<NR, NS, KR, WAVE_NAN>(A, (tile % A.n_strips) * A.SW, y0, rows, P, Hc);
}

// Rows per block.  Few tiles are marked and a wave walks its rows one after another
// (about 3.5 us each with three radii, after 2R + 1 start-up rows that only add), so
// whole tiles left the launch waiting for single waves (30 rows: 98 us a window, as
// long as the plain launch over all tiles).  Four rows as long as the whole window's
// blocks would come to at most three rounds, for windows where every tile is marked:
// radii 2, 8, 32 at 1 % of discs / 30 % of single cells missing, a call in us with 8
// and with 4 rows: 512^2 89 / 58 and 78 / 48, 1700^2 104 / 78 and 96 / 94, 2400^2
// (past the line) 120 / 124 and 109 / 144.  Else an eighth of a tile, 8 rows at
// least; at most 64, the workgroup kernels' block, since an infinity makes NaN of a
// block's rows from where its sums meet it.
constexpr int WAVE_NAN_ROWS = 8, WAVE_NAN_FEW = 4, WAVE_NAN_MOST = 64;

template <int NR, int NS, int KR>
static int launch(const WaveArgs& A, hipStream_t s) {
  static const int cap = wave_resident(k_usm_wave_nan<NR, NS, KR>);
  const bool few = (int64_t)A.n_strips * ((A.rh + WAVE_NAN_FEW - 1) / WAVE_NAN_FEW) <= 3 * cap;
  const int sub = few ? WAVE_NAN_FEW
                      : std::min(WAVE_NAN_MOST, std::max(WAVE_NAN_ROWS, (A.SH + 7) / 8));
  TimedScope ts("k_usm_main", s);
  hipLaunchKernelGGL((k_usm_wave_nan<NR, NS, KR>), dim3(A.per_xcd * 8, (A.SH + sub - 1) / sub),
                     dim3(64), 0, s, A, sub);
  FSG_CHECK_LAUNCH("k_usm_wave_nan");
  return FSG_OK;
}

int launch_wave_nan(const WaveArgs& A, int nr, int ns, hipStream_t s) {
  if (nr == 3 && A.rad[0] == 2 && A.rad[1] == 8 && A.rad[2] == 32) {
    if (ns == 0) return launch<3, 0, 1>(A, s);
    if (ns == 1) return launch<3, 1, 1>(A, s);
    if (ns == 2) return launch<3, 2, 1>(A, s);
    if (ns == 3) return launch<3, 3, 1>(A, s);
  }
#define FSG_WAVE_CASE(NRV, NSV) \
  if (nr == NRV && ns == NSV) return launch<NRV, NSV, 0>(A, s);
  FSG_WAVE_CASE(1, 0) FSG_WAVE_CASE(1, 1) FSG_WAVE_CASE(1, 2) FSG_WAVE_CASE(1, 3)
  FSG_WAVE_CASE(2, 0) FSG_WAVE_CASE(2, 1) FSG_WAVE_CASE(2, 2) FSG_WAVE_CASE(2, 3)
  FSG_WAVE_CASE(3, 0) FSG_WAVE_CASE(3, 1) FSG_WAVE_CASE(3, 2) FSG_WAVE_CASE(3, 3)
#undef FSG_WAVE_CASE
  return fail(FSG_E_UNSUPPORTED, "k_usm_wave_nan: unsupported term counts");
}

}  // namespace fsg
