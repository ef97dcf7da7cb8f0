// Planning of the middle-batch GEMM (awq_mid_kernel.h) and its instantiations for up to 64 rows,
// whose weights enter the MFMA unrounded; awq_mid_rounded.hip holds the ones above.
#include <algorithm>

#include "awq_mid_kernel.h"

namespace awq_host {
using namespace awq;

// One block per CU; a block's time on MI355X is 2 us + 0.35 us per 16 rows outside its K loop and 0.21 us +
// 0.08 us per 16 rows for each k-step of a share (128 k of the block), which reproduces N = 24576, K = 4096
// at one round of blocks (M = 32 / 48 / 64 / 80 / 96 / 128: 18.2 / 20.2 / 22.3 / 24.5 / 28.7 / 33.1 us) to
// 5%: fp16 in groups of 128.  The measured time over this estimate, above 64 rows (means over K = 768 ..
// 14336): groups of 128 0.93 .. 1.07 fp16, 1.06 .. 1.18 bf16; of 64 0.96 .. 1.10, 1.11 .. 1.23; of 32 1.06
// .. 1.17, 1.16 .. 1.27.  The plan itself hardly depends on that factor, the choice of kernel does
// (mid_least_rows, range_serves).  K ranges add, up to 64 rows, the hand-off (1.5 us) and one block's
// reading of its tile's partials (8 KB per range and 16 rows at about 100 bytes a ns), above them the
// reduction launch (3 us) and the partials' round trip (about 6 TB/s).  Up to 64 rows there is one row tile;
// above, row tiles of 64 .. 128 rows: the plan with the least estimated time.
MidPlan plan_mid(int64_t M, int64_t N, int64_t K, int64_t G) {
  const int64_t tiles = cdiv(N, 128), cus = num_cus();
  const int64_t unit = mid_unit(G >= 128 ? 128 : (int)G), units = cdiv(K, unit);
  MidPlan best{};
  const int most = M <= 64 ? (int)std::max<int64_t>(2, cdiv(M, 16)) : 8, least = M <= 64 ? most : 4;
  for (int rows = most; rows >= least; --rows) {
    if (rows == 8 && G == 32) continue;  // its activation stages leave no LDS for a constant set per k-step
    MidPlan m{};
    m.tiles = (int)tiles;
    m.row_tiles = (int)cdiv(M, 16 * rows);
    m.mt = std::max(std::min(least, 4), (int)cdiv(cdiv(M, m.row_tiles), 16));
    for (int64_t S = 1; S <= 16 && (S == 1 || (units >= 4 * S && tiles * m.row_tiles * S <= cus)); ++S) {
      m.per = (int)cdiv(units, S);
      m.splits = (int)cdiv(units, m.per);
      const size_t parts = m.splits > 1 ? (size_t)m.splits * (size_t)cdiv(M, 4) * (size_t)tiles * 2048 : 0;
      if (M <= 64 && parts > kMidPartialMax) break;
      const double rounds = (double)cdiv(tiles * m.row_tiles * m.splits, cus);
      const double ksteps = (double)cdiv(m.per, kMidShares) * (double)(unit / 32);
      m.us = 2.0 + rounds * (2.0 + 0.35 * m.mt + ksteps * (0.21 + 0.08 * m.mt)) + (m.splits == 1 ? 0.0 : M <= 64 ? 1.5 + 0.08 * m.mt * m.splits : 3.0 + (double)parts / 3e6);
      m.ws_bytes = parts ? kCounterBytes + parts : 0;
      if (best.mt == 0 || m.us < best.us) best = m;
    }
  }
  return best;
}

template <typename T, bool FAST>
static bool launch_unr(const GemmArgs& a, int mt, const MidWork& wk, hipStream_t st) {
  if (mt <= 2) return launch_mid_g<2, true, T, FAST>(a, wk, st);
  if (mt == 3) return launch_mid_g<3, true, T, FAST>(a, wk, st);
  return launch_mid_g<4, true, T, FAST>(a, wk, st);
}

bool launch_mid(const GemmArgs& a, const MidPlan& m, int act, int sdt, hipStream_t st) {
  const MidWork wk{m.tiles, m.splits, m.row_tiles, m.per, __builtin_ctz((unsigned)a.G), sdt == AWQ_DTYPE_BF16 ? 1 : 0};
  bool done;
  if (a.M > 64) done = launch_mid_rounded(a, m.mt, wk, act, sdt, st);
  else if (act == AWQ_DTYPE_F16 && sdt == AWQ_DTYPE_F16) done = launch_unr<f16, true>(a, m.mt, wk, st);
  else if (act == AWQ_DTYPE_F16) done = launch_unr<f16, false>(a, m.mt, wk, st);
  else done = launch_unr<bf16, false>(a, m.mt, wk, st);
  if (done && a.M > 64 && m.splits > 1) {
    const dim3 grid((unsigned)cdiv(cdiv(a.M, 4) * m.tiles, 4));
    if (act == AWQ_DTYPE_F16) hipLaunchKernelGGL((mid_reduce_kernel<f16>), grid, dim3(256), 0, st, a, wk);
    else hipLaunchKernelGGL((mid_reduce_kernel<bf16>), grid, dim3(256), 0, st, a, wk);
  }
  return done;
}

}  // namespace awq_host
