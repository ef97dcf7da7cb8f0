// The middle-batch GEMM (awq_mid_kernel.h) above 64 rows: weights rounded once, as in the prefill kernels.
#include "awq_mid_kernel.h"

namespace awq_host {
using namespace awq;

template <typename T, bool FAST>
static bool launch_r(const GemmArgs& a, int mt, const MidWork& wk, hipStream_t st) {
  if (mt <= 4) return launch_mid_g<4, false, T, FAST>(a, wk, st);
  if (mt == 5) return launch_mid_g<5, false, T, FAST>(a, wk, st);
  if (mt == 6) return launch_mid_g<6, false, T, FAST>(a, wk, st);
  if (mt == 7) return launch_mid_g<7, false, T, FAST>(a, wk, st);
  return launch_mid_g<8, false, T, FAST>(a, wk, st);
}

bool launch_mid_rounded(const GemmArgs& a, int mt, const MidWork& wk, int act, int sdt, hipStream_t st) {
  if (act == AWQ_DTYPE_F16 && sdt == AWQ_DTYPE_F16) return launch_r<f16, true>(a, mt, wk, st);
  if (act == AWQ_DTYPE_F16) return launch_r<f16, false>(a, mt, wk, st);
  return launch_r<bf16, false>(a, mt, wk, st);
}

}  // namespace awq_host
