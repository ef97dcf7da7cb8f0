// The middle-batch GEMM (awq_mid_kernel.h) above 64 rows: weights rounded once, as in the prefill kernels.
#include "awq_mid_kernel.h"

namespace awq_host {
using namespace awq;

template <typename T, bool FAST>
static void launch_r(const GemmArgs& a, int mt, const MidWork& wk, hipStream_t st) {
  if (mt <= 4) launch_mid_g<4, false, T, FAST>(a, wk, st);
  else if (mt == 5) launch_mid_g<5, false, T, FAST>(a, wk, st);
  else if (mt == 6) launch_mid_g<6, false, T, FAST>(a, wk, st);
  else if (mt == 7) launch_mid_g<7, false, T, FAST>(a, wk, st);
  else launch_mid_g<8, false, T, FAST>(a, wk, st);
}

void launch_mid_rounded(const GemmArgs& a, int mt, const MidWork& wk, int act, int sdt, hipStream_t st) {
  if (act == AWQ_DTYPE_F16 && sdt == AWQ_DTYPE_F16) launch_r<f16, true>(a, mt, wk, st);
  else if (act == AWQ_DTYPE_F16) launch_r<f16, false>(a, mt, wk, st);
  else launch_r<bf16, false>(a, mt, wk, st);
}

}  // namespace awq_host
