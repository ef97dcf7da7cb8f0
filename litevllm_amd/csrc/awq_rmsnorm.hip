// RMSNorm prologue of the fused RMSNorm + int4 GEMM (rmsnorm_awq_fused_linear,
// vllm/kernels/triton/rmsnorm_awq_fused.py:43-189).
//
// The reference recomputes each row's sum of squares inside every output tile (each of its
// N / 64 programs reads the row twice).  Here one block per row reduces the row once and
// writes the normalised fp16 row; the GEMM kernels then read it like any activation.
//
// Arithmetic of the reference (rmsnorm_awq_fused.py:108-131), step for step:
//   var  = sum over k of fp32(x)^2       (fp32 in the reference, in 32-element chunks; here the
//                                         exact squares are added in fp64 and rounded once to
//                                         fp32, which makes the order of the adds invisible)
//   rrms = rsqrt(var / K + eps)          (var / K + eps in fp32; the rsqrt correctly rounded)
//   xn   = fp16_rne((fp32(x) * rrms) * fp32(norm_w))     (two fp32 products, one rounding)
#include <algorithm>

#include "awq_common.h"
#include "awq_launch.h"

namespace awq {

constexpr int kNormThreads = 256;

// One block per row.  COLS > 0: the row and the norm weights (K <= COLS * 2048) come into registers
// with one wait, which is what bounds a few rows (graph replays, 8 rows of 4096: 2.14 us against 2.53, of 12288 2.9 against 4.2 with a second
// reading of both after the sum); otherwise the second pass reads them again.
template <typename T, typename NT, int COLS>
__global__ void __launch_bounds__(kNormThreads) rmsnorm_rows_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                                    const uint16_t* __restrict__ nw, float eps,
                                                                    uint16_t* __restrict__ xn, int64_t ldo, int K) {
  __shared__ double part[kNormThreads / 64];
  const uint16_t* row = x + (int64_t)blockIdx.x * ldx;
  uint16_t* orow = xn + (int64_t)blockIdx.x * ldo;
  const int t = threadIdx.x;
  u32x4 xv[COLS > 0 ? COLS : 1], gv[COLS > 0 ? COLS : 1];
  if constexpr (COLS > 0) {
#pragma unroll
    for (int u = 0; u < COLS; ++u) {
      const int k = (t + u * kNormThreads) * 8;
      xv[u] = k < K ? *(const u32x4*)(row + k) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < COLS; ++u) {
      const int k = (t + u * kNormThreads) * 8;
      gv[u] = k < K ? *(const u32x4*)(nw + k) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  // sum of squares, 8 elements (16 bytes) per lane and step; the squares are exact in fp64 and the
  // fp64 sum is within about K * 2^-53 of the exact one, so rounding it once to fp32 gives the
  // correctly rounded var (whatever the order of the adds) unless the exact sum lies that close to
  // an fp32 rounding boundary
  double ss = 0.0;
  auto squares = [&](const u32x4& v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double lo = from_bits<T>((uint16_t)(v[j] & 0xFFFF)), hi = from_bits<T>((uint16_t)(v[j] >> 16));
      ss += lo * lo;
      ss += hi * hi;
    }
  };
  if constexpr (COLS > 0) {
#pragma unroll
    for (int u = 0; u < COLS; ++u) squares(xv[u]);
  } else {
    for (int k = t * 8; k < K; k += kNormThreads * 8) squares(*(const u32x4*)(row + k));
  }
  ss = wave_sum_f64(ss);
  if ((t & 63) == 0) part[t >> 6] = ss;
  __syncthreads();
  double var = 0.0;
#pragma unroll
  for (int w = 0; w < kNormThreads / 64; ++w) var += part[w];  // same order in every lane
  const float rrms = rms_scale((float)var, K, eps);
  // the row scaled and rounded once to fp16
  auto scaled = [&](const u32x4& v, const u32x4& g) {
    u32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = fp32_rounded((from_bits<T>((uint16_t)(v[j] & 0xFFFF)) * rrms) * from_bits<NT>((uint16_t)(g[j] & 0xFFFF)));
      const float hi = fp32_rounded((from_bits<T>((uint16_t)(v[j] >> 16)) * rrms) * from_bits<NT>((uint16_t)(g[j] >> 16)));
      r[j] = (uint32_t)f2h_bits(lo) | ((uint32_t)f2h_bits(hi) << 16);
    }
    return r;
  };
  if constexpr (COLS > 0) {
#pragma unroll
    for (int u = 0; u < COLS; ++u) {
      const int k = (t + u * kNormThreads) * 8;
      if (k < K) *(u32x4*)(orow + k) = scaled(xv[u], gv[u]);
    }
  } else {
    for (int k = t * 8; k < K; k += kNormThreads * 8) *(u32x4*)(orow + k) = scaled(*(const u32x4*)(row + k), *(const u32x4*)(nw + k));
  }
}

}  // namespace awq

namespace awq_host {
using namespace awq;

template <typename T, typename NT>
static void rows_t(const void* x, int64_t ldx, const void* nw, float eps, void* xn, int64_t ldo, int64_t M, int64_t K,
                   hipStream_t st) {
  const dim3 grid((unsigned)M), block(kNormThreads);
  const auto* xs = (const uint16_t*)x;
  const auto* ns = (const uint16_t*)nw;
  auto* o = (uint16_t*)xn;
  const int cols = (int)std::min<int64_t>(cdiv(K, kNormThreads * 8), 9);
  if (cols <= 2) rmsnorm_rows_kernel<T, NT, 2><<<grid, block, 0, st>>>(xs, ldx, ns, eps, o, ldo, (int)K);
  else if (cols <= 4) rmsnorm_rows_kernel<T, NT, 4><<<grid, block, 0, st>>>(xs, ldx, ns, eps, o, ldo, (int)K);
  else if (cols <= 8) rmsnorm_rows_kernel<T, NT, 8><<<grid, block, 0, st>>>(xs, ldx, ns, eps, o, ldo, (int)K);
  else rmsnorm_rows_kernel<T, NT, 0><<<grid, block, 0, st>>>(xs, ldx, ns, eps, o, ldo, (int)K);
}

int launch_rmsnorm_rows(const void* x, int64_t ldx, const void* nw, float eps, void* xn, int64_t ldo, int64_t M,
                        int64_t K, int act, int ndt, hipStream_t st) {
  if (M <= 0) return AWQ_OK;
  if (M > 0x7FFFFFFFLL) return AWQ_ERR_UNSUPPORTED;
  const bool xb = act == AWQ_DTYPE_BF16, nb = ndt == AWQ_DTYPE_BF16;
  if (!xb && !nb) rows_t<f16, f16>(x, ldx, nw, eps, xn, ldo, M, K, st);
  else if (!xb && nb) rows_t<f16, bf16>(x, ldx, nw, eps, xn, ldo, M, K, st);
  else if (xb && !nb) rows_t<bf16, f16>(x, ldx, nw, eps, xn, ldo, M, K, st);
  else rows_t<bf16, bf16>(x, ldx, nw, eps, xn, ldo, M, K, st);
  return hipGetLastError() == hipSuccess ? AWQ_OK : AWQ_ERR_LAUNCH;
}

}  // namespace awq_host
