// GEMM of middle-sized batches (17 rows to a few hundred) on the stream layout of the weights,
// gfx950: the role of _awq_native_tiled_gemm_autotuned at BLOCK_M = 32 .. 128
// (vllm/kernels/triton/awq_fused_gemm.py:2296-2392).
//
//  * Block tile 16 MT rows x 128 columns (one stream tile), 8 waves: 2 column halves x 4 shares
//    of the block's K range.  A wave takes one 16-byte piece of the stream layout per lane and
//    32-row k-step (half e of a word: nibble positions 4 e .. 4 e + 3 over 8 k-rows, already
//    paired), forms four MFMA operands of it and multiplies each into MT row tiles
//    (v_mfma_f32_16x16x32), so a weight is dequantized once per block.
//  * Everything a k-step needs comes into LDS by DMA ahead of time: the share's activation rows
//    in stages of two k-steps (a ring of NA, shared by the two halves), the wave's own weight
//    pieces (a ring of R k-steps) and group constants.  The wave waits for them by count, so no
//    register is ever the target of a load in flight; one barrier per stage.
//  * The operands of k-step n + 1 are formed between the MFMAs of k-step n: on this part a wave's
//    own VALU work between its MFMAs is nearly free up to three instructions each, and adds in
//    full anywhere else.
//  * UNR (M <= 64): the weights enter the MFMA as exact integers and each group's sum is scaled once in
//    fp32, the decode kernels' unrounded formulation: q - z for fp16, and for bf16 in groups of 32; 128 + q
//    for bf16 in larger groups (exact q - z takes three conversions a pair), with (128 + z) times the
//    activation sums, an MFMA against ones per row tile, taken off per group.  The bias costs precision
//    where one activation is far above the others (1e4 among N(0, 1), group 32: 2.2 bf16 ulps against 0.5)
//    and turns an infinite one into NaN in every column, so it is taken only where the decode kernels'
//    two-tile form takes it.  Otherwise they enter as (q - z) * s rounded once, the prefill kernels'.
//  * The shares' sums meet in LDS in share order; with one K range the block writes its outputs,
//    with several it writes fp32 partials, which the tile's last block (UNR) or a second launch adds
//    in range order.
//  * The blocks of a column tile's row tiles are dispatched together on one XCD and read the
//    tile's weights through its L2.
//  * What bounds it: short calls, fixed costs (M = 64, N = K = 4096, 14.6 us: 1.3 us to the first operands and
//    3.4 us of K loop; the rest is the shares' sum, the partials and the last block's reading of them, the launch
//    and its gap); long loops, in about
//    equal parts and only partly overlapped, the MFMAs (M = 64: 0.27 us of a k-step's 0.5 us), the
//    operand VALU and the DMA issue (8 rows x 128 bytes a request move 70 bytes a ns and CU, half of what
//    linear requests do).  Tried: 32x32x16 MFMAs (5 VALU instructions per MFMA free instead of one, but
//    32-row granularity): 2 - 10% slower; weights in registers two stages ahead with the stage's requests
//    issued at once: 3 - 15% slower; shares interleaved over K in 256-byte steps, against L2 channel
//    conflicts: unchanged.
//  * fp16, K = 4096, before (decode chunks of 32 rows, or 256-row prefill tiles cut in K ranges) and now:
//    M = 57 N = 4096 24.3 -> 14.2 us, N = 24576 36.7 -> 21.6; M = 200 N = 6144 30.1 -> 20.7; M = 640
//    N = 24576 204 -> 130; M = 256 K = 12288 N = 4096 50.9 -> 33.2.
#pragma once

#include "awq_common.h"
#include "awq_launch.h"

namespace awq {

// Column tiles x K ranges x row tiles of a launch: range s of the K units (mid_unit rows each)
// takes units s * per .. (s + 1) * per - 1.
struct MidWork {
  int tiles, splits, row_tiles, per, log2g, scale_bf16;
};

constexpr int kMidShares = 4;
// rows of a K unit: whole stages (64) and whole groups up to 128
__host__ __device__ constexpr int mid_unit(int gk) { return gk > 64 ? gk : 64; }

// LDS of an instantiation: NA activation stages, R k-steps of weight pieces per wave (R <= 2 NA, so
// the counted waits hold from the first k-step on), and the constant sets that R k-steps span.
struct MidLds {
  int na, r, ncs, bytes;
};
__host__ __device__ constexpr MidLds mid_lds(int mt, int gk) {
  const int stage = kMidShares * mt * 16 * 128;
  MidLds best{0, 0, 0, 0};
  for (int na = 2; na <= 4; ++na)
    for (int r = 3; r <= 2 * na; ++r) {
      const int spg = gk / 32, ncs = (r + spg - 1) / spg;
      const int bytes = na * stage + 8 * (r * 1024 + ncs * 512);
      if (bytes <= 163840 && r >= best.r) best = MidLds{na, r, ncs, bytes};
    }
  return best;
}

template <bool NT>
__device__ __forceinline__ void mid_dma_w(const u32x4& rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
  else
    lds_dma16(rsrc, lds, voff, soff);
}

// GK: rows per set of group constants (32, 64, or 128 for every larger group).
// FAST: fp16 scales (with fp16 activations, rounded form: packed fp16 multiply).
template <int MT, bool UNR, typename T, bool FAST, int GK>
__global__ void __launch_bounds__(512, 2) mid_kernel(const GemmArgs p, const MidWork wk) {
  constexpr int ROWS = 16 * MT;
  constexpr int ABYTES = ROWS * 128;                // one share's activation stage (64 k)
  constexpr int STAGE = kMidShares * ABYTES;
  constexpr MidLds L = mid_lds(MT, GK);
  constexpr int NA = L.na, R = L.r, NCS = L.ncs;
  static_assert(R >= 3 && R <= 2 * NA, "");
  constexpr int SPG = GK / 32;                      // k-steps per constant set
  constexpr int ND = MT;                            // activation DMA instructions per wave and stage
  // the final sum: 64 rows (16 quads) per pass, [share][quad][128 columns] x 4 rows, then the
  // 16-bit outputs [64][128]
  constexpr int RPASS = MT > 4 ? 64 : ROWS;
  constexpr int RED = kMidShares * RPASS * 512;
  constexpr int LDS_N = L.bytes > RED + RPASS * 256 ? L.bytes : RED + RPASS * 256;
  static_assert(LDS_N <= 163840, "");
  __shared__ __align__(16) unsigned char lds[LDS_N];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e = wave & 1, part = wave >> 1;
  const int q = lane >> 4, r = lane & 15;

  // block -> (range, column tile, row tile); a tile's row tiles on one XCD, next to each other
  const int nbase = wk.tiles * wk.splits;
  int base, rt;
  if (wk.row_tiles == 1) {
    base = (int)blockIdx.x;
    rt = 0;
  } else if ((nbase & 7) == 0) {
    const int b = (int)blockIdx.x, i = b >> 3;
    base = (i / wk.row_tiles) * 8 + (b & 7);
    rt = i % wk.row_tiles;
  } else {
    base = (int)blockIdx.x / wk.row_tiles;
    rt = (int)blockIdx.x % wk.row_tiles;
  }
  const int split = base / wk.tiles, t = base - split * wk.tiles;
  const int m0 = rt * ROWS;

  constexpr int UK = mid_unit(GK) / 32;             // k-steps per unit
  const int KS = p.K >> 5;
  const int nunits = (KS + UK - 1) / UK;
  const int u0 = min(split * wk.per, nunits), u1 = min(u0 + wk.per, nunits);
  const int len = u1 - u0;
  const int us = u0 + len * part / kMidShares, ue = u0 + len * (part + 1) / kMidShares;
  const int ks0 = us * UK, nk = min(ue * UK, KS) - ks0;      // this share's k-steps
  const int nkmax = (len + kMidShares - 1) / kMidShares * UK;  // ... of the longest share, whole units

  // ---- requests.  k-step n of the share: weight piece into ring slot n % R, constants (where a set
  // starts) into set slot (n / SPG) % NCS; past the share's end through empty descriptors (zeros),
  // so the number of requests never varies ----
  const int NW = p.N >> 3;
  const int ngroups = p.K / p.G;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  const uint32_t lds_w = lds0 + (uint32_t)(NA * STAGE + wave * R * 1024);
  const uint32_t lds_c = lds0 + (uint32_t)(NA * STAGE + 8 * R * 1024 + wave * NCS * 512);
  const uint64_t wbase = (uint64_t)(uintptr_t)p.qw, sbase = (uint64_t)(uintptr_t)p.sc;
  const uint64_t zbase = (uint64_t)(uintptr_t)(p.qz ? (const void*)p.qz : (const void*)p.sc);
  const uint64_t abase = (uint64_t)(uintptr_t)p.a;
  const uint32_t w_bytes = (uint32_t)wk.tiles * (uint32_t)KS * 2048u;
  const uint32_t s_bytes = (uint32_t)((uint64_t)ngroups * p.N * 2u);
  const uint32_t z_bytes = p.qz ? (uint32_t)((uint64_t)ngroups * NW * 4u) : 0u;
  const uint32_t z_none = p.qz ? 0u : 0x88888888u;
  const uint32_t a_bytes = (uint32_t)((uint64_t)p.M * (uint64_t)p.lda * 2u);
  const uint32_t w_voff = (uint32_t)t * (uint32_t)KS * 2048u + (uint32_t)e * 1024u + (uint32_t)lane * 16u;
  const uint32_t s_voff = min((uint32_t)t * 256u + (uint32_t)lane * 4u, (uint32_t)p.N * 2u - 4u);
  const uint32_t z_voff = 4u * (uint32_t)min(t * 16 + r, NW - 1);
  const int log2spg = wk.log2g - 5;
  auto req_w = [&](int n, int wslot) {
    const u32x4 wrs = {(uint32_t)wbase, (uint32_t)(wbase >> 32) & 0xFFFFu, n < nk ? w_bytes : 0u, 0x00020000u};
    mid_dma_w<UNR>(wrs, lds_w + (uint32_t)wslot * 1024u, w_voff, (uint32_t)(ks0 + n) * 2048u);
  };
  auto req_c = [&](int n, int cslot, bool zeros) {
    const uint32_t g = (uint32_t)min((ks0 + n) >> log2spg, ngroups - 1);
    const uint64_t base_ = zeros ? zbase : sbase;
    const u32x4 crs = {(uint32_t)base_, (uint32_t)(base_ >> 32) & 0xFFFFu, n < nk ? (zeros ? z_bytes : s_bytes) : 0u, 0x00020000u};
    lds_dma4(crs, lds_c + (uint32_t)cslot * 512u + (zeros ? 256u : 0u), zeros ? z_voff : s_voff,
             g * (zeros ? (uint32_t)NW * 4u : (uint32_t)p.N * 2u));
  };
  // activations: a DMA instruction fills 8 rows of a stage, lane l row l / 8, slot l % 8, which holds
  // chunk slot ^ swz(row) (an operand read, 16 rows at 4 chunks, then covers all 64 banks); wave e of
  // a share issues its half of them.  Rows past M repeat the last one and are never stored.
  auto swz = [](int row) { return (row ^ (row >> 3)) & 7; };
  uint32_t a_voff[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int row = 8 * (e * ND + i) + (lane >> 3);
    const int kc = (lane & 7) ^ swz(row & 15);
    a_voff[i] = ((uint32_t)min(m0 + row, p.M - 1) * (uint32_t)p.lda + (uint32_t)(kc * 8)) * 2u;
  }
  // activation instruction i of stage s into ring slot `aslot`
  auto req_a = [&](int s, int aslot, int i) {
    const int k = (ks0 + 2 * s) * 32;
    const u32x4 ars = {(uint32_t)abase, (uint32_t)(abase >> 32) & 0xFFFFu, 2 * s < nk ? a_bytes : 0u, 0x00020000u};
    uint32_t vo = a_voff[i];
    if (GK == 32 && k + 64 > p.K) {  // K ends inside the stage: chunks past it read zero
      const int kc = (lane & 7) ^ swz((8 * (e * ND + i) + (lane >> 3)) & 15);
      vo = k + kc * 8 >= p.K ? 0x80000000u : vo;
    }
    lds_dma16(ars, lds0 + (uint32_t)(aslot * STAGE + part * ABYTES + (e * ND + i) * 1024), vo, (uint32_t)(k * 2));
  };

  constexpr bool BIAS = UNR && std::is_same<T, bf16>::value && GK != 32;
  f32x4 acc[MT][4];
  f32x4 ax[BIAS ? MT : 1];  // the group's activation sums
  f32x4 tot[UNR ? MT : 1][4];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int P = 0; P < 4; ++P) {
      acc[mt][P] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (BIAS) ax[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (UNR) tot[mt][P] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  // ---- operands ----
  const MagicK mk = magic_consts();
  const BiasK bk = bias_consts<bf16>();
  const u32x4 ones = {ones2<T>(), ones2<T>(), ones2<T>(), ones2<T>()};
  uint32_t zmag = 0x54006400u;
  asm volatile("" : "+s"(zmag));
  const uint32_t ssel = e ? 0x07060302u : 0x05040100u;  // half e of two scale words
  const uint32_t zsel0 = 0x07000500u | ((uint32_t)(2 * e) << 16) | (uint32_t)(2 * e);
  uint32_t zmp[2] = {0u, 0u}, sc2[2] = {0u, 0u};  // biased zeros and scales of nibble positions 2 j, 2 j + 1
  uint32_t scd[2] = {0u, 0u}, zmd[2] = {0u, 0u};  // UNR: those of the group whose sums acc holds
  auto rd = [&](uint32_t addr) { return *(__attribute__((address_space(3))) const u32x4*)(uintptr_t)addr; };
  int rcslot = 0;  // set slot of the next read
  auto prep = [&] {
    const uint32_t ca = lds_c + (uint32_t)rcslot * 512u;
    rcslot = rcslot + 1 == NCS ? 0 : rcslot + 1;
    const u32x4 s4 = rd(ca + 16u * (uint32_t)r);
    const uint32_t zw = *(__attribute__((address_space(3))) const uint32_t*)(uintptr_t)(ca + 256u + 4u * (uint32_t)r) | z_none;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      scd[h] = sc2[h];
      zmd[h] = zmp[h];
      zmp[h] = __builtin_amdgcn_perm(zmag, zw, zsel0 + (uint32_t)h * 0x00010001u) & 0xFFF0FF0Fu;
      sc2[h] = __builtin_amdgcn_perm(s4[2 * h + 1], s4[2 * h], ssel);
    }
  };
  auto scale_of = [&](uint32_t pair, int P) {
    const uint16_t sb = (uint16_t)(pair >> (16 * (P & 1)));
    return FAST || !wk.scale_bf16 ? h_bits2f(sb) : bf_bits2f(sb);
  };
  // nibble position P of a weight piece -> the MFMA operand of its 16 columns
  auto operand = [&](const u32x4& w, auto pc) {
    constexpr int P = decltype(pc)::value;
    const f16x2 zh = as_h2(zmp[P >> 1]);
    const f16x2 zz = (P & 1) ? __builtin_shufflevector(zh, zh, 1, 1) : __builtin_shufflevector(zh, zh, 0, 0);
    u32x4 v;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (BIAS) {
        v[u] = ((w[u] >> (4 * P)) & bk.mask) | bk.magic;  // 128 + q
        continue;
      }
      const f16x2 d = as_h2(magic_bits<P>(w[u], mk)) - zz;  // exact q - z
      if constexpr (UNR) {
        if constexpr (std::is_same<T, f16>::value) v[u] = as_u(d);
        else v[u] = pack2<T>((float)d.x, (float)d.y);
      } else if constexpr (FAST) {
        const f16x2 sh = as_h2(sc2[P >> 1]);
        const f16x2 ss = (P & 1) ? __builtin_shufflevector(sh, sh, 1, 1) : __builtin_shufflevector(sh, sh, 0, 0);
        v[u] = as_u(d * ss);
      } else {
        const float sf = scale_of(sc2[P >> 1], P);
        v[u] = pack2<T>(scaled_int(d.x, sf), scaled_int(d.y, sf));
      }
    }
    return v;
  };
  u32x4 op[2][4];  // operands of the current and the next k-step
  auto form = [&](const u32x4& w, int P) {  // P is a constant after unrolling
    return P == 0   ? operand(w, std::integral_constant<int, 0>{})
           : P == 1 ? operand(w, std::integral_constant<int, 1>{})
           : P == 2 ? operand(w, std::integral_constant<int, 2>{})
                    : operand(w, std::integral_constant<int, 3>{});
  };
  auto read_w = [&](int wslot) { return rd(lds_w + (uint32_t)wslot * 1024u + (uint32_t)lane * 16u); };
  // tot += the finished group's sums (its scales and biased zeros in `s`, `z`)
  auto scale_row = [&](int mt, const uint32_t (&s)[2], const uint32_t (&z)[2]) {
    if constexpr (UNR) {
#pragma unroll
      for (int P = 0; P < 4; ++P) {
        const float sf = scale_of(s[P >> 1], P);
        // 1024 + z and 64 + z of the fp16 form -> 128 + z
        const f16x2 zh = as_h2(z[P >> 1]);
        const float cz = BIAS ? (((P & 1) ? (float)zh.y + 64.0f : (float)zh.x - 896.0f) * sf) : 0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float t = __builtin_fmaf(acc[mt][P][v], sf, tot[mt][P][v]);
          if constexpr (BIAS) t = __builtin_fmaf(-cz, ax[mt][v], t);
          tot[mt][P][v] = t;
        }
      }
    }
  };
  // operand read addresses of a stage's two k-steps (row tile mt at + 2048 mt)
  uint32_t ra[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) ra[j] = lds0 + (uint32_t)(part * ABYTES + r * 128 + ((4 * j + q) ^ swz(r)) * 16);

  // Requests of k-step n, in this order: the first (even n) or second half of the activations of stage
  // n / 2 + NA - 1, the weight piece of k-step n + R, its constants if a set starts there.  A wave
  // issuing them in a row would wait for the CU's texture path at each, so they are spread over the
  // k-step's MFMAs.  a_count and req_count are their numbers per phase (n modulo the loop's unroll).
  constexpr int UN = UK > 2 ? UK : 2;
  auto a_count = [](int n) constexpr { return (n & 1) ? ND / 2 : ND - ND / 2; };
  auto req_count = [a_count](int n) constexpr { return a_count(n) + 1 + ((n + R) % SPG == 0 ? 2 : 0); };
  // requests still allowed in flight at the top of k-step n (n large): weights and constants of k-step
  // n + 1 (requested at n + 1 - R) have landed and, where a stage starts, its activations (whose second
  // half came first in k-step n - 2 NA + 3)
  auto in_flight = [a_count, req_count](int n) constexpr {
    int w = 0;
    for (int m = n + 2 - R; m <= n - 1; ++m) w += req_count(m);
    if (n % 2 == 0) {
      int a = -a_count(n - 2 * NA + 3);
      for (int m = n - 2 * NA + 3; m <= n - 1; ++m) a += req_count(m);
      w = a < w ? a : w;
    }
    return w;
  };
  // request i of k-step n (phase u); slots: of stage n / 2 + NA - 1, of weights n + R, of the next set
  int wslot = 0, cslot = 0;  // ring slots: weight piece of the next k-step to read, next set to request
  auto request = [&](int n, int u, int i, int aslot, int wslot_) {
    const int na = a_count(u);
    if (i < na) req_a((n >> 1) + NA - 1, aslot, (u & 1) ? ND - ND / 2 + i : i);
    else if (i == na) req_w(n + R, wslot_);
    else req_c(n + R, cslot, i == na + 2);
  };
  int raslot = 0;  // activation slot of the current stage
  u32x4 a[2];
  auto kstep = [&](int n0, auto uc) {
    constexpr int u = decltype(uc)::value;  // n = n0 + u
    constexpr bool fresh = UNR && u % SPG == 0;
    constexpr int left = in_flight(u + 8 * UN);
    constexpr int nreq = req_count(u + 8 * UN);
    AWQ_WAIT_VMCNT(left);
    const uint32_t sg[2] = {scd[0], scd[1]}, zg[2] = {zmd[0], zmd[1]};
    if constexpr (u % 2 == 0) __syncthreads();
    else asm volatile("" ::: "memory");
    const uint32_t addr = ra[u & 1] + (uint32_t)(raslot * STAGE), addr1 = ra[1] + (uint32_t)(raslot * STAGE);
    const int fslot = raslot == 0 ? NA - 1 : raslot - 1;  // the slot the last stage left
    if constexpr (u % 2 == 0) a[0] = rd(addr);
    const int rw = wslot + 1 == R ? 0 : wslot + 1;
    const u32x4 w = read_w(rw);
    if constexpr ((u + 1) % SPG == 0) prep();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int ai = (u % 2) * MT + mt;  // parity of the operand buffers over the stage
      if (mt + 1 < MT) a[(ai + 1) & 1] = rd(addr + (uint32_t)((mt + 1) * 2048));
      else if constexpr (u % 2 == 0) a[(ai + 1) & 1] = rd(addr1);
      if constexpr (fresh) scale_row(mt, sg, zg);
#pragma unroll
      for (int P = 0; P < 4; ++P)
        acc[mt][P] = MfmaOp<T>::run(a[ai & 1], op[u & 1][P], fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mt][P]);
      if constexpr (BIAS) ax[mt] = MfmaOp<T>::run(a[ai & 1], ones, fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : ax[mt]);
#pragma unroll
      for (int P = mt * 4 / MT; P < (mt + 1) * 4 / MT; ++P) op[(u + 1) & 1][P] = form(w, P);
#pragma unroll
      for (int i = mt * nreq / MT; i < (mt + 1) * nreq / MT; ++i) request(n0 + u, u + 8 * UN, i, fslot, wslot);
      __builtin_amdgcn_sched_barrier(0);
    }
    wslot = rw;
    if constexpr ((u + R) % SPG == 0) cslot = cslot + 1 == NCS ? 0 : cslot + 1;
    if constexpr (u % 2 == 1) raslot = raslot + 1 == NA ? 0 : raslot + 1;
  };

  // prologue: the requests that the k-steps -2 NA + 2 .. -1 would have made
#pragma unroll
  for (int m = -(R > 2 * NA - 2 ? R : 2 * NA - 2); m < 0; ++m) {
    if (m >= -2 * NA + 2)
#pragma unroll
      for (int i = 0; i < a_count(m + 8 * UN); ++i) {
        const int st = ((m + 8 * UN) >> 1) - 4 * UN + NA - 1;
        req_a(st, st, (m & 1) ? ND - ND / 2 + i : i);
      }
    if (m >= -R) {
      req_w(m + R, m + R);
      if ((m + R) % SPG == 0) {
        req_c(m + R, cslot, false);
        req_c(m + R, cslot, true);
        cslot = cslot + 1 == NCS ? 0 : cslot + 1;
      }
    }
  }
  {
    constexpr int left0 = in_flight(8 * UN - 1);  // k-step 0's weights and constants
    AWQ_WAIT_VMCNT(left0);
    asm volatile("" ::: "memory");  // the reads stay behind the wait
    const u32x4 w = read_w(0);
    prep();
#pragma unroll
    for (int P = 0; P < 4; ++P) op[0][P] = form(w, P);
  }
  for (int n = 0; n < nkmax; n += UN) {
    kstep(n, std::integral_constant<int, 0>{});
    kstep(n, std::integral_constant<int, 1>{});
    if constexpr (UN == 4) {
      kstep(n, std::integral_constant<int, 2>{});
      kstep(n, std::integral_constant<int, 3>{});
    }
  }
  if constexpr (UNR)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) scale_row(mt, scd, zmd);
  AWQ_WAIT_VMCNT0();  // no DMA may land in the LDS that the sums below reuse

  // ---- the shares' sums meet: [share][row quad][column] x 4 rows; column 8 r + 2 P + e of the tile at
  // 64 e + 16 P + r.  Each output is summed in share order ----
  constexpr int RQ = RPASS / 4;
  const int rq_total = (p.M + 3) >> 2, rq0 = m0 >> 2;
  // partials: [range][row quad][column tile][128 columns] x 4 rows
  const __amdgpu_buffer_rsrc_t prs = make_rsrc(p.partial, (uint32_t)wk.splits * (uint32_t)rq_total * (uint32_t)wk.tiles * 2048u);
  const uint32_t pbase = (uint32_t)((split * rq_total + rq0) * wk.tiles + t) * 2048u;
  // four rows of columns 8 r + 2 P and the next -> the block's 16-bit output tile in LDS; whole rows of it
  // then leave in 16-byte pieces
  auto stage_out = [&](int rq, int pr, const f32x4 (&o)[2]) {
    __attribute__((address_space(3))) uint32_t* outl = (__attribute__((address_space(3))) uint32_t*)(uintptr_t)(lds0 + RED);
    const int P = pr >> 4, c = pr & 15, col = t * 128 + 8 * c + 2 * P;
    float b0 = 0.f, b1 = 0.f;
    if (p.bias && col < p.N) {
      b0 = load_bias(p.bias, p.bias_dtype, col);
      b1 = load_bias(p.bias, p.bias_dtype, col + 1);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) outl[(4 * rq + v) * 64 + 4 * c + P] = pack2<T>(o[0][v] + b0, o[1][v] + b1);
  };
  auto write_out = [&](int mp, int nq) {
    __syncthreads();
    for (int i = tid; i < nq * 64; i += 512) {  // (row, word)
      const int row = i >> 4, c = i & 15, grow = m0 + 16 * mp + row, gword = t * 16 + c;
      u32x4 v = rd(lds0 + (uint32_t)(RED + row * 256 + c * 16));
      if (std::is_same<T, f16>::value && p.c_bf16) v = via_bf16_words(v);
      if (grow < p.M && gword < NW) *(u32x4*)(p.c + (int64_t)grow * p.ldc + 8 * gword) = v;
    }
    __syncthreads();
  };
#pragma unroll
  for (int mp = 0; mp < MT; mp += 4) {
    __syncthreads();
#pragma unroll
    for (int mt = mp; mt < (mp + 4 < MT ? mp + 4 : MT); ++mt)
#pragma unroll
      for (int P = 0; P < 4; ++P)
        *(__attribute__((address_space(3))) f32x4*)(uintptr_t)(
            lds0 + (uint32_t)(((part * RQ + 4 * (mt - mp) + q) * 128 + 64 * e + 16 * P + r) * 16)) =
            UNR ? tot[UNR ? mt : 0][P] : acc[mt][P];
    __syncthreads();
    const int nq = (ROWS - 16 * mp < RPASS ? ROWS - 16 * mp : RPASS) / 4;
    for (int i = tid; i < nq * 64; i += 512) {  // (row quad, P, r): columns 8 r + 2 P, 8 r + 2 P + 1
      const int rq = i >> 6, pr = i & 63;
      f32x4 o[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t ad = lds0 + (uint32_t)((rq * 128 + 64 * h + pr) * 16);
        o[h] = *(__attribute__((address_space(3))) const f32x4*)(uintptr_t)ad;
#pragma unroll
        for (int w = 1; w < kMidShares; ++w)
          o[h] += *(__attribute__((address_space(3))) const f32x4*)(uintptr_t)(ad + (uint32_t)(w * RQ * 2048));
      }
      if (wk.splits == 1) {
        stage_out(rq, pr, o);
      } else if (rq0 + 4 * mp + rq < rq_total) {
        const int off = (int)pbase + ((4 * mp + rq) * wk.tiles * 128 + pr) * 16;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[0]), prs, off, 0, kDeviceCoherent);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[1]), prs, off + 1024, 0, kDeviceCoherent);
      }
    }
    if (wk.splits == 1) write_out(mp, nq);
  }
  if (!UNR || wk.splits == 1) return;

  // ---- K ranges, up to 64 rows: the block that arrives last at its (column tile, row tile) adds the ranges' partials in
  // range order.  The count is an agent-scope release after the block's (device-scope) stores and the
  // last block takes an acquire fence, as in the decode kernels.  Against a second launch over the
  // partials, N = K = 4096: M = 32 11.7 -> 10.5 us, M = 57 14.6 -> 13.3; above 64 rows, where one block
  // would read up to 400 KB and the tile's other row tiles wait, the second launch stays ahead
  // (mid_reduce_kernel; four projections of 200 rows, twice: 270 against 289 us) ----
  __attribute__((address_space(3))) int* s_last = (__attribute__((address_space(3))) int*)(uintptr_t)lds0;  // the sums are done with
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int* counter = p.counters + rt * wk.tiles + t;
  if (tid == 0) {
    *s_last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) == wk.splits - 1;
    if (*s_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  if (!*s_last) return;
  const uint32_t plane = (uint32_t)rq_total * (uint32_t)wk.tiles * 2048u;  // bytes between ranges
#pragma unroll
  for (int mp = 0; mp < MT; mp += 4) {
    const int nq = (ROWS - 16 * mp < RPASS ? ROWS - 16 * mp : RPASS) / 4;
    for (int i = tid; i < nq * 64; i += 512) {
      const int rq = i >> 6, pr = i & 63;
      if (rq0 + 4 * mp + rq >= rq_total) continue;
      const uint32_t off = (uint32_t)(((rq0 + 4 * mp + rq) * wk.tiles + t) * 128 + pr) * 16u;
      f32x4 o[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
      for (int s0 = 0; s0 < wk.splits; s0 += 4) {  // four ranges' loads in flight; those past the last read zero
        f32x4 v[4][2];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            v[s][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                    prs, s0 + s < wk.splits ? (int)(off + (uint32_t)(s0 + s) * plane + 1024u * h) : (int)0x80000000,
                                                    0, kDeviceCoherent));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          o[0] += v[s][0];
          o[1] += v[s][1];
        }
      }
      stage_out(rq, pr, o);
    }
    write_out(mp, nq);
  }
  if (tid == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// c[4 rq + v][...] = round(sum over splits, in split order, of the partials + bias): a wave per (row
// quad, column tile), lane (P, r) holding columns 8 r + 2 P and the next; rows leave through LDS in
// 16-byte pieces.
template <typename T>
__global__ void __launch_bounds__(256) mid_reduce_kernel(const GemmArgs p, const MidWork wk) {
  __shared__ uint32_t outl[4][256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rq_total = (p.M + 3) >> 2;
  const int item = (int)blockIdx.x * 4 + wave;  // (row quad, column tile)
  const bool on = item < rq_total * wk.tiles;
  const int rq = item / wk.tiles, t = item - rq * wk.tiles;
  const int P = lane >> 4, c = lane & 15;
  if (on) {
    const size_t plane = (size_t)rq_total * (size_t)wk.tiles * 128;
    const f32x4* src = (const f32x4*)p.partial + (size_t)item * 128 + lane;
    f32x4 o[2] = {src[0], src[64]};
    for (int s = 1; s < wk.splits; ++s) {
      o[0] += src[(size_t)s * plane];
      o[1] += src[(size_t)s * plane + 64];
    }
    const int col = t * 128 + 8 * c + 2 * P;
    float b0 = 0.f, b1 = 0.f;
    if (p.bias && col < p.N) {
      b0 = load_bias(p.bias, p.bias_dtype, col);
      b1 = load_bias(p.bias, p.bias_dtype, col + 1);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) outl[wave][v * 64 + 4 * c + P] = pack2<T>(o[0][v] + b0, o[1][v] + b1);
  }
  __syncthreads();
  const int grow = 4 * rq + P, gword = t * 16 + c;
  if (on && grow < p.M && gword < (p.N >> 3)) {
    u32x4 v = *(const u32x4*)&outl[wave][P * 64 + 4 * c];
    if (std::is_same<T, f16>::value && p.c_bf16) v = via_bf16_words(v);
    *(u32x4*)(p.c + (int64_t)grow * p.ldc + 8 * gword) = v;
  }
}

}  // namespace awq

namespace awq_host {
using namespace awq;

// Partials of a plan up to 64 rows: at most what the allocation-free entry point's scratch holds.
constexpr size_t kMidPartialMax = (size_t)8 << 20;
bool launch_mid_rounded(const GemmArgs& a, int mt, const MidWork& wk, int act, int sdt, hipStream_t st);

// false: no such instantiation (eight row blocks leave no LDS for the constant sets of groups of 32)
template <int MT, bool UNR, typename T, bool FAST>
inline bool launch_mid_g(const GemmArgs& a, const MidWork& wk, hipStream_t st) {
  const dim3 grid((unsigned)(wk.tiles * wk.splits * wk.row_tiles)), block(512);
  if (a.G >= 128) hipLaunchKernelGGL((mid_kernel<MT, UNR, T, FAST, 128>), grid, block, 0, st, a, wk);
  else if (a.G == 64) hipLaunchKernelGGL((mid_kernel<MT, UNR, T, FAST, 64>), grid, block, 0, st, a, wk);
  else if constexpr (mid_lds(MT, 32).r > 0) hipLaunchKernelGGL((mid_kernel<MT, UNR, T, FAST, 32>), grid, block, 0, st, a, wk);
  else return false;
  return true;
}

}  // namespace awq_host
