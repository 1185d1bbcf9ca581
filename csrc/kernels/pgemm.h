// What the prompt GEMMs share: the LDS-DMA piece, the epilogues' arithmetic, and what the persistent kernel takes.
#pragma once

#include <algorithm>

#include "common.h"

namespace {

typedef __attribute__((address_space(3))) void pg_lds_t;

// PG_F32: the fp32 accumulators themselves (row stride ldo in floats): a tensor-parallel row-parallel
// projection's partial, all-reduced in fp32 and rounded to bf16 once, as TP = 1 rounds the full sum
enum { PG_BF16 = 0, PG_BIAS = 1, PG_BIAS_GELU = 2, PG_SWIGLU = 3, PG_F32 = 4, PG_GLU = 5, PG_RELU2 = 6 };

// One 1-KB LDS-DMA piece from sbase + voff (per lane): lane l's 16 bytes land at lds_addr + 16 l.
// SGPR base + 32-bit VGPR offset (one VGPR per piece instead of a 64-bit pointer).  M0 is saved and
// restored inside the statement.
__device__ __forceinline__ void pg_glds16(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  unsigned keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(voff), "s"(sbase), "s"(lds_addr)
      : "memory");
}

// x Phi(x) = max(x, 0) - |x| erfc(|x| / sqrt 2) / 2, erfc by Hastings' rational approximation (Abramowitz and
// Stegun 7.1.26: t = 1 / (1 + p y), five terms, times exp(-y^2), within 1.5e-7).  About 15 instructions, two of
// them transcendental, where erff takes some fifty; as far from x Phi(x) as that is below x = -3, where 1 + erf
// cancels, within 4e-7 everywhere.  Rounded to bf16 (over all bf16 x, rms against 64 bits) as near as erff's above -3 and
// below -4, where that loses all digits by -6, 0.2 % further between.  The encoder's up product over 65 k rows with both:
// 230 -> 155 us.
// The last product takes min(x, FLT_MAX): exp(-y^2) of +inf is 0, and inf * 0 no number; of -inf it stays none, as
// x Phi(x) computed by its factors.
__device__ __forceinline__ float pg_gelu(float v) {
  const float a = fabsf(v);
  const float t = __builtin_amdgcn_rcpf(fmaf(a, 0.3275911f * 0.70710678f, 1.f));
  float q = fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
  q = fmaf(q, t, 0.5f * 1.421413741f);
  q = fmaf(q, t, 0.5f * -0.284496736f);
  q = fmaf(q, t, 0.5f * 0.254829592f) * t;
  return fmaf(-fabsf(fminf(v, 3.402823466e38f)), q * __builtin_amdgcn_exp2f(a * a * (-0.5f * 1.44269504f)), fmaxf(v, 0.f));
}

__device__ __forceinline__ float pg_bfr(float v) { return bf2f(f2bf(v)); }

// Gated epilogues over 8-row interleaved gate / up weights: PG_SWIGLU silu(g) * u, and PG_GLU
// min(g, limit) sigmoid(alpha g (1 + cubic g^2)) (clamp(u, +-limit) + beta) with the constants of PgGlu.
struct PgGlu { float limit = 0.f, alpha = 1.f, beta = 0.f, cubic = 0.f; };
constexpr bool pg_gated(int epi) { return epi == PG_SWIGLU || epi == PG_GLU; }

// SwiGLU of one 4-value accumulator group (16-row n-tile = 8 gate rows then 8 up rows: lanes
// g = 0, 1 hold gate columns, lanes g = 2, 3 -- lane ^ 32 -- the matching up columns).  One VALU lane
// swap (v_permlane32_swap, common.h) of (v[0], v[2]) gives every lane a (gate, up) pair -- element 0
// in lanes g < 2, element 2 in lanes g >= 2 -- and one of (v[1], v[3]) elements 1 / 3, so every lane
// computes two outputs (no idle lane half, no LDS-crossbar shuffles) and returns them packed: output
// columns pg_gate_col(g) + {0, 1} of the n-tile's 8.  Same values and rounding as the unfused
// GEMM -> silu_mul path: bf16 of gate and up, silu(g) * u in fp32.
template <int EPI>
__device__ __forceinline__ uint32_t pg_gate2(const float (&v)[4], const PgGlu& p) {
  float g0 = v[0], u0 = v[2], g1 = v[1], u1 = v[3];
  swap32(g0, u0);
  swap32(g1, u1);
  if constexpr (EPI == PG_GLU) {
    auto glu = [&](float gate, float up) {
      const float gg = fminf(gate, p.limit), uu = fminf(fmaxf(up, -p.limit), p.limit);
      return gg * __builtin_amdgcn_rcpf(1.f + __expf(-p.alpha * gg * (1.f + p.cubic * gg * gg))) * (uu + p.beta);
    };
    return pack2bf(glu(g0, u0), glu(g1, u1));
  }
  auto f = [](float gate, float up) {
    const float gg = pg_bfr(gate);
    return gg * __builtin_amdgcn_rcpf(1.f + __expf(-gg)) * pg_bfr(up);
  };
  return pack2bf(f(g0, u0), f(g1, u1));
}

__device__ __forceinline__ int pg_gate_col(int g) { return 4 * (g & 1) + 2 * (g >> 1); }

// what a value leaves as: PG_RELU2 its squared positive part
template <int EPI>
__device__ __forceinline__ float pg_out(float v) {
  if constexpr (EPI == PG_RELU2) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

// us of pgemm's persistent kernel in tiles of 32 mt x 256 (mt = 6, 7, 8): a K-tile of 256 rows takes 1.4 in a full round of
// workgroups, 0.8 to 1.22 in a partial one; of 224 rows 0.91 of that, of 192 0.83, on an idle chip 0.95 and 0.88 to 0.97 (what
// the waves read from LDS, not the MFMAs, takes the time there); all of it 0.945, and 7 % more in a run of 1.2 ms or longer, whose clock
// is lower, 1 or 2 % more again in the lower tiles.  Within 3 to 4 % of 1650 measured: 257 to 15 049 rows of 1024 .. 28672 x 2048 .. 14336.
inline double ppp_us_at(int M, int N, int K, int mt) {
  constexpr int CUS = 256;
  const int64_t tiles = (int64_t)((M + 32 * mt - 1) / (32 * mt)) * ((N + 255) / 256);
  const double full = (double)(tiles / CUS), fill = (double)(tiles % CUS) / CUS;
  const double part = fill > 0 ? 0.8 + 0.42 * fill : 0.0;
  const double all = mt == 6 ? 0.83 : mt == 7 ? 0.91 : 1.0;
  const double idle = mt == 6 ? (full > 0 ? 0.14 : 0.05) : mt == 7 && full > 0 ? 0.04 : 0.0;
  const double us = 12.0 + K / 64 * (1.4 * full * all + part * (all + idle * (1.0 - fill)));
  const double slow = us < 1200.0 ? us / 1200.0 : 1.0;
  return us * (0.945 + 0.07 * slow) * (1.0 + 0.01 * (8 - mt) * slow);
}

// The height that takes the least: fewer rows than 256 where they leave fewer rows of the last tile unused or fill the last
// round (us of 28672 x 4096, 256 rows -> this: 285 / 351 rows 85 -> 76 / 87 -> 74 and
// 1107 243 -> 226 in 192; 433 88 -> 82, 896 175 -> 163 and 1344 256 -> 242 in 224; 4096 x 14336 3491 282 -> 276): 0.3 % more than the fastest of the three
// on average of the sizes above.
// The sums are the same in every height, so it changes no bit.
inline int ppp_height(int M, int N, int K) {
  int best = 8;
  double least = 0.985 * ppp_us_at(M, N, K, 8);
  for (int mt = 7; mt >= 6; --mt) {
    const double t = ppp_us_at(M, N, K, mt);
    if (t < least) least = t, best = mt;
  }
  return best;
}

}  // namespace
