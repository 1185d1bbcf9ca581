// Sentence-encoder layers for gfx950, post-LN BERT with hidden 384 and inner 1536 (MiniLM-L6, bge-small), bf16 in and out:
//   x1 = LN(a Wo^T + bo + x), h = GELU(x1 Wu^T + bu), y = LN(h Wd^T + bd + x1), qkv = y Wq^T + bq
// around the attention (attention.hip).
//
// Many rows: one kernel from the attention's output to the layer's.  Product by product these have K = 384 or 1536 and
// outputs up to four times their inputs: over 65 k rows 311 us (o 45, up 155, down 110), 600 MB of rows written and read
// again, each tile's epilogue alone on its CU.  Here a row never leaves its lane between them, 226 us:
//
//   * a workgroup owns 128 rows, 32 in each of four pairs of waves.  v_mfma_f32_32x32x16_bf16 with the WEIGHTS as A and
//     the rows as B: a lane's accumulators are columns of ONE row (lane & 31), half of them its own, half those of
//     lane ^ 32, so a LayerNorm is a sum over the lane's registers and one lane swap;
//   * a pair of waves shares a SIMD and its 32 rows, half the registers each.  One holds the rows as operands (96
//     registers) and takes the up product, 32 hidden columns at a time, with the GELU of the 32 before them between its
//     MFMAs; the other holds 384 columns of accumulators (192), takes the attention's projection, the down product and
//     both norms, and issues the weights' loads.  Hidden rows go from one to the other through 2 KB of LDS a pair;
//   * the accumulator layout of one product becomes the B operand of the next by packing to bf16 and one
//     v_permlane32_swap per two registers (trade): rows and residuals stay in registers, and an accumulator starts from
//     its bias and residual;
//   * only the weights move: stages of 24 KB (32 columns x 384, or 384 columns x 32), five in a ring of LDS-DMA behind
//     counted waits, two an interval, one barrier per interval of 24 MFMAs of either wave.
// What bounds it: with all CUs at work the clock, 1.9 GHz of 2.4 (products alone, without GELU, LDS reads and loads,
// take 81 us for a block of rows), and on an idle chip the up wave, whose 24 MFMAs, as many LDS reads and waits and 270
// vector instructions of GELU take 2500 cycles an interval (matrix cores 1536).  A block of rows takes 70 us on an idle
// chip and 100 with all CUs at work; one wave per SIMD with all 384 registers took 87 and 114 (an instruction every six
// cycles), two waves with half the columns each and opposite phases 90 and 115 (both wait for the one with the GELU).
#include "common.h"

#include <cstring>

namespace {

typedef __attribute__((address_space(3))) void en_lds_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int EN_H = 384, EN_F = 1536;           // hidden, inner
constexpr int EN_T = EN_H / 32;                  // 32-column tiles of a row
constexpr int EN_S = EN_H / 16;                  // 16-deep k steps of a row
constexpr int EN_ROWS = 128;                     // rows per workgroup, 32 per wave or pair of waves
constexpr int EN_STAGE = 24 * 1024, EN_RING = 5; // a stage of weights, stages

__device__ __forceinline__ f32x16_t mfma32(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// One 1-KB LDS-DMA piece: lane l's 16 bytes of sbase + voff land at lds_addr + 16 l (M0 kept).
__device__ __forceinline__ void en_glds16(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  unsigned keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(voff), "s"(sbase), "s"(lds_addr)
      : "memory");
}

// x Phi(x) = max(x, 0) - |x| erfc(|x| / sqrt 2) / 2, erfc by Abramowitz and Stegun 7.1.26 (as pgemm.h's, but none of
// +inf: either way the row's norm makes no number of all its states), in three parts of about an MFMA's length.
struct Gelu { float t, m, q; };
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }
template <int PART>
__device__ __forceinline__ void en_gelu(Gelu& g, float& v) {
  if constexpr (PART == 0) {
    pin(v);
    g.t = __builtin_amdgcn_rcpf(fmaf(fabsf(v), 0.3275911f * 0.70710678f, 1.f));
    g.m = v * v * (-0.5f * 1.44269504f);
    pin(g.t);
    pin(g.m);
  } else if constexpr (PART == 1) {
    pin(g.m);
    const float e = __builtin_amdgcn_exp2f(g.m);
    float q = fmaf(g.t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
    q = fmaf(q, g.t, 0.5f * 1.421413741f);
    q = fmaf(q, g.t, 0.5f * -0.284496736f);
    q = fmaf(q, g.t, 0.5f * 0.254829592f) * g.t;
    g.q = q * e;
    pin(g.q);
  } else {
    pin(g.q);
    v = fmaf(-fabsf(v), g.q, fmaxf(v, 0.f));
    pin(v);
  }
}

// of a whole accumulator, part by part: one value's chain of operations is the others' waits
template <int N>
__device__ __forceinline__ void en_gelus(float __attribute__((ext_vector_type(N))) & a) {
  Gelu ge[N];
  float v[N];
#pragma unroll
  for (int e = 0; e < N; ++e) v[e] = a[e], en_gelu<0>(ge[e], v[e]);
#pragma unroll
  for (int e = 0; e < N; ++e) en_gelu<1>(ge[e], v[e]);
#pragma unroll
  for (int e = 0; e < N; ++e) en_gelu<2>(ge[e], v[e]), a[e] = v[e];
}

// Sixteen columns of a row block between its two layouts, its own inverse.  Accumulators: a lane holds columns
// 4 hi + 0..3 and 8 + 4 hi + 0..3 (hi = lane >> 5); operands: columns 8 hi + 0..7.
__device__ __forceinline__ u32x4_t trade(u32x4_t v) {
  const auto p = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
  const auto q = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  return u32x4_t{p[0], q[0], p[1], q[1]};
}

// accumulators 8 s .. 8 s + 7 of a tile -> operand of k step s
__device__ __forceinline__ bf16x8_t frag_of(const f32x16_t& a, int s) {
  const u32x4_t v = {pack2bf(a[8 * s], a[8 * s + 1]), pack2bf(a[8 * s + 2], a[8 * s + 3]), pack2bf(a[8 * s + 4], a[8 * s + 5]),
                     pack2bf(a[8 * s + 6], a[8 * s + 7])};
  return __builtin_bit_cast(bf16x8_t, trade(v));
}

struct EncLayer {
  const uint16_t *wo, *bo, *g1, *b1, *wu, *bu, *wd, *bd, *g2, *b2;
};

// Intervals, each with the stages 2 T and 2 T + 1 of the weight stream: 6 of Wo (two 32-deep slices each), then 50 of the
// feed-forward (group g's up columns and the down slice g - 2: GELU of g - 1 lies between).
constexpr int EN_O = EN_T / 2, EN_C = EN_F / 32;
constexpr int EN_HX = 2 * 4 * 2048;              // hidden rows in LDS: two groups of 128 x 32
constexpr int EN_VEC = 5;                        // vectors in LDS: g1, b1, bd, g2, b2
constexpr int EN_LDS = EN_RING * EN_STAGE + EN_HX + 4 * EN_F + EN_VEC * 4 * EN_H;
constexpr int EN_UA = 6, EN_DA = 4;              // fragments read ahead of their MFMA, by the up and the other waves
constexpr int EN_MEET = 20;                      // MFMAs of a group ahead of its barrier: all its fragments are read by then
static_assert(EN_MEET + EN_UA >= 24 && EN_MEET + EN_DA >= 24 && EN_LDS <= 160 * 1024, "");

__device__ __forceinline__ void en_meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// acc: the rows less their means, and 1 / their deviations.  Four chains of sums: one would wait for each addition.
__device__ __forceinline__ float en_center(f32x16_t (&acc)[EN_T], float eps) {
  float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < EN_T; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r & 3] += acc[t][r];
  const float mean = xor32_sum((p[0] + p[1]) + (p[2] + p[3])) * (1.f / EN_H);
  float q[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < EN_T; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[t][r] -= mean;
      q[r & 3] = fmaf(acc[t][r], acc[t][r], q[r & 3]);
    }
  return rsqrtf(xor32_sum((q[0] + q[1]) + (q[2] + q[3])) * (1.f / EN_H) + eps);
}

__global__ void __launch_bounds__(512, 2)
    enc_layer_kernel(const uint16_t* __restrict__ att, const uint16_t* x, EncLayer L, uint16_t* xout, int M, float eps) {
  extern __shared__ __attribute__((aligned(16))) char en_smem[];
  const int lane = threadIdx.x & 63, hi = lane >> 5, r32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wave & 3;
  const int row = blockIdx.x * EN_ROWS + w * 32 + r32;
  typedef const __attribute__((address_space(3))) bf16x8_t* lds_frag_t;
  typedef __attribute__((address_space(3))) bf16x8_t* lds_out_t;

  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(en_lds_t*)en_smem);
  const uint32_t hx = lds0 + EN_RING * EN_STAGE + w * 2048 + lane * 16;
  const uint32_t trade_at = lds0 + w * 12288 + lane * 16;
  float* bu = reinterpret_cast<float*>(en_smem + EN_RING * EN_STAGE + EN_HX);
  float* vec = bu + EN_F;

  // ---- weight stream.  Slices (384 rows x 64 B): pieces of 16 rows, 16-byte chunk c of row r at slot c ^ ((r >> 2) & 3);
  // column groups (32 rows x 768 B): pieces of 8 rows x 128 B, chunk c at slot c ^ ((r >> 1) & 7).  LDS serves sixteen
  // lanes' 16 bytes a cycle where they lie in 64 banks: rows of 128 bytes need the swizzle to step every second row (r & 7
  // there reads 1.6 times as long).
  const int srow = lane >> 2;
  const uint32_t sch = ((lane & 3) ^ (srow >> 2)) << 4;
  const char* wo = reinterpret_cast<const char*>(L.wo) + (size_t)w * 96 * EN_H * 2;
  const char* wd = reinterpret_cast<const char*>(L.wd) + (size_t)w * 96 * EN_F * 2;
  const char* wu = reinterpret_cast<const char*>(L.wu) + (size_t)w * 8 * EN_H * 2;
  const uint32_t v_o = srow * EN_H * 2 + sch, v_d = srow * EN_F * 2 + sch;
  const uint32_t v_n = (lane >> 3) * EN_H * 2 + (((lane & 7) ^ (((w & 1) << 2) + (lane >> 4))) << 4);
  auto slot_of = [](int idx) { return (uint32_t)(idx % EN_RING); };
  auto place = [&](int idx) { return lds0 + slot_of(idx) * EN_STAGE; };
  // wave w's piece i (0 .. 5) of a stage: number 6 w + i of a slice, w + 4 i of a group; past either end, of no use
  auto piece_o = [&](int k, int i, uint32_t at) { en_glds16(v_o, wo + i * (16 * EN_H * 2) + 64 * k, at + (6 * w + i) * 1024); };
  auto piece_d = [&](int g, int i, uint32_t at) {
    en_glds16(v_d, wd + i * (16 * EN_F * 2) + 64 * min(max(g - 2, 0), EN_C - 1), at + (6 * w + i) * 1024);
  };
  auto piece_u = [&](int g, int i, uint32_t at) {
    en_glds16(v_n, wu + (uint32_t)min(g, EN_C - 1) * (32u * EN_H * 2) + 128 * i, at + (w + 4 * i) * 1024);
  };

  struct Base { uint32_t s[4]; };
  uint32_t so[2], go[4];
#pragma unroll
  for (int s = 0; s < 2; ++s) so[s] = r32 * 64 + (((2 * s + hi) ^ ((r32 >> 2) & 3)) << 4);
#pragma unroll
  for (int s = 0; s < 4; ++s) go[s] = r32 * 128 + (((2 * s + hi) ^ ((r32 >> 1) & 7)) << 4);
  auto ld = [](uint32_t a) { return *reinterpret_cast<lds_frag_t>(a); };

  if (wave >= 4) {
    // ================================================= the up product and its GELU; Wo's stream
    __builtin_amdgcn_s_setprio(2);                // the longer of the two: 102 -> 100 us
    bf16x8_t fr[EN_UA];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int i = 0; i < 6; ++i) piece_o(q, i, place(q));
    for (int i = threadIdx.x - 256; i < EN_F; i += 256) bu[i] = bf2f(L.bu[i]);
    {
      const uint16_t* src[EN_VEC] = {L.g1, L.b1, L.bd, L.g2, L.b2};
#pragma unroll
      for (int v = 0; v < EN_VEC; ++v)
        for (int i = threadIdx.x - 256; i < EN_H; i += 256) vec[v * EN_H + i] = bf2f(src[v][i]);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int T = 0; T < EN_O; ++T) {
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        if (T + 1 < EN_O) piece_o(2 * T + 3, i, place(2 * T + 3));
        else piece_d(0, i, place(2 * T + 3));
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        if (T + 2 < EN_O) piece_o(2 * T + 4, i, place(2 * T + 4));
        else piece_u(T + 2 - EN_O, i, place(2 * T + 4));
      }
      if (T + 1 < EN_O) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    bf16x8_t xf[EN_S];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      en_meet();                                  // half the operands are there
#pragma unroll
      for (int i = 0; i < 12; ++i) xf[12 * p + i] = ld(trade_at + i * 1024);
      en_meet();                                  // and read
    }
    f32x16_t a, b;
    auto biases = [&](f32x16_t& v, int g, int i) {
      const float4 f = *reinterpret_cast<const float4*>(bu + 32 * min(g, EN_C - 1) + 8 * i + 4 * hi);
      v[4 * i] = f.x; v[4 * i + 1] = f.y; v[4 * i + 2] = f.z; v[4 * i + 3] = f.w;
    };
    Base cur;
    auto base_of = [&](int T) {
      Base p;
#pragma unroll
      for (int s = 0; s < 4; ++s) p.s[s] = place(2 * T) + go[s];
      return p;
    };
    cur = base_of(EN_O);
#pragma unroll
    for (int i = 0; i < EN_UA; ++i) fr[i] = ld(cur.s[i & 3] + (i >> 2) * 4096);
#pragma unroll
    for (int i = 0; i < 4; ++i) biases(a, 0, i);
#pragma unroll
    for (int r = 0; r < 16; ++r) b[r] = 0.f;
    // group g into `up` while the GELU of the group before, in `old`, runs; `old` then starts from the biases of g + 1
    auto group = [&](int g, f32x16_t& up, f32x16_t& old) {
      const uint32_t hout = hx + ((g + 1) & 1) * (4 * 2048);
      Base nb = cur;
      Gelu ge[2];
      u32x4_t hp;
#pragma unroll
      for (int i = 0; i < 24; ++i) {
        if (i == EN_MEET) {
          en_meet();
          nb = base_of(EN_O + g + 1);
        }
        up = mfma32(fr[i % EN_UA], xf[i], up);
        if (i + EN_UA < 24) fr[i % EN_UA] = ld(cur.s[(i + EN_UA) & 3] + ((i + EN_UA) >> 2) * 4096);
        if (i >= EN_MEET) {
#pragma unroll
          for (int n = i == EN_MEET ? 0 : i + EN_UA - 24; n <= i + EN_UA - 24; ++n) fr[n] = ld(nb.s[n & 3] + (n >> 2) * 4096);
        }
#pragma unroll
        for (int q = i * 24 / EN_MEET; i < EN_MEET && q < (i + 1) * 24 / EN_MEET; ++q) {     // two elements' GELU, a third at a time
          const int e = q / 3 * 2;
          float v0 = old[e], v1 = old[e + 1];
          if (q % 3 == 0) { en_gelu<0>(ge[0], v0); en_gelu<0>(ge[1], v1); }
          if (q % 3 == 1) { en_gelu<1>(ge[0], v0); en_gelu<1>(ge[1], v1); }
          if (q % 3 == 2) {
            en_gelu<2>(ge[0], v0);
            en_gelu<2>(ge[1], v1);
            hp[(e >> 1) & 3] = pack2bf(v0, v1);
            asm volatile("" : "+v"(hp[(e >> 1) & 3]));
            if ((e & 7) == 6) *reinterpret_cast<lds_out_t>(hout + (e >> 3) * 1024) = __builtin_bit_cast(bf16x8_t, trade(hp));
          }
        }
        if (i >= EN_MEET) biases(old, g + 1, i - EN_MEET);
        __builtin_amdgcn_sched_barrier(0);
      }
      cur = nb;
    };
    for (int g = 0; g < EN_C + 2; g += 2) {
      group(g, a, b);
      group(g + 1, b, a);
    }
    return;
  }

  // =================================================== the products into 384 columns, the norms; the feed-forward's stream
  f32x16_t acc[EN_T];
  bf16x8_t af[4], fr[EN_DA];                      // of the rows, of the weights
  const uint16_t* ar = att + (size_t)min(row, M - 1) * EN_H + 8 * hi;
  const uint16_t* xr = x + (size_t)min(row, M - 1) * EN_H + 8 * hi;
#pragma unroll
  for (int i = 0; i < 4; ++i) af[i] = *reinterpret_cast<const bf16x8_t*>(ar + 16 * i);
  // columns 8 i + 4 hi + 0..3 of tile t, of a vector in LDS
  auto four = [&](const float* p, int t, int i) { return *reinterpret_cast<const float4*>(p + 32 * t + 8 * i + 4 * hi); };
  // v[4 i ..] += the operand pair's bf16 values
  auto add2 = [](f32x16_t& v, int i, uint32_t a, uint32_t b) {
    v[4 * i] += __uint_as_float(a << 16); v[4 * i + 1] += __uint_as_float(a & 0xffff0000u);
    v[4 * i + 2] += __uint_as_float(b << 16); v[4 * i + 3] += __uint_as_float(b & 0xffff0000u);
  };
#pragma unroll
  for (int t = 0; t < EN_T; ++t) {                // the product starts from its bias and the residual
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint2 b = *reinterpret_cast<const uint2*>(L.bo + 32 * t + 8 * i + 4 * hi);
      acc[t][4 * i] = __uint_as_float(b.x << 16); acc[t][4 * i + 1] = __uint_as_float(b.x & 0xffff0000u);
      acc[t][4 * i + 2] = __uint_as_float(b.y << 16); acc[t][4 * i + 3] = __uint_as_float(b.y & 0xffff0000u);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x4_t r = trade(*reinterpret_cast<const u32x4_t*>(xr + 32 * t + 16 * s));
      add2(acc[t], 2 * s, r[0], r[1]);
      add2(acc[t], 2 * s + 1, r[2], r[3]);
    }
  }
  Base cur;
  auto base_of = [&](int idx) {
    Base p;
#pragma unroll
    for (int s = 0; s < 2; ++s) p.s[s] = place(idx) + so[s];
    return p;
  };
  auto frag = [&](const Base& p, int i) { return ld(p.s[i / EN_T] + (i % EN_T) * 2048); };
  en_meet();
#pragma unroll 1
  for (int T = 0; T < EN_O; ++T) {
    const Base st[2] = {base_of(2 * T), base_of(2 * T + 1)};
    ar += 64;
    const uint16_t* nx = T + 1 < EN_O ? ar : xr;   // the next interval's operands, at the end of no use
#pragma unroll
    for (int i = 0; i < EN_DA; ++i) fr[i] = frag(st[0], i);
#pragma unroll
    for (int i = 0; i < 48; ++i) {
      const int k = i / EN_T;
      acc[i % EN_T] = mfma32(fr[i % EN_DA], af[k], acc[i % EN_T]);
      if (i + EN_DA < 48) fr[i % EN_DA] = frag(st[(i + EN_DA) / 24], (i + EN_DA) % 24);
      if (i % EN_T == EN_T - 1) af[k] = *reinterpret_cast<const bf16x8_t*>(nx + 16 * k);
      __builtin_amdgcn_sched_barrier(0);
    }
    en_meet();
  }
  {
    const float rstd = en_center(acc, eps);
#pragma unroll
    for (int t = 0; t < EN_T; ++t) {
      // to the other waves through the two stages that are free, half the columns at a time
      if (t == EN_T / 2) { en_meet(); en_meet(); }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        u32x4_t y;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float4 g = four(vec, t, 2 * s + i), b = four(vec + EN_H, t, 2 * s + i), d = four(vec + 2 * EN_H, t, 2 * s + i);
          const int o = 8 * s + 4 * i;
          y[2 * i] = pack2bf(fmaf(acc[t][o], rstd * g.x, b.x), fmaf(acc[t][o + 1], rstd * g.y, b.y));
          y[2 * i + 1] = pack2bf(fmaf(acc[t][o + 2], rstd * g.z, b.z), fmaf(acc[t][o + 3], rstd * g.w, b.w));
          acc[t][o] = d.x; acc[t][o + 1] = d.y; acc[t][o + 2] = d.z; acc[t][o + 3] = d.w;
          add2(acc[t], 2 * s + i, y[2 * i], y[2 * i + 1]);      // the next product starts from its bias and these rows
        }
        *reinterpret_cast<lds_out_t>(trade_at + ((2 * t + s) % 12) * 1024) = __builtin_bit_cast(bf16x8_t, trade(y));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  en_meet();
  en_meet();

  cur = base_of(2 * EN_O + 1);
#pragma unroll
  for (int i = 0; i < EN_DA; ++i) fr[i] = frag(cur, i);
  bf16x8_t h0, h1;
  h0 = h1 = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});            // the first two groups add zeros
  for (int g = 0; g < EN_C + 2; ++g) {
    const int T = EN_O + g;
    const uint32_t hin = hx + ((g + 1) & 1) * (4 * 2048), pd = place(2 * T + 3), pu = place(2 * T + 4);
    Base nb = cur;
#pragma unroll
    for (int i = 0; i < 24; ++i) {
      if (i == EN_MEET) {
        asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        nb = base_of(2 * T + 3);
      }
      acc[i % EN_T] = mfma32(fr[i % EN_DA], i < EN_T ? h0 : h1, acc[i % EN_T]);
      if (i + EN_DA < 24) fr[i % EN_DA] = frag(cur, i + EN_DA);
      if (i >= EN_MEET) {
#pragma unroll
        for (int n = i == EN_MEET ? 0 : i + EN_DA - 24; n <= i + EN_DA - 24; ++n) fr[n] = frag(nb, n);
      }
      if (i < 6) piece_d(g + 1, i, pd);
      else if (i < 12) piece_u(g + 2, i - 6, pu);
      if (i == 22 && g > 0) h0 = ld(hin);          // group g - 1, for the next interval
      if (i == 23 && g > 0) h1 = ld(hin + 1024);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nb;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the stream runs past its end
  uint16_t* o = xout + (size_t)row * EN_H + 8 * hi;
  const float rstd = en_center(acc, eps);
#pragma unroll
  for (int t = 0; t < EN_T; ++t) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u32x4_t y;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float4 g = four(vec + 3 * EN_H, t, 2 * s + i), b = four(vec + 4 * EN_H, t, 2 * s + i);
        const int at = 8 * s + 4 * i;
        y[2 * i] = pack2bf(fmaf(acc[t][at], rstd * g.x, b.x), fmaf(acc[t][at + 1], rstd * g.y, b.y));
        y[2 * i + 1] = pack2bf(fmaf(acc[t][at + 2], rstd * g.z, b.z), fmaf(acc[t][at + 3], rstd * g.w, b.w));
      }
      if (row < M) *reinterpret_cast<u32x4_t*>(o + 32 * t + 16 * s) = trade(y);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---- y = x W^T + b for a 384-wide x and W of 32 N32 rows (the attention's projections), the same way: rows in registers
// as B operands, W in column groups through a ring of three stages.  No accumulators to hold beside them, so two
// workgroups share a CU and one's waits are the other's matrix time.  65 k rows x 1152 in 78 us, 256 x 256 tiles of
// both operands in LDS took 112; more than 32 k rows now take the kernel after this one.
constexpr int EP_RING = 3, EP_AHEAD = 8;

__global__ void __launch_bounds__(256, 2)
    enc_proj_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ W, const uint16_t* __restrict__ bias,
                    uint16_t* __restrict__ out, int M, int groups) {
  __shared__ __attribute__((aligned(16))) char smem[EP_RING * EN_STAGE];
  const int lane = threadIdx.x & 63, hi = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.x * EN_ROWS + w * 32 + (lane & 31);
  const uint32_t v_n = (lane >> 3) * EN_H * 2 + (((lane & 7) ^ (lane >> 4)) << 4);     // of even pieces
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(en_lds_t*)smem);
  auto issue = [&](int n, uint32_t place) {       // rows 32 n .. of W; past the end, of no use
    const char* src = reinterpret_cast<const char*>(W) + (size_t)min(n, groups - 1) * (32 * EN_H * 2);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int p = 6 * w + i;
      en_glds16(i & 1 ? v_n ^ 64 : v_n, src + (p & 3) * (8 * EN_H * 2) + (p >> 2) * 128, place + p * 1024);
    }
  };
  issue(0, lds0);
  issue(1, lds0 + EN_STAGE);
  bf16x8_t xf[EN_S];
  {
    const uint16_t* xr = x + (size_t)min(row, M - 1) * EN_H + 8 * hi;
#pragma unroll
    for (int s = 0; s < EN_S; ++s) xf[s] = *reinterpret_cast<const bf16x8_t*>(xr + 16 * s);
  }
  const int r32 = lane & 31;
  uint32_t go[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) go[s] = r32 * 128 + (((2 * s + hi) ^ ((r32 >> 1) & 7)) << 4);
  uint16_t* o = out + (size_t)row * 32 * groups + 8 * hi;
  uint32_t here = lds0, before = lds0 + (EP_RING - 1) * EN_STAGE;
  auto four = [&](int n, int i, f32x16_t& a) {
    const uint2 b = *reinterpret_cast<const uint2*>(bias + 32 * n + 8 * i + 4 * hi);
    a[4 * i] = __uint_as_float(b.x << 16); a[4 * i + 1] = __uint_as_float(b.x & 0xffff0000u);
    a[4 * i + 2] = __uint_as_float(b.y << 16); a[4 * i + 3] = __uint_as_float(b.y & 0xffff0000u);
  };
  for (int n = 0; n < groups; ++n) {
    // group n is in LDS in every wave, and group n - 1 read: the one after the next takes its place.  Stores of the
    // group before are younger than its pieces: the count is safe with them.
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue(n + 2, before);
    uint32_t a[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) { a[s] = here + go[s]; asm volatile("" : "+v"(a[s])); }
    auto frag = [&](int i) {
      typedef const __attribute__((address_space(3))) bf16x8_t* lds_frag_t;
      return *reinterpret_cast<lds_frag_t>(a[i & 3] + (uint32_t)((i >> 2) * 4096));
    };
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) four(n, i, acc);
    bf16x8_t fr[EP_AHEAD];
#pragma unroll
    for (int i = 0; i < EP_AHEAD; ++i) fr[i] = frag(i);
#pragma unroll
    for (int i = 0; i < EN_S; ++i) {
      acc = mfma32(fr[i % EP_AHEAD], xf[i], acc);
      if (i + EP_AHEAD < EN_S) fr[i % EP_AHEAD] = frag(i + EP_AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
    const bf16x8_t y0 = frag_of(acc, 0), y1 = frag_of(acc, 1);
    if (row < M) {
      *reinterpret_cast<bf16x8_t*>(o + 32 * n) = y0;
      *reinterpret_cast<bf16x8_t*>(o + 32 * n + 16) = y1;
    }
    before = here;
    here = here == lds0 + (EP_RING - 1) * EN_STAGE ? lds0 : here + EN_STAGE;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the stream runs past its end
}

// The same for more rows than one workgroup of 128 a CU: above, every fragment of W that a wave reads from LDS feeds one
// MFMA, and with two waves a SIMD those reads take all of the LDS's 128 bytes a cycle.  Here a wave holds 64 rows, two MFMAs a
// fragment, one wave a SIMD (260 registers); what it has to wait for is asked for a group ahead: fragments and bias of the
// next group in the last third of this one, after a barrier in its middle that says that the next group is there and the last
// one read; the last group's rows leave while this one is multiplied, two groups at a time by way of the LDS, so that eight
// lanes store a whole line of a row.  The same sums.  us in a forward of 49266 / 65484 rows: workgroups of 128 rows 73 / 78,
// this with 32-byte pieces of rows stored 63 / 69, with whole lines 62.5 / 62.8; without any stores 45 / 55.
constexpr int EW_ROWS = 256, EW_AHEAD = 4, EW_RING = EW_AHEAD + 1, EW_FR = 8, EW_MEET = 12, EW_GROUPS = 3 * EN_T;

__global__ void __launch_bounds__(256, 1)
    enc_proj_wide_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ W, const uint16_t* __restrict__ bias,
                         uint16_t* __restrict__ out, int M) {
  constexpr int groups = EW_GROUPS;
  __shared__ __attribute__((aligned(16))) char smem[EW_RING * EN_STAGE];
  __shared__ __attribute__((aligned(16))) float bias_s[32 * groups];
  __shared__ __attribute__((aligned(16))) char turn[4][64 * 128];      // two groups of a wave's rows, on their way out
  const int lane = threadIdx.x & 63, hi = lane >> 5, r32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = blockIdx.x * EW_ROWS + w * 64 + r32;
  const uint32_t v_n = (lane >> 3) * EN_H * 2 + (((lane & 7) ^ (lane >> 4)) << 4);     // of even pieces
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(en_lds_t*)smem);
  auto issue = [&](int n, int slot) {       // rows 32 n .. of W; past the end, of no use
    const char* src = reinterpret_cast<const char*>(W) + (size_t)min(n, groups - 1) * (32 * EN_H * 2);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int p = 6 * w + i;
      en_glds16(i & 1 ? v_n ^ 64 : v_n, src + (p & 3) * (8 * EN_H * 2) + (p >> 2) * 128, lds0 + slot * EN_STAGE + p * 1024);
    }
  };
#pragma unroll
  for (int n = 0; n < EW_AHEAD; ++n) issue(n, n);
  for (int i = threadIdx.x; i < 32 * groups; i += 256) bias_s[i] = bf2f(bias[i]);
  bf16x8_t xf[2][EN_S];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint16_t* xr = x + (size_t)min(row0 + 32 * t, M - 1) * EN_H + 8 * hi;
#pragma unroll
    for (int s = 0; s < EN_S; ++s) xf[t][s] = *reinterpret_cast<const bf16x8_t*>(xr + 16 * s);
  }
  uint32_t go[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) go[s] = r32 * 128 + (((2 * s + hi) ^ ((r32 >> 1) & 7)) << 4);
  // stores to rows past the last are issued and dropped: the waits below count them
  const int first = blockIdx.x * EW_ROWS;
  const uintptr_t ob = (uintptr_t)(out + (size_t)first * 32 * groups);
  const __amdgpu_buffer_rsrc_t os = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(ob >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)ob)),
      (short)0, min(EW_ROWS, M - first) * 64 * groups, 0x00020000);
  // eight lanes a row: whole lines, in place of 32-byte pieces of them
  const int o = (w * 64 + (lane >> 3)) * 64 * groups + 16 * (lane & 7);
  char* const turn_in = turn[w] + r32 * 128;
  const char* const turn_out = turn[w] + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
  struct At { uint32_t a[4]; };
  auto at_slot = [&](int slot) {
    At r;
#pragma unroll
    for (int s = 0; s < 4; ++s) { r.a[s] = lds0 + slot * EN_STAGE + go[s]; asm volatile("" : "+v"(r.a[s])); }
    return r;
  };
  auto frag = [&](const At& b, int i) {
    typedef const __attribute__((address_space(3))) bf16x8_t* lds_frag_t;
    return *reinterpret_cast<lds_frag_t>(b.a[i & 3] + (uint32_t)((i >> 2) * 4096));
  };
  // the first groups, the rows and the bias are there, in every wave
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  At cur = at_slot(0);
  bf16x8_t fr[EW_FR];
#pragma unroll
  for (int i = 0; i < EW_FR; ++i) fr[i] = frag(cur, i);
  f32x16_t start;                          // a group's bias, what both row tiles' sums start from
  auto biases = [&](int n) {
    const float* b = bias_s + 32 * n + 4 * hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = *reinterpret_cast<const float4*>(b + 8 * i);
      start[4 * i] = v.x; start[4 * i + 1] = v.y; start[4 * i + 2] = v.z; start[4 * i + 3] = v.w;
    }
  };
  biases(0);
  int slot = 0;
  // chunk 4 (n & 1) + 2 s + hi of rows 32 t + r32; chunk c of row r at c ^ (r & 7)
  auto turn_chunk = [&](const f32x16_t& a, int t, int s, int n) {
    *reinterpret_cast<u32x4_t*>(turn_in + t * 32 * 128 + (((4 * (n & 1) + 2 * s + hi) ^ (r32 & 7)) << 4)) = __builtin_bit_cast(u32x4_t, frag_of(a, s));
  };
  auto leave = [&](int k, int n) {          // rows 8 k .. 8 k + 7 of groups n - 1 and n
    __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_t*>(turn_out + k * 1024), os, o + k * 8 * 64 * groups, 64 * (n - 1), 0);
  };
  auto group = [&](int n, f32x16_t (&acc)[2], f32x16_t (&last)[2]) {
    At next = cur;
    const int fill = slot == 0 ? EW_RING - 1 : slot - 1;
    slot = slot + 1 == EW_RING ? 0 : slot + 1;
#pragma unroll
    for (int i = 0; i < EN_S; ++i) {
      if (i == EW_MEET) {
        // group n + 1, asked for three groups ago, is there; every wave is past group n - 1, whose place takes n + 4
        // (younger than its pieces: two groups', and the eight stores of every second group; the first four groups came
        // before the loop)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(6 * (EW_AHEAD - 2) + 8) : "memory");
        issue(n + EW_AHEAD, fill);
        next = at_slot(slot);
      }
      acc[0] = mfma32(fr[i % EW_FR], xf[0][i], i ? acc[0] : start);
      acc[1] = mfma32(fr[i % EW_FR], xf[1][i], i ? acc[1] : start);
      fr[i % EW_FR] = i + EW_FR < EN_S ? frag(cur, i + EW_FR) : frag(next, i + EW_FR - EN_S);
      if (n > 0 && i >= 2 && i < 10 && i % 2 == 0) turn_chunk(last[(i - 2) / 4], (i - 2) / 4, (i - 2) / 2 % 2, n - 1);
      if (n > 0 && n % 2 == 0 && i >= 14 && i < 22) leave(i - 14, n - 1);
      if (i == EN_S - 4) biases(min(n + 1, groups - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = next;
  };
  static_assert(EN_S % EW_FR == 0 && EN_S - EW_FR >= EW_MEET && groups % 2 == 0 && groups > EW_AHEAD);
  f32x16_t a[2], b[2];
  for (int n = 0; n < groups; n += 2) {
    group(n, a, b);
    group(n + 1, b, a);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < 2; ++s) turn_chunk(b[t], t, s, groups - 1);
#pragma unroll
  for (int k = 0; k < 8; ++k) leave(k, groups - 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the stream runs past its end
}

// ================================================================ few rows
// A query or a few texts would leave most CUs idle above, and one CU brings in no more than some 30 bytes a
// nanosecond: a layer's 3.5 MB of weights have to be spread over many.  All four products run in tiles of 16 or 32 rows and
// 64 or 16 columns; what a LayerNorm follows leaves unnormed, and every tile of the next product norms its rows itself
// (a launch less, and rows that few are in every L2).  A launch of so little is one wait for memory after another, so a
// workgroup asks for all that it reads at once: rows in batches took a wait each, and 64 of them to a tile the norms of all of
// them in each of 24 tiles (us of a launch, 73 rows: up product 12.2 -> 4.6, down 11.4 -> 5.1, query, key and value 11.1 -> 4.6;
// six layers of MiniLM, 73 / 150 / 300 rows: 192 / 199 / 206 -> 130 / 134 / 167).

// What the next product reads: x, or LN(proj + bias + res) rounded to bf16, which the first column's tiles also
// store to x for the next residual.
struct EncNorm {
  const uint16_t *proj, *bias, *res, *gamma, *beta;
  float eps;
};

__device__ __forceinline__ float row16_sum(float v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  return v + row_ror<1>(v);
}

// p: LN(v + bias + q) of a row in bf16, sixteen lanes a row, three chunks each
__device__ __forceinline__ void en_norm16(float (&v)[24], uint4 (&p)[3], const uint4 (&q)[3], const uint4 (&bias)[3],
                                          const uint4 (&gamma)[3], const uint4 (&beta)[3], float eps) {
  float s = 0.f, d2 = 0.f;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    float t[8], b[8];
    unpack8(q[j], t);
    unpack8(bias[j], b);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[8 * j + i] = v[8 * j + i] + b[i] + t[i];
      s += v[8 * j + i];
    }
  }
  const float mean = row16_sum(s) * (1.f / EN_H);
#pragma unroll
  for (int i = 0; i < 24; ++i) {
    v[i] -= mean;
    d2 = fmaf(v[i], v[i], d2);
  }
  const float rstd = rsqrtf(row16_sum(d2) * (1.f / EN_H) + eps);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    float ga[8], be[8];
    unpack8(gamma[j], ga);
    unpack8(beta[j], be);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[8 * j + i] = fmaf(v[8 * j + i] * rstd, ga[i], be[i]);
    p[j] = pack8(v + 8 * j);
  }
}

// y = x W^T + b (GELU: x Phi(x) of it) for a 384-wide x and a W of N rows, in tiles of 16 RG rows and 64 columns.  A wave
// owns 16 columns: its fragments of W go straight to registers, all in flight with all of the tile's rows.
template <bool GELU, bool LN, int RG>
__global__ void __launch_bounds__(256) enc_tile_kernel(uint16_t* x, EncNorm ln, const uint16_t* __restrict__ W,
                                                       const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N) {
  constexpr int CH = EN_H / 8, KS = EN_H / 32;    // 16-byte chunks of a row, k steps
  constexpr int B = RG;                           // rows of a lane group: four rows a wave at a time, 16 lanes each
  static_assert(CH == 48);
  __shared__ __attribute__((aligned(16))) char smem[16 * RG * EN_H * 2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  const int n0 = (blockIdx.x * 4 + w) * 16, m0 = blockIdx.y * 16 * RG, rows = min(16 * RG, M - m0);
  uint4 wf[KS], q[B][3];
  u32x4_t p[B][3];      // as uint4 rows that no norm follows went through scratch: 6.7 us of 73 rows, 6.2 of 300, so 4.3 and 4.9
  // row 4 (w + 4 b) + g, its chunks r16 + 16 j
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const size_t at = (size_t)(m0 + min(4 * (w + 4 * b) + g, rows - 1)) * EN_H + 8 * r16;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      p[b][j] = *reinterpret_cast<const u32x4_t*>((LN ? ln.proj : x) + at + 128 * j);
      if constexpr (LN) q[b][j] = *reinterpret_cast<const uint4*>(ln.res + at + 128 * j);
    }
  }
  const uint16_t* wr = W + (size_t)(n0 + r16) * EN_H + 8 * g;
  uint4 vb[3], vg[3], ve[3];
  if constexpr (LN) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      vb[j] = *reinterpret_cast<const uint4*>(ln.bias + 8 * r16 + 128 * j);
      vg[j] = *reinterpret_cast<const uint4*>(ln.gamma + 8 * r16 + 128 * j);
      ve[j] = *reinterpret_cast<const uint4*>(ln.beta + 8 * r16 + 128 * j);
    }
  }
#pragma unroll
  for (int k = 0; k < KS; ++k) wf[k] = *reinterpret_cast<const uint4*>(wr + 32 * k);
  const uint2 bb = *reinterpret_cast<const uint2*>(bias + n0 + 4 * g);
  __builtin_amdgcn_sched_barrier(0);
  // chunk c of row r at slot c ^ (r & 7): 16-row fragment reads without bank conflicts
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int r = 4 * (w + 4 * b) + g;
    if constexpr (LN) {
      float v[24];
#pragma unroll
      for (int j = 0; j < 3; ++j) unpack8(__builtin_bit_cast(uint4, p[b][j]), v + 8 * j);
      uint4 y[3];
      en_norm16(v, y, q[b], vb, vg, ve, ln.eps);
#pragma unroll
      for (int j = 0; j < 3; ++j) p[b][j] = __builtin_bit_cast(u32x4_t, y[j]);
      if (blockIdx.x == 0 && r < rows)
#pragma unroll
        for (int j = 0; j < 3; ++j) *reinterpret_cast<u32x4_t*>(x + (size_t)(m0 + r) * EN_H + 8 * r16 + 128 * j) = p[b][j];
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) *reinterpret_cast<u32x4_t*>(smem + r * (EN_H * 2) + (((r16 + 16 * j) ^ (r & 7)) << 4)) = p[b][j];
  }
  __syncthreads();
  const float b[4] = {__uint_as_float(bb.x << 16), __uint_as_float(bb.x & 0xffff0000u), __uint_as_float(bb.y << 16),
                      __uint_as_float(bb.y & 0xffff0000u)};
  f32x4_t acc[RG];
#pragma unroll
  for (int i = 0; i < RG; ++i) acc[i] = f32x4_t{b[0], b[1], b[2], b[3]};
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int i = 0; i < RG; ++i) {                // rows past `rows` repeat the last one and are not stored
      const uint4 xv = *reinterpret_cast<const uint4*>(smem + (16 * i + r16) * (EN_H * 2) + (((4 * k + g) ^ (r16 & 7)) << 4));
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[k]), __builtin_bit_cast(bf16x8_t, xv), acc[i], 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < RG; ++i) {
    if constexpr (GELU) {
      en_gelus(acc[i]);
    }
    if (16 * i + r16 < rows)
      *reinterpret_cast<uint2*>(out + (size_t)(m0 + 16 * i + r16) * N + n0 + 4 * g) = make_uint2(pack2bf(acc[i][0], acc[i][1]), pack2bf(acc[i][2], acc[i][3]));
  }
}

// y = x W^T for a K-wide x and a W of 384 rows, rounded to bf16: 16 RG rows x 16 columns a workgroup, a quarter of K per wave
// with W's and the rows' fragments straight from memory, all in flight at once, the quarters summed through LDS.
template <int K, int RG>
__global__ void __launch_bounds__(256) enc_ksplit_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ W,
                                                         uint16_t* __restrict__ out, int M) {
  constexpr int KS = K / 128;                     // k steps of a wave
  __shared__ float part[4][RG][64][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * RG, rows = min(16 * RG, M - m0);
  const int k0 = w * (K / 4) + 8 * g;
  uint4 wf[KS], xv[RG][KS];
#pragma unroll
  for (int i = 0; i < RG; ++i)
#pragma unroll
    for (int k = 0; k < KS; ++k) xv[i][k] = *reinterpret_cast<const uint4*>(x + (size_t)(m0 + min(16 * i + r16, rows - 1)) * K + k0 + 32 * k);
#pragma unroll
  for (int k = 0; k < KS; ++k) wf[k] = *reinterpret_cast<const uint4*>(W + (size_t)(n0 + r16) * K + k0 + 32 * k);
  __builtin_amdgcn_sched_barrier(0);
  f32x4_t acc[RG];
#pragma unroll
  for (int i = 0; i < RG; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int i = 0; i < RG; ++i)
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[k]), __builtin_bit_cast(bf16x8_t, xv[i][k]), acc[i], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < RG; ++i) *reinterpret_cast<f32x4_t*>(part[w][i][lane]) = acc[i];
  __syncthreads();
  // wave q takes the sums of row group q
  if (w >= RG) return;
  f32x4_t s = *reinterpret_cast<const f32x4_t*>(part[0][w][lane]);
#pragma unroll
  for (int q = 1; q < 4; ++q) s += *reinterpret_cast<const f32x4_t*>(part[q][w][lane]);
  if (16 * w + r16 < rows)
    *reinterpret_cast<uint2*>(out + (size_t)(m0 + 16 * w + r16) * EN_H + n0 + 4 * g) = make_uint2(pack2bf(s[0], s[1]), pack2bf(s[2], s[3]));
}

// x = LN(proj + bias + res) of 32-bit projections, sixteen lanes a row (a wave a row took 5.5 and 8.7 us of 4823 and 12184 rows of
// 16-bit ones where this takes 4.4 and 7.4).
__global__ void __launch_bounds__(256) enc_norm_kernel(uint16_t* __restrict__ x, const float* __restrict__ proj, EncNorm ln, int M) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  const int r = xcd_remap(blockIdx.x, gridDim.x) * 16 + 4 * w + g;      // the XCD that has them from the product
  const size_t at = (size_t)min(r, M - 1) * EN_H + 8 * r16;
  float4 f[3][2];
  uint4 p[3], q[3], vb[3], vg[3], ve[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    f[j][0] = *reinterpret_cast<const float4*>(proj + at + 128 * j);
    f[j][1] = *reinterpret_cast<const float4*>(proj + at + 128 * j + 4);
    q[j] = *reinterpret_cast<const uint4*>(ln.res + at + 128 * j);
    vb[j] = *reinterpret_cast<const uint4*>(ln.bias + 8 * r16 + 128 * j);
    vg[j] = *reinterpret_cast<const uint4*>(ln.gamma + 8 * r16 + 128 * j);
    ve[j] = *reinterpret_cast<const uint4*>(ln.beta + 8 * r16 + 128 * j);
  }
  float v[24];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v[8 * j + 4 * i] = f[j][i].x; v[8 * j + 4 * i + 1] = f[j][i].y;
      v[8 * j + 4 * i + 2] = f[j][i].z; v[8 * j + 4 * i + 3] = f[j][i].w;
    }
  en_norm16(v, p, q, vb, vg, ve, ln.eps);
  if (r < M)
#pragma unroll
    for (int j = 0; j < 3; ++j) *reinterpret_cast<uint4*>(x + at + 128 * j) = p[j];
}

// ================================================================ between few and many rows
// From some 300 rows on a tile's norms, made again for each column of tiles, cost more than a launch of their own, and fragments
// straight from memory bring each row into a CU once per 16 columns (2201 rows: up product 26.9 us, down 30); up to 16 k rows
// the kernels of 128 rows a workgroup leave CUs without one and the 256-row tiles of the general products leave most.
// y = x W^T (32-bit: LayerNorm reads it as the matrix cores left it), or x W^T + b, or GELU of that (bf16), in tiles of BM rows
// and BN columns, both through a ring of NS LDS-DMA stages 64 deep; a wave takes 32 TM rows and 32 TN columns.  K is 6 or 24
// stages, so a tile is mostly start and end: two or three workgroups a CU cover one another's.  An XCD takes neighbouring rows in
// every launch of a layer, which then are in its L2 (six layers of 4823 / 12184 rows 386 / 748 -> 342 / 676 us).
// Six layers of MiniLM before and now: 481 rows 216 -> 187 us, 1218 323 -> 208, 2201 502 -> 239, 4823 721 -> 342, 8000 745 -> 481,
// 12184 815 -> 669, 16000 838 -> 767.  What bounds it: launches of 3 to 5 us up to 1000 rows; then the LDS, which every MFMA
// takes 1 to 1.5 KB from, and the GELU (8000 rows: up 19.9 us = 470 TFLOP/s, down 16.0).
enum { EG_RAW = 0, EG_BIAS = 1, EG_GELU = 2 };
template <int K, int BM, int BN, int TM, int TN, int NS, int EPI>
__global__ void __launch_bounds__((BM / 32 / TM) * (BN / 32 / TN) * 64)
    enc_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ W, const uint16_t* __restrict__ bias,
                    void* __restrict__ out, int M, int N) {
  constexpr int WM = BM / 32 / TM, NW = WM * (BN / 32 / TN), S = K / 64, PIECES = (BM + BN) / 8, PW = PIECES / NW, STAGE = (BM + BN) * 128;
  static_assert(PIECES % NW == 0 && S >= NS);
  extern __shared__ __attribute__((aligned(16))) char eg_smem[];
  const int lane = threadIdx.x & 63, hi = lane >> 5, r32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // an XCD takes neighbouring rows, all columns of them
  const int cols = N / BN, tile = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = tile / cols * BM, n0 = tile % cols * BN;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(en_lds_t*)eg_smem);
  // piece p: rows 8 p .. 8 p + 7 of the tile's BM rows of x, then of its BN rows of W; chunk c of row r at c ^ (r >> 1 & 7)
  uint32_t voff[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int p = PW * w + i, r = 8 * p + (lane >> 3);
    const int row = p < BM / 8 ? min(m0 + r, M - 1) : n0 + r - BM;
    voff[i] = (uint32_t)row * (K * 2) + (((lane & 7) ^ (r >> 1 & 7)) << 4);
  }
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int p = PW * w + i;
      en_glds16(voff[i], reinterpret_cast<const char*>(p < BM / 8 ? x : W) + st * 128, lds0 + slot * STAGE + p * 1024);
    }
  };
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) issue(st, st);
  const int wm = w % WM, wn = w / WM;
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    f32x16_t a;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint2 v = make_uint2(0, 0);
      if constexpr (EPI != EG_RAW) v = *reinterpret_cast<const uint2*>(bias + n0 + 32 * (wn * TN + b) + 8 * i + 4 * hi);
      a[4 * i] = __uint_as_float(v.x << 16); a[4 * i + 1] = __uint_as_float(v.x & 0xffff0000u);
      a[4 * i + 2] = __uint_as_float(v.y << 16); a[4 * i + 3] = __uint_as_float(v.y & 0xffff0000u);
    }
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[t][b] = a;
  }
  uint32_t go[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) go[s] = r32 * 128 + (((2 * s + hi) ^ (r32 >> 1 & 7)) << 4);
  typedef const __attribute__((address_space(3))) bf16x8_t* lds_frag_t;
#pragma unroll
  for (int st = 0; st < S; ++st) {
    constexpr int AHEAD = NS - 2;
    // stage st is there in every wave, and stage st - 1 read (the bias was asked for later than the first stages: counted safe)
    const int left = S - 1 - st < AHEAD ? S - 1 - st : AHEAD;
    if (left == 0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(PW) : "memory");
    else if (left == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(2 * PW) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(3 * PW) : "memory");
    if (st + NS - 1 < S) issue(st + NS - 1, (st + NS - 1) % NS);
    const uint32_t base = lds0 + (st % NS) * STAGE;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8_t fx[TM], fw[TN];
#pragma unroll
      for (int t = 0; t < TM; ++t) fx[t] = *reinterpret_cast<lds_frag_t>(base + (wm * TM + t) * 4096 + go[s]);
#pragma unroll
      for (int b = 0; b < TN; ++b) fw[b] = *reinterpret_cast<lds_frag_t>(base + BM * 128 + (wn * TN + b) * 4096 + go[s]);
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[t][b] = mfma32(fw[b], fx[t], acc[t][b]);
    }
  }
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int row = m0 + 32 * (wm * TM + t) + r32;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      f32x16_t a = acc[t][b];
      if constexpr (EPI == EG_GELU) {
        en_gelus(a);
      }
      const int n = n0 + 32 * (wn * TN + b);
      if constexpr (EPI == EG_RAW) {
        if (row < M)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4*>((float*)out + (size_t)row * N + n + 8 * i + 4 * hi) = make_float4(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]);
      } else {
        const bf16x8_t y0 = frag_of(a, 0), y1 = frag_of(a, 1);
        if (row < M) {
          uint16_t* o = (uint16_t*)out + (size_t)row * N + n + 8 * hi;
          *reinterpret_cast<bf16x8_t*>(o) = y0;
          *reinterpret_cast<bf16x8_t*>(o + 16) = y1;
        }
      }
    }
  }
}

// ================================================================ a query or a few short texts
// Up to 64 tokens, all layers in one launch: five launches a layer, each waiting for the one before, take 17 to 20 us (small tiles; 27
// when this kernel was written) of which the work itself is 3.  60 workgroups of three kinds: one per head takes the layer's q, k, v and attention of its head,
// 24 take 16 columns each of the output projection and of the down product, 24 take 64 columns of the up product.
// Those that need normed rows norm all of them and keep them in registers, so nothing but products passes between
// workgroups: attention, o, hidden rows and down, four hand-overs a layer.  Each goes through a place of its own per layer
// that is filled with ~0 before the launch.  A word of two bf16 that is not ~0 is there, so a reader polls the data itself:
// one store and one load across the chip, no barrier and no flag.  Both are past the XCDs' own L2 (agent scope).
// Weights come a layer ahead of their use, straight to the registers they are used from; a CU brings in some 25 B/ns, so
// they are spread (a quarter of the workgroups took 94 us where these take 80), and are asked for only when nothing is
// waited for, as loads return in order (104 -> 94 us).
// MiniLM's six layers in small tiles and in this, us of a captured forward: 1 token 100 and 69, 12 108 and 81, 16 113 and 84, 24 114 and 113,
// 32 115 and 119, 33 118 and 162, 64 122 and 179 (136, 188 and 295 of 12, 32 and 64 in the tiles of its day): from some 30 rows on
// small tiles are the faster ones now, though their sums come in another order.  A layer's 12 us are
// its four hand-overs of 2 to 2.5 us (a store and a poll of about 1 us each), two norms and the products between.
//
// The workgroups wait for one another, so all have to be resident, and nothing can promise that: launches of other streams
// and processes may hold the CUs that some of them need, and wait for others of their own.  So a wait is bounded: a wave that
// has polled `polls` times takes what is there and says so in the workspace's last word, which ends all waits for it, and
// a launch of one workgroup behind this one, which waits for nothing, looks at that word and takes all layers by itself,
// the same products in the same order: the same bits, in 1.5 ms of 12 tokens and 2.5 of 64 (6 layers).  Where no wait was
// given up it is over in 2 us, so a call of 12 tokens takes 85.6 us, 83.7 without it.
constexpr int EN_TINY_ROWS = 64, EN_TINY_LAYERS = 24, EN_POLLS = 1 << 14;
constexpr uint32_t EN_EMPTY = ~0u;
constexpr int EN_HEADS = EN_H / 32, EN_BLOCKS = EN_H / 16, EN_INNER = EN_F / 64;      // workgroups of each kind

struct EncTiny {
  const uint16_t *word, *pos, *type, *g, *b;
  const uint16_t* layer[EN_TINY_LAYERS][12];
};

__global__ void __launch_bounds__(256) enc_empty_kernel(uint4* __restrict__ p, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = make_uint4(EN_EMPTY, EN_EMPTY, EN_EMPTY, EN_EMPTY);
}

// Sixteen bytes at every off + 64 s, once none of their words is empty (the words are looked at one by one: a load need be
// no more than them in one piece).  With pauses and at low priority: loads go out oldest wave first, and waves that poll
// without a pause keep a younger one of their CU from ever storing what they wait for.
struct EncWait {
  int polls;              // left
  uint32_t* late;         // empty, until a wave gave up
};
template <int N, int S>
__device__ __forceinline__ void en_take(const uint16_t* base, int bytes, const uint32_t (&off)[N], uint4 (&v)[N][S], EncWait& wait) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, bytes, 0x00020000);
  __builtin_amdgcn_s_setprio(0);
  for (;;) {
    bool all = true;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int s = 0; s < S; ++s)                 // 16: sc1, past what this XCD's L2 holds
        v[i][s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[i] + 64 * s, 0, 16));
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int s = 0; s < S; ++s) all &= v[i][s].x != EN_EMPTY && v[i][s].y != EN_EMPTY && v[i][s].z != EN_EMPTY && v[i][s].w != EN_EMPTY;
    if (__all(all)) break;
    if (wait.polls <= 0) {
      __hip_atomic_store(wait.late, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    --wait.polls;
    __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");                // loaded again
  }
  __builtin_amdgcn_s_setprio(1);
}

// Four bf16 for the others: no word of them is the empty one (a pair of NaN of another payload instead).
__device__ __forceinline__ void en_give(uint16_t* p, const f32x4_t& v) {
  const uint64_t a = min(pack2bf(v[0], v[1]), EN_EMPTY - 1), b = min(pack2bf(v[2], v[3]), EN_EMPTY - 1);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), a | b << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t four_bf(uint2 b) {
  return f32x4_t{__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xffff0000u), __uint_as_float(b.y << 16), __uint_as_float(b.y & 0xffff0000u)};
}

// Whether either bf16 of the word is no finite number.
__device__ __forceinline__ bool infinite(uint32_t v) { return (v & 0x7f80u) == 0x7f80u || (v & 0x7f800000u) == 0x7f800000u; }

// G groups of 16 rows, T of them rows; grid EN_HEADS + EN_BLOCKS + EN_INNER.  ALONE: one workgroup, which does all in turn
// if a wait of the launch before it was given up.
template <int G, bool ALONE>
__global__ void __launch_bounds__(512, 2)
    enc_tiny_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ pos, EncTiny W, const int32_t* __restrict__ cu,
                    const int32_t* __restrict__ tile_seq, int n_tiles, int layers, uint16_t* buf, uint16_t* __restrict__ out, int T,
                    float scale_log2, float eps, int polls) {
  constexpr int U = 2 * G, V = U < 4 ? U : 4, ROW = EN_H * 2;     // rows of a wave (w, w + 8, ..), at a time; bytes of a row
  extern __shared__ __attribute__((aligned(16))) char en_smem[];
  char* rows = en_smem;                           // [16 G][384], chunk c of row r at slot c ^ (r & 15)
  char* rest = en_smem + 16 * G * ROW;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const bool on = lane < EN_H / 8;                // a row's chunks
  const int c = on ? lane : 0;
  const size_t place = (size_t)T * (3 * EN_H + EN_F);
  EncWait wait = {polls, reinterpret_cast<uint32_t*>(buf + layers * place)};
  if (ALONE && *wait.late == EN_EMPTY) return;
  __builtin_amdgcn_s_setprio(1);
  uint4 x[U];                                     // this wave's rows of the layer's input, then of what lies between its sublayers

  auto put = [&]() {                              // to where the products read them
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = w + 8 * u;
      if (on && r < T) *reinterpret_cast<uint4*>(rows + r * ROW + ((c ^ (r & 15)) << 4)) = x[u];
    }
  };
  auto frag = [&](int i, int k) { return *reinterpret_cast<const uint4*>(rows + (16 * i + r16) * ROW + (((4 * k + g) ^ r16) << 4)); };
  // x[u0 ..] = LN(v) gamma + beta
  auto norm = [&](int u0, float (&v)[V][8], uint4 gamma, uint4 beta) {
    float ga[8], be[8], s[V], q[V];
    unpack8(gamma, ga);
    unpack8(beta, be);
#pragma unroll
    for (int u = 0; u < V; ++u) {
      s[u] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[u][j] = on ? v[u][j] : 0.f;
        s[u] += v[u][j];
      }
    }
#pragma unroll
    for (int u = 0; u < V; ++u) s[u] = wave_sum(s[u]) * (1.f / EN_H);
#pragma unroll
    for (int u = 0; u < V; ++u) {
      q[u] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[u][j] -= s[u];
        q[u] += on ? v[u][j] * v[u][j] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < V; ++u) q[u] = rsqrtf(wave_sum(q[u]) * (1.f / EN_H) + eps);
#pragma unroll
    for (int u = 0; u < V; ++u) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[u][j] = v[u][j] * q[u] * ga[j] + be[j];
      x[u0 + u] = pack8(v[u]);
    }
  };
  // x = LN(y + bias + x) gamma + beta of a finished product's rows y
  auto next = [&](const uint16_t* y, const uint16_t* bias, const uint16_t* gamma, const uint16_t* beta) {
    const uint4 pb = *reinterpret_cast<const uint4*>(bias + 8 * c), ga = *reinterpret_cast<const uint4*>(gamma + 8 * c),
                be = *reinterpret_cast<const uint4*>(beta + 8 * c);
    uint32_t at[U];
    uint4 t[U][1];
#pragma unroll
    for (int u = 0; u < U; ++u) at[u] = min(w + 8 * u, T - 1) * ROW + 16 * c;
    en_take(y, T * ROW, at, t, wait);
    float b[8];
    unpack8(pb, b);
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += V) {
      float v[V][8];
#pragma unroll
      for (int u = 0; u < V; ++u) {
        float r[8];
        unpack8(t[u0 + u][0], v[u]);
        unpack8(x[u0 + u], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[u][j] += b[j] + r[j];
      }
      norm(u0, v, ga, be);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  {                                               // embeddings; rows past T stay zeros
    for (int i = threadIdx.x; i < G * ROW; i += 512) *reinterpret_cast<uint4*>(rows + 16 * i) = make_uint4(0, 0, 0, 0);
    const uint4 ga = *reinterpret_cast<const uint4*>(W.g + 8 * c), be = *reinterpret_cast<const uint4*>(W.b + 8 * c);
    float t[8];
    unpack8(*reinterpret_cast<const uint4*>(W.type + 8 * c), t);
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += V) {
      float v[V][8];
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int r = min(w + 8 * (u0 + u), T - 1);
        float p[8];
        unpack8(*reinterpret_cast<const uint4*>(W.word + (size_t)ids[r] * EN_H + 8 * c), v[u]);
        unpack8(*reinterpret_cast<const uint4*>(W.pos + (size_t)pos[r] * EN_H + 8 * c), p);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[u][j] += p[j] + t[j];
      }
      norm(u0, v, ga, be);
    }
    __syncthreads();
  }

  // ---- a head: waves 0 .. 5 take 16 of q's, k's and v's 32 columns each, waves 0 .. G - 1 a group of queries
  constexpr int QS = 80, VS = 32 * ((G + 1) / 2) + 8;      // row strides: bytes of q and k, values of V^T
  char *q = rest, *k = q + 16 * G * QS;
  uint16_t* vt = reinterpret_cast<uint16_t*>(k + 16 * G * QS);
  int *from = reinterpret_cast<int*>(vt + 32 * VS), *to = from + 16 * G, *odd = to + 16 * G;
  auto texts = [&]() {                            // which keys a row sees; V^T past the rows: zeros
    if (threadIdx.x == 0) *odd = 0;
    for (int i = threadIdx.x; i < 32 * VS; i += 512) vt[i] = 0;
    for (int i = threadIdx.x; i < 16 * G; i += 512) from[i] = i, to[i] = i + 1;
    __syncthreads();
    for (int i = threadIdx.x; i < n_tiles; i += 512) {
      const int a = cu[tile_seq[i]], b = min(cu[tile_seq[i] + 1], T);
      for (int t = max(a, 0); t < b; ++t) from[t] = a, to[t] = b;
    }
  };
  uint4 wf[12];
  uint2 bb;
  auto load_head = [&](int l, int head) {
    if (w >= 6) return;
    const int n0 = (w >> 1) * EN_H + head * 32 + (w & 1) * 16;
    const uint16_t* p = W.layer[l][0] + (size_t)(n0 + r16) * EN_H + 8 * g;
#pragma unroll
    for (int s = 0; s < 12; ++s) wf[s] = *reinterpret_cast<const uint4*>(p + 32 * s);
    bb = *reinterpret_cast<const uint2*>(W.layer[l][1] + n0 + 4 * g);
  };
  auto attend = [&](int head, uint16_t* att) {
    if (w < 6) {
      f32x4_t a[G];
#pragma unroll
      for (int i = 0; i < G; ++i) a[i] = four_bf(bb);
#pragma unroll
      for (int s = 0; s < 12; ++s)
#pragma unroll
        for (int i = 0; i < G; ++i) a[i] = mfma16(wf[s], frag(i, s), a[i]);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int t = 16 * i + r16;
        const uint2 y = make_uint2(pack2bf(a[i][0], a[i][1]), pack2bf(a[i][2], a[i][3]));
        if (w < 4) {
          *reinterpret_cast<uint2*>((w < 2 ? q : k) + t * QS + 32 * (w & 1) + 8 * g) = y;
        } else {
          uint16_t* v = vt + (16 * (w & 1) + 4 * g) * VS + t;
          v[0] = (uint16_t)y.x; v[VS] = (uint16_t)(y.x >> 16); v[2 * VS] = (uint16_t)y.y; v[3 * VS] = (uint16_t)(y.y >> 16);
          if (infinite(y.x) || infinite(y.y)) *odd = 1;
        }
      }
    }
    __syncthreads();
    if (w >= G) return;
    // scores with the keys along a lane's registers: key 16 i + 4 g + e of query 16 w + r16
    const uint4 qf = *reinterpret_cast<const uint4*>(q + (16 * w + r16) * QS + 16 * g);
    const int t = 16 * w + r16, a = from[t], b = to[t];
    f32x4_t s[2 * ((G + 1) / 2)];
    float m = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * ((G + 1) / 2); ++i) {
      s[i] = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (i >= G) continue;
      const f32x4_t z = mfma16(*reinterpret_cast<const uint4*>(k + (16 * i + r16) * QS + 16 * g), qf, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * i + 4 * g + e;
        s[i][e] = j >= a && j < b ? z[e] * scale_log2 : -INFINITY;
        m = fmaxf(m, s[i][e]);
      }
    }
    m = xor32_max(xor16_max(m));
    const float ref = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int i = 0; i < 2 * ((G + 1) / 2); ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[i][e] = __builtin_amdgcn_exp2f(s[i][e] - ref);
        sum += s[i][e];
      }
    sum = xor32_sum(xor16_sum(sum));
    f32x4_t o[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
    uint4 p[(G + 1) / 2];                         // 32 keys each, in the order that the scores have them
#pragma unroll
    for (int i = 0; i < (G + 1) / 2; ++i)
      p[i] = make_uint4(pack2bf(s[2 * i][0], s[2 * i][1]), pack2bf(s[2 * i][2], s[2 * i][3]), pack2bf(s[2 * i + 1][0], s[2 * i + 1][1]),
                        pack2bf(s[2 * i + 1][2], s[2 * i + 1][3]));
    auto values = [&](int i, int d) {
      const uint16_t* v = vt + (16 * d + r16) * VS + 32 * i + 4 * g;
      const uint2 lo = *reinterpret_cast<const uint2*>(v), hi = *reinterpret_cast<const uint2*>(v + 16);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    if (__builtin_amdgcn_readfirstlane(*odd) == 0) {
#pragma unroll
      for (int i = 0; i < (G + 1) / 2; ++i)
#pragma unroll
        for (int d = 0; d < 2; ++d) o[d] = mfma16(values(i, d), p[i], o[d]);
    } else {
      // Zero weights of other texts' keys do not take their infinite values out: text after text, its keys' values alone.
      for (int j = 0; j < T;) {
        const int a0 = from[j], b0 = to[j];
        j = max(b0, j + 1);
        if (!__any(a == a0)) continue;
        f32x4_t z[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < (G + 1) / 2; ++i) {
          auto keep = [&](int at) {               // of keys at and at + 1
            const int key = 32 * i + 4 * g + at;
            return (key >= a0 && key < b0 ? 0xffffu : 0u) | (key + 1 >= a0 && key + 1 < b0 ? 0xffff0000u : 0u);
          };
          const uint4 m = make_uint4(keep(0), keep(2), keep(16), keep(18));
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            const uint4 v = values(i, d);
            z[d] = mfma16(make_uint4(v.x & m.x, v.y & m.y, v.z & m.z, v.w & m.w), p[i], z[d]);
          }
        }
        if (a == a0) o[0] = z[0], o[1] = z[1];
      }
    }
    const float inv = 1.f / sum;
#pragma unroll
    for (int d = 0; d < 2; ++d)
      if (t < T) en_give(att + (size_t)t * EN_H + head * 32 + 16 * d + 4 * g, o[d] * inv);
  };

  // ---- 64 inner columns: 16 per wave of a group of rows
  auto load_up = [&](int l, int block) {
    const int n0 = block * 64 + 16 * (w & 3);
    const uint16_t* p = W.layer[l][6] + (size_t)(n0 + r16) * EN_H + 8 * g;
#pragma unroll
    for (int s = 0; s < 12; ++s) wf[s] = *reinterpret_cast<const uint4*>(p + 32 * s);
    bb = *reinterpret_cast<const uint2*>(W.layer[l][7] + n0 + 4 * g);
  };
  auto up = [&](int block, uint16_t* h) {
    const int n0 = block * 64 + 16 * (w & 3);
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if ((i & 1) != w >> 2) continue;
      f32x4_t a = four_bf(bb);
#pragma unroll
      for (int s = 0; s < 12; ++s) a = mfma16(wf[s], frag(i, s), a);
      Gelu ge;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = a[e];
        en_gelu<0>(ge, v);
        en_gelu<1>(ge, v);
        en_gelu<2>(ge, v);
        a[e] = v;
      }
      if (16 * i + r16 < T) en_give(h + (size_t)(16 * i + r16) * EN_F + n0 + 4 * g, a);
    }
  };

  // ---- 16 columns of o (waves 4 .. 7, a quarter of K each) and of down (an eighth of K per wave)
  f32x4_t *po = reinterpret_cast<f32x4_t*>(rest), *pd = po + 4 * G * 64;        // parts of sums [4][G][64], [8][G][64]
  uint4 wo[3], wd[6];
  auto load_block = [&](int l, int block) {
    const int n0 = block * 16;
    const uint16_t *p = W.layer[l][2] + (size_t)(n0 + r16) * EN_H + 96 * (w & 3) + 8 * g, *q = W.layer[l][8] + (size_t)(n0 + r16) * EN_F + 192 * w + 8 * g;
#pragma unroll
    for (int s = 0; s < 3; ++s) wo[s] = *reinterpret_cast<const uint4*>(p + 32 * s);
#pragma unroll
    for (int s = 0; s < 6; ++s) wd[s] = *reinterpret_cast<const uint4*>(q + 32 * s);
  };
  auto project = [&](int block, const uint16_t* att, uint16_t* y1) {
    if (w >= 4) {
      uint32_t at[G];
      uint4 v[G][3];
#pragma unroll
      for (int i = 0; i < G; ++i) at[i] = min(16 * i + r16, T - 1) * ROW + 192 * (w & 3) + 16 * g;
      en_take(att, T * ROW, at, v, wait);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 3; ++s) a = mfma16(wo[s], v[i][s], a);
        po[((w & 3) * G + i) * 64 + lane] = a;
      }
    }
    __syncthreads();
    if (w >= 4 && w - 4 < G) {
      const int i = w - 4, t = 16 * i + r16;
      f32x4_t a = po[i * 64 + lane];
#pragma unroll
      for (int s = 1; s < 4; ++s) a += po[(s * G + i) * 64 + lane];
      if (t < T) en_give(y1 + (size_t)t * EN_H + block * 16 + 4 * g, a);
    }
  };
  auto down = [&](int block, const uint16_t* h, uint16_t* y2) {
#pragma unroll
    for (int i0 = 0; i0 < G; i0 += 2) {
      constexpr int N = G < 2 ? G : 2;            // at a time: registers
      uint32_t at[N];
      uint4 v[N][6];
#pragma unroll
      for (int i = 0; i < N; ++i) at[i] = min(16 * (i0 + i) + r16, T - 1) * (2 * EN_F) + 384 * w + 16 * g;
      en_take(h, T * 2 * EN_F, at, v, wait);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 6; ++s) a = mfma16(wd[s], v[i][s], a);
        pd[(w * G + i0 + i) * 64 + lane] = a;
      }
    }
    __syncthreads();
    if (w < G) {
      const int t = 16 * w + r16;
      f32x4_t a = pd[w * 64 + lane];
#pragma unroll
      for (int s = 1; s < 8; ++s) a += pd[(s * G + w) * 64 + lane];
      if (t < T) en_give(y2 + (size_t)t * EN_H + block * 16 + 4 * g, a);
    }
  };

  if constexpr (ALONE) {
    // what one product left is there for the next one: stored, and all waves past it
    auto settle = [&]() {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    };
    put();
    for (int l = 0; l < layers; ++l) {
      uint16_t *att = buf + l * place, *y1 = att + (size_t)T * EN_H, *h = y1 + (size_t)T * EN_H, *y2 = h + (size_t)T * EN_F;
      texts();                                    // again: the parts of sums lay there
      for (int head = 0; head < EN_HEADS; ++head) {
        load_head(l, head);
        settle();
        attend(head, att);
      }
      settle();
      for (int block = 0; block < EN_BLOCKS; ++block) {
        load_block(l, block);
        project(block, att, y1);
        settle();
      }
      next(y1, W.layer[l][3], W.layer[l][4], W.layer[l][5]);
      put();
      settle();
      for (int block = 0; block < EN_INNER; ++block) {
        load_up(l, block);
        up(block, h);
      }
      settle();
      for (int block = 0; block < EN_BLOCKS; ++block) {
        load_block(l, block);
        down(block, h, y2);
        settle();
      }
      next(y2, W.layer[l][9], W.layer[l][10], W.layer[l][11]);
      put();
      settle();
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (on && w + 8 * u < T) *reinterpret_cast<uint4*>(out + (size_t)(w + 8 * u) * EN_H + 8 * c) = x[u];
    return;
  }

  if (blockIdx.x < EN_HEADS) {
    const int head = blockIdx.x;
    texts();
    load_head(0, head);
    put();
    for (int l = 0; l < layers; ++l) {
      uint16_t *att = buf + l * place, *y1 = att + (size_t)T * EN_H, *y2 = y1 + (size_t)T * (EN_H + EN_F);
      __syncthreads();                            // the rows are there
      attend(head, att);
      if (l + 1 < layers) load_head(l + 1, head); // loads return in order: ahead of nothing that is waited for
      next(y1, W.layer[l][3], W.layer[l][4], W.layer[l][5]);
      next(y2, W.layer[l][9], W.layer[l][10], W.layer[l][11]);
      put();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = w + 8 * u;
      if (on && r < T && r % EN_HEADS == head) *reinterpret_cast<uint4*>(out + (size_t)r * EN_H + 8 * c) = x[u];
    }
    return;
  }

  if (blockIdx.x >= EN_HEADS + EN_BLOCKS) {
    const int block = blockIdx.x - EN_HEADS - EN_BLOCKS;
    load_up(0, block);
    for (int l = 0; l < layers; ++l) {
      const uint16_t* y1 = buf + l * place + (size_t)T * EN_H;
      uint16_t* h = buf + l * place + (size_t)T * 2 * EN_H;
      next(y1, W.layer[l][3], W.layer[l][4], W.layer[l][5]);
      put();                                      // the rows before were read: these came of what was made of them
      __syncthreads();
      up(block, h);
      if (l + 1 < layers) {
        load_up(l + 1, block);                    // loads return in order: ahead of nothing that is waited for
        next(h + (size_t)T * EN_F, W.layer[l][9], W.layer[l][10], W.layer[l][11]);
      }
    }
    return;
  }

  const int block = blockIdx.x - EN_HEADS;
  load_block(0, block);
  for (int l = 0; l < layers; ++l) {
    uint16_t *att = buf + l * place, *y1 = att + (size_t)T * EN_H, *h = y1 + (size_t)T * EN_H, *y2 = h + (size_t)T * EN_F;
    project(block, att, y1);
    down(block, h, y2);
    if (l + 1 < layers) load_block(l + 1, block);
  }
}

// Bytes of LDS: the rows, and the larger of what either kind keeps beside them.
constexpr int en_tiny_lds(int G) { return 16 * G * EN_H * 2 + 12 * G * 1024; }
static_assert(2 * 16 * 1 * 80 + 32 * 40 * 2 + 2 * 16 * 4 + 4 <= 12 * 1024 && 2 * 64 * 80 + 32 * 72 * 2 + 2 * 64 * 4 + 4 <= 48 * 1024, "");

}  // namespace

CFC_API int cfc_layernorm(void* out, const void* x, const void* bias, const void* residual, const void* gamma, const void* beta,
                          const int32_t* ids, const int32_t* pos, const void* pos_emb, const void* type_emb, int rows, int dim,
                          float eps, int mode, hipStream_t stream);
CFC_API int cfc_encoder_attention(const void* qkv, const int32_t* cu_seqlens, const int32_t* tile_seq, const int32_t* tile_q0,
                                  int n_tiles, int tile_rows, int H, int head_dim, int max_seqlen, float scale, void* out,
                                  hipStream_t stream);

// A few texts of 64 rows in all: enc_tiny_kernel.  More take small tiles up to 320 rows, LDS tiles up to 16383 and the layer's one
// kernel above from there on (six layers of MiniLM in LDS tiles and in it: 14000 rows 712 and 826 us, 16000 767 and 838, 18000 845
// and 848).
constexpr int EN_FUSED_ROWS = 16384;

// Whether T rows are as many as the layer's one kernel takes, which needs no y and h.
CFC_API int cfc_enc_fused(int T) { return T >= EN_FUSED_ROWS; }

// Values of workspace (bf16) that the one launch for T rows of a model takes on a stream; 0: it does not take them, or so few
// CUs are the stream's that its workgroups would be long in coming.
CFC_API int cfc_enc_tiny(int T, int layers, int heads, hipStream_t stream) {
  if (T < 1 || T > EN_TINY_ROWS || layers < 1 || layers > EN_TINY_LAYERS || heads != EN_HEADS) return 0;
  uint32_t mask[8];                               // 256 CUs
  int cus = 0;
  if (hipExtStreamGetCUMask(stream, 8, mask) != hipSuccess) return 0;
  for (const uint32_t m : mask) cus += __builtin_popcount(m);
  return cus >= 4 * (EN_HEADS + EN_BLOCKS + EN_INNER) ? layers * T * (3 * EN_H + EN_F) + 8 : 0;
}

namespace {
constexpr int EN_CUS = 256;

template <bool GELU, bool LN>
void en_tile(int groups, uint16_t* x, const EncNorm& ln, const uint16_t* W, const uint16_t* bias, uint16_t* out, int T, int N, hipStream_t stream) {
  const dim3 grid(N / 64, (T + 16 * groups - 1) / (16 * groups));
  if (groups == 1) enc_tile_kernel<GELU, LN, 1><<<grid, 256, 0, stream>>>(x, ln, W, bias, out, T, N);
  else enc_tile_kernel<GELU, LN, 2><<<grid, 256, 0, stream>>>(x, ln, W, bias, out, T, N);
}

template <int K>
void en_ksplit(int groups, const uint16_t* x, const uint16_t* W, uint16_t* out, int T, hipStream_t stream) {
  const dim3 grid(EN_H / 16, (T + 16 * groups - 1) / (16 * groups));
  if (groups == 1) enc_ksplit_kernel<K, 1><<<grid, 256, 0, stream>>>(x, W, out, T);
  else enc_ksplit_kernel<K, 2><<<grid, 256, 0, stream>>>(x, W, out, T);
}

template <int K, int BM, int BN, int TM, int TN, int NS, int EPI>
void en_gemm(const uint16_t* x, const uint16_t* W, const uint16_t* bias, void* out, int T, int N, hipStream_t stream) {
  constexpr int LDS = NS * (BM + BN) * 128;
  enc_gemm_kernel<K, BM, BN, TM, TN, NS, EPI><<<N / BN * ((T + BM - 1) / BM), 64 * (BM / 32 / TM) * (BN / 32 / TN), LDS, stream>>>(x, W, bias, out, T, N);
}

// The tiles of the products of 384-wide rows with 1152 or 1536 columns, and of those that leave 384 columns: the largest whose
// workgroups, of which as many fit a CU as the LDS has rings for, are about one round of the chip.  Us of six layers with 64 x 64
// / 64 x 128 / 128 x 128 tiles of the wide products: 1000 rows 197 / 212 / 228, 1800 249 / 245 / 252, 3600 320 / 303 / 310,
// 4823 366 / 353 / 340, 9500 593 / 550 / 532, 16000 903 / 810 / 776; of the down product: 2560 247 / 263 / 278, 3000 286 / 278 /
// 292, 6500 451 / 452 / 434, 9500 568 / 551 / 540, 11000 659 / 657 / 668.
template <int EPI>
void en_wide(const uint16_t* x, const uint16_t* W, const uint16_t* bias, uint16_t* out, int T, int N, hipStream_t stream) {
  if (T <= 1280) en_gemm<EN_H, 64, 64, 1, 1, 4, EPI>(x, W, bias, out, T, N, stream);
  else if (T <= 4096) en_gemm<EN_H, 64, 128, 1, 2, 2, EPI>(x, W, bias, out, T, N, stream);
  else en_gemm<EN_H, 128, 128, 2, 2, 2, EPI>(x, W, bias, out, T, N, stream);
}

template <int K>
void en_raw(const uint16_t* x, const uint16_t* W, void* y, int T, hipStream_t stream) {
  if (T <= 2688) en_gemm<K, 64, 64, 1, 1, 4, EG_RAW>(x, W, nullptr, y, T, EN_H, stream);
  else if (K == EN_F && T > 5440 && T <= 10880) en_gemm<EN_F, 128, 128, 1, 2, 3, EG_RAW>(x, W, nullptr, y, T, EN_H, stream);
  else en_gemm<K, 64, 128, 1, 2, 3, EG_RAW>(x, W, nullptr, y, T, EN_H, stream);
}
}  // namespace

// Token states of a packed batch: embeddings, then every layer, one call for all launches.  W: host array of twelve
// device pointers per layer (qkv, qkv_b, o, o_b, ln1_g, ln1_b, up, up_b, down, down_b, ln2_g, ln2_b).  x [T][384] the
// states; att [T][384], qkv [T][1152], and unless cfc_enc_fused y [T][384] of 32 bits and h [T][1536]: workspace.  All else
// bf16, all 16-byte aligned.  With att null, h is the workspace of cfc_enc_tiny and no other is read; a wait in that launch is given up after
// `polls` loads (below 0: EN_POLLS).
CFC_API int cfc_enc_forward(const int32_t* ids, const int32_t* pos, const void* word, const void* pos_emb, const void* type_emb,
                            const void* emb_g, const void* emb_b, const int32_t* cu, const int32_t* tile_seq, const int32_t* tile_q0,
                            int n_tiles, int tile_rows, int max_seqlen, int layers, const void* const* W, int heads, float scale,
                            float eps, int T, void* x, void* y, void* att, void* qkv, void* h, int polls, hipStream_t stream) {
  const bool fused = cfc_enc_fused(T);
  if (att == nullptr) {
    const int n = cfc_enc_tiny(T, layers, heads, stream);
    if (n == 0 || h == nullptr || tile_rows < EN_TINY_ROWS || n_tiles < 0) return -1;
    EncTiny w = {(const uint16_t*)word, (const uint16_t*)pos_emb, (const uint16_t*)type_emb, (const uint16_t*)emb_g, (const uint16_t*)emb_b};
    memcpy(w.layer, W, sizeof(void*) * 12 * layers);
    enc_empty_kernel<<<min(256, (n / 8 + 255) / 256), 256, 0, stream>>>((uint4*)h, n / 8);
#define TINY(G, ALONE, GRID, POLLS) enc_tiny_kernel<G, ALONE><<<GRID, 512, en_tiny_lds(G), stream>>>(ids, pos, w, cu, tile_seq, n_tiles, layers, \
                                                                                         (uint16_t*)h, (uint16_t*)x, T, scale * 1.44269504f, eps, POLLS)
#define TINY_GO(G)                                                                                         \
  do {                                                                                                     \
    TINY(G, false, EN_HEADS + EN_BLOCKS + EN_INNER, polls < 0 ? EN_POLLS : polls);                          \
    TINY(G, true, 1, 0);                                                                                    \
  } while (0)
    if (T <= 16) TINY_GO(1);
    else if (T <= 32) TINY_GO(2);
    else TINY_GO(4);
#undef TINY_GO
#undef TINY
    return CFC_CHECK_LAUNCH();
  }
  if (T < 1 || layers < 1 || heads < 1 || EN_H % heads || (!fused && (h == nullptr || y == nullptr))) return -1;
  int rc = cfc_layernorm(x, word, nullptr, nullptr, emb_g, emb_b, ids, pos, pos_emb, type_emb, T, EN_H, eps, 2, stream);
  uint16_t *xp = (uint16_t*)x, *yp = (uint16_t*)y, *ap = (uint16_t*)att, *qp = (uint16_t*)qkv, *hp = (uint16_t*)h;
  const int blocks = (T + EN_ROWS - 1) / EN_ROWS;
  const uint16_t* const* P = (const uint16_t* const*)W;
  // Small tiles of 16 or 32 rows while a round of the chip takes those of the widest product's 24 columns (160 / 161 rows: 134 /
  // 161 us; of 16 rows still: 161), else tiles by way of the LDS (300 rows 167 in small tiles and 187; 350 rows 186 and 187)
  const int small = (T + 15) / 16 * 24 <= EN_CUS ? 1 : (T + 31) / 32 * 24 <= EN_CUS ? 2 : 0;
  auto attend = [&]() { return cfc_encoder_attention(qkv, cu, tile_seq, tile_q0, n_tiles, tile_rows, heads, EN_H / heads, max_seqlen, scale, att, stream); };
  for (int l = 0; l < layers && rc == 0; ++l) {
    const uint16_t* const* p = P + 12 * l;
    if (fused) {
      if (T > EN_CUS * EN_ROWS)       // more than a workgroup of 128 rows a CU
        enc_proj_wide_kernel<<<(T + EW_ROWS - 1) / EW_ROWS, 256, 0, stream>>>(xp, p[0], p[1], qp, T);
      else
        enc_proj_kernel<<<blocks, 256, 0, stream>>>(xp, p[0], p[1], qp, T, 3 * EN_T);
      if ((rc = attend())) break;
      const EncLayer L = {p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11]};
      enc_layer_kernel<<<blocks, 512, EN_LDS, stream>>>(ap, xp, L, xp, T, eps);
    } else if (small) {
      // a sublayer's last product waits in y for the next tiles' norm, which puts the layer's states in x, those between its
      // sublayers in att (the attention's output is used up by then)
      const EncNorm first = l ? EncNorm{yp, p[-3], ap, p[-2], p[-1], eps} : EncNorm{}, second = {yp, p[3], xp, p[4], p[5], eps};
      if (l == 0) en_tile<false, false>(small, xp, first, p[0], p[1], qp, T, 3 * EN_H, stream);
      else en_tile<false, true>(small, xp, first, p[0], p[1], qp, T, 3 * EN_H, stream);
      if ((rc = attend())) break;
      en_ksplit<EN_H>(small, ap, p[2], yp, T, stream);
      en_tile<true, true>(small, ap, second, p[6], p[7], hp, T, EN_F, stream);
      en_ksplit<EN_F>(small, hp, p[8], yp, T, stream);
    } else {
      en_wide<EG_BIAS>(xp, p[0], p[1], qp, T, 3 * EN_H, stream);
      if ((rc = attend())) break;
      en_raw<EN_H>(ap, p[2], y, T, stream);
      enc_norm_kernel<<<(T + 15) / 16, 256, 0, stream>>>(ap, (const float*)y, EncNorm{nullptr, p[3], xp, p[4], p[5], eps}, T);
      en_wide<EG_GELU>(ap, p[6], p[7], hp, T, EN_F, stream);
      en_raw<EN_F>(hp, p[8], y, T, stream);
      enc_norm_kernel<<<(T + 15) / 16, 256, 0, stream>>>(xp, (const float*)y, EncNorm{nullptr, p[9], ap, p[10], p[11], eps}, T);
    }
  }
  if (rc) return rc;
  if (!fused && small) {
    const uint16_t* const* p = P + 12 * layers;
    return cfc_layernorm(x, y, p[-3], att, p[-2], p[-1], nullptr, nullptr, nullptr, nullptr, T, EN_H, eps, 1, stream);
  }
  return CFC_CHECK_LAUNCH();
}
