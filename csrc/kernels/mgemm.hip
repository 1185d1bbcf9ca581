// Prompt GEMM for gfx950 between the decode GEMM (up to 128 rows) and the 256 x 256 tiles of pgemm.hip
// (thousands of rows):  Y[M, N] = X[M, K] . W[N, K]^T  (bf16 in, fp32 accumulate, W fragment-packed).
//
// A product of a few hundred rows has too few 256 x 256 tiles for 256 CUs (4096 columns of 1536 rows: 96), and the
// decode GEMM's waves, 16 columns each, read every X fragment from LDS for one MFMA.  Here a workgroup makes a
// 32 MT x 128 tile, MT = 4 .. 8 (the height that wastes the fewest rows and CUs), of all of K or of one of `split`
// slices, whose fp32 slabs the consumer adds up.  What bounds it is how fast a CU pulls X and W through its L2:
// 55 - 66 B/ns with every CU at it (30 for lines that miss), so a 64-deep stage of 32 / 40 / 48 KB (MT = 4 / 6 / 8)
// takes 0.37 / 0.44 / 0.54 us on a chip that is half idle, 0.53 / 0.62 / 0.75 on a full one; about 10 us of a
// call are its start, the first stages' way and the stores.
//
//   * 8 waves in two groups of 2 x 2; both groups hold the whole tile, a wave 16 MT x 64 of it, and group g
//     multiplies k = 32 g .. 32 g + 31 of every stage: 4 MT MFMAs per MT + 4 fragment reads, where eight waves side
//     by side on the tile would read half as much again.  Their sums meet in LDS at the end, each group finishing
//     half of the columns;
//   * the groups run one barrier apart (as in pgemm.hip): one's MFMAs cover the other's LDS-DMA issue and fragment
//     reads;
//   * a ring of R = 3 .. 5 stages (160 KB): a stage is issued into the slot that both groups read one stage earlier
//     and has R - 2 stages' time to land;
//   * X image: row r's chunk c at r * 128 + ((c ^ (r & 7)) << 4), swizzled through the DMA source; W: one 1-KB piece per
//     16 x 32 fragment.  Reads of both are free of bank conflicts;
//   * consecutive workgroups of an XCD take the M-tiles of one run of columns, so W comes from memory once.
//
// us with the sum of the slabs, N x K 6144 x 4096 / 4096 x 4096 / 4096 x 14336, before (decode GEMM or pgemm) -> here:
//   160 rows 29 / 23 / 44 -> 25 / 22 / 37;  420 rows 40 / 35 / 69 -> 35 / 28 / 59;
//   1024 rows 74 / 74 / 129 -> 51 / 41 / 105;  1536 rows (75 in pgemm) / 74 / 227 -> - / 50 / 148.
#include <algorithm>
#include <type_traits>

#include "pgemm.h"

namespace {

constexpr int MG_BN = 128, MG_BK = 64;

template <int MT>
struct MgShape {
  static constexpr int BM = 32 * MT;
  static constexpr int XB = BM * 128;                  // X image of a stage
  static constexpr int STAGE = XB + MG_BN * 128;
  static constexpr int P = (4 * MT + 16 + 7) / 8;      // 1-KB DMA pieces per wave and stage
  static constexpr int R = 163840 / STAGE < 5 ? 163840 / STAGE : 5;
};

template <int N>
__device__ __forceinline__ void mg_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}
__device__ __forceinline__ void mg_barrier() { asm volatile("s_barrier" ::: "memory"); }

// at most `ahead` stages of P pieces stay in flight
template <int P, int MAXA>
__device__ __forceinline__ void mg_wait_ahead(int ahead) {
  if constexpr (MAXA == 0) {
    mg_wait_barrier<0>();
  } else {
    if (ahead >= MAXA) mg_wait_barrier<MAXA * P>();
    else mg_wait_ahead<P, MAXA - 1>(ahead);
  }
}

template <int MT, int EPI>
__global__ void __launch_bounds__(512, 1)
    mgemm_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, float* __restrict__ part,
                 uint16_t* __restrict__ out, int M, int N, int K, int ldo, int tiles_m, int tiles_n, int split, int wnw,
                 PgGlu gp, const int32_t* __restrict__ in_of) {
  using S = MgShape<MT>;
  constexpr int P = S::P, R = S::R;
  __shared__ __attribute__((aligned(16))) char smem[R * S::STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = w >> 2, wr = (w >> 1) & 1, wc = w & 1;

  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = id % (tiles_m * tiles_n), ks = id / (tiles_m * tiles_n);
  const int m0 = tile % tiles_m * S::BM, n0 = tile / tiles_m * MG_BN;
  // several inputs [inputs][M][K]: columns n0 .. n0 + 127 multiply input in_of[n0 / 128]
  if (in_of) X += (size_t)__builtin_amdgcn_readfirstlane(in_of[tile / tiles_m]) * M * K;
  const int nks = K / MG_BK;
  const int kb = (int)((long)ks * nks / split), nst = (int)((long)(ks + 1) * nks / split) - kb;

  // ---- DMA sources of pieces w, w + 8, ...: 4 MT of X (8 image rows each), 16 of W (fragments)
  uint32_t voff[P];
  const char* src[P];
  uint32_t adv[P];
  const int kg_all = K / 32;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int p = min(w + 8 * i, 4 * MT + 15);
    if (p < 4 * MT) {
      const int r = 8 * p + (lane >> 3), c = (lane & 7) ^ (r & 7);
      voff[i] = ((uint32_t)min(m0 + r, M - 1) * (uint32_t)K + 8u * c) * 2u;
      adv[i] = MG_BK * 2;
      src[i] = reinterpret_cast<const char*>(X) + (size_t)kb * adv[i];
    } else {
      const int f = p - 4 * MT, g = min(n0 / 16 + (f >> 1), N / 16 - 1);
      voff[i] = (uint32_t)(((g / wnw) * kg_all + (f & 1)) * wnw + g % wnw) * 1024u + 16u * lane;
      adv[i] = (uint32_t)wnw * 2048u;
      src[i] = reinterpret_cast<const char*>(W) + (size_t)kb * adv[i];
    }
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(pg_lds_t*)smem);
  auto issue = [&](int slot) {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      pg_glds16(voff[i], src[i], lds0 + slot * S::STAGE + min(w + 8 * i, 4 * MT + 15) * 1024);
      src[i] += adv[i];
    }
  };

  f32x4_t acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int xrd = (16 * MT * wr + (lane & 15)) * 128 + (((4 * grp + (lane >> 4)) ^ (lane & 7)) << 4);
  const int wrd = S::XB + (8 * wc + grp) * 1024 + 16 * lane;

  // ---- prologue: R - 1 stages under way, the first one landed in every wave
#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < nst) issue(s);
  mg_wait_ahead<P, R - 2>(nst - 1);
  if (grp == 1) mg_barrier();   // the stagger: group 1 runs one barrier behind group 0
  int slot = 0, fill = R - 1;
  auto stage = [&](int t, auto last) {
    constexpr bool LAST = decltype(last)::value;   // nothing left to issue
    bf16x8_t xf[MT], wf[4];
    if constexpr (!LAST) issue(fill);
    const char* img = smem + slot * S::STAGE;
#pragma unroll
    for (int j = 0; j < 4; ++j) wf[j] = *reinterpret_cast<const bf16x8_t*>(img + wrd + j * 2048);
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[i] = *reinterpret_cast<const bf16x8_t*>(img + xrd + i * 2048);
    // this wave's pieces of stage t + 1 and its reads of stage t
    if constexpr (LAST) mg_wait_ahead<P, R - 2>(nst - 2 - t);
    else mg_wait_barrier<P * (R - 2)>();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[i], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    mg_barrier();
    slot = slot + 1 == R ? 0 : slot + 1;
    fill = fill + 1 == R ? 0 : fill + 1;
  };
  int t = 0;
  for (; t + R - 1 < nst; ++t) stage(t, std::false_type{});
  for (; t < nst; ++t) stage(t, std::true_type{});
  if (grp == 0) mg_barrier();   // matches the stagger: every read and every DMA is over

  // ---- the two groups' sums: group 0 finishes n-tiles 0, 1 of each wave, group 1 n-tiles 2, 3
  float4* ex = reinterpret_cast<float4*>(smem) + lane;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float4 give;
      float* gv = &give.x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = acc[i][j][e], b = acc[i][2 + j][e];
        gv[e] = grp ? a : b;
        acc[i][j][e] = grp ? b : a;      // what this wave finishes
      }
      ex[(((w ^ 4) * MT + i) * 2 + j) * 64] = give;
    }
  __syncthreads();
  const int g = lane >> 4;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + 16 * (MT * wr + i) + (lane & 15);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float4 o = ex[((w * MT + i) * 2 + j) * 64];
      float v[4] = {acc[i][j][0] + o.x, acc[i][j][1] + o.y, acc[i][j][2] + o.z, acc[i][j][3] + o.w};
      const int nb = n0 + 64 * wc + 32 * grp + 16 * j, n = nb + 4 * g;
      if constexpr (pg_gated(EPI)) {
        const uint32_t y = pg_gate2<EPI>(v, gp);
        if (m < M && nb < N) *reinterpret_cast<uint32_t*>(out + (size_t)m * ldo + nb / 2 + pg_gate_col(g)) = y;
      } else if constexpr (EPI == PG_F32) {
        if (m < M && n < N)
          *reinterpret_cast<float4*>(part + ((size_t)ks * M + m) * N + n) = make_float4(v[0], v[1], v[2], v[3]);
      } else if (m < M && n < N) {
        *reinterpret_cast<uint2*>(out + (size_t)m * ldo + n) =
            make_uint2(pack2bf(pg_out<EPI>(v[0]), pg_out<EPI>(v[1])), pack2bf(pg_out<EPI>(v[2]), pg_out<EPI>(v[3])));
      }
    }
  }
}

template <int EPI>
int mgemm_launch(const void* x, const void* w, void* out, int M, int N, int K, int ldo, int bm, int split, int wnw,
                 const PgGlu& gp, hipStream_t stream, const int32_t* in_of = nullptr) {
  const int tm = (M + bm - 1) / bm, tn = (N + MG_BN - 1) / MG_BN;
#define MG_CASE(MT)                                                                                                 \
  case 32 * MT:                                                                                                     \
    mgemm_kernel<MT, EPI><<<tm * tn * split, 512, 0, stream>>>((const uint16_t*)x, (const uint16_t*)w, (float*)out, \
                                                               (uint16_t*)out, M, N, K, ldo, tm, tn, split, wnw, gp, in_of); \
    break;
  switch (bm) {
    MG_CASE(4)
    MG_CASE(5)
    MG_CASE(6)
    MG_CASE(7)
    MG_CASE(8)
    default: return (int)hipErrorInvalidValue;
  }
#undef MG_CASE
  return (int)hipGetLastError();
}

// ---- which rows of a product run here.  All times in us, fitted to N, K of 1024 .. 28672 and 129 .. 5500 rows.
constexpr int MG_CUS = 256;
constexpr int MG_PGEMM_TILES = 96;        // fewer tiles than this are not taken to pgemm by its callers

// mgemm_kernel in bm-row tiles, mostly within 10 %.  A 64-deep stage takes 0.2 + 0.0013 bm on an idle chip, up to 0.42
// more of that on a full one (0.55 in all rounds but the last), and no less than its 16 KB of W and its rows of X at
// 67 B/ns: a last tile of few rows runs ahead and brings W into the L2 for the others (385 rows 31 us, 384 rows 40), so
// they count as fewer rows.  One row tile alone waits for W from memory, 0.59 (64 workgroups) to 0.75.  4 per round of
// workgroups, 6 per call; slabs are written and read, one fp32 result is written, at 7 TB/s.
double mgemm_us(int M, int N, int K, int bm, int split, bool fp32) {
  const int tm = (M + bm - 1) / bm, last = M - (tm - 1) * bm;
  const double rows = last + 0.6 * (bm - last) * (1.0 - 1.0 / tm);
  const int64_t wgs = (int64_t)tm * ((N + MG_BN - 1) / MG_BN) * split;
  const double full = (double)((wgs - 1) / MG_CUS), fill = ((wgs - 1) % MG_CUS + 1) / (double)MG_CUS;
  const double stages = (K + 64 * split - 1) / (64 * split), idle = 0.2 + 0.0013 * bm;
  const double least = std::max((16384 + 128 * rows) / 67e3, tm == 1 ? 0.51 + 0.24 * std::min(1.0, wgs / 192.0) : 0.0);
  double t = 6.0 + full * (4.0 + stages * std::max(idle * 1.55, least)) + 4.0 +
             stages * std::max(idle * (1.0 + 0.42 * fill * fill * fill), least);
  t = std::max(t, 10.0 + (double)N * K * 2 / 5.0e6);
  return t + (split > 1 ? 8.0 * split : 4.0 * fp32) * M * N / 7.0e6;
}

// What X alone takes: an XCD's workgroups share columns, not rows, so each of up to 8 runs of columns (and K slices) brings
// X into its XCD's L2, 7.6 TB/s in all (16041 rows of 512 x 4096 83, in pgemm 67; 8171 of 1024 x 4096 81 and 69).
double mgemm_x_us(int M, int N, int K, int split) {
  const int64_t runs = (int64_t)((N + MG_BN - 1) / MG_BN) * split;
  return 12.0 + (double)M * K * 2 * std::max(1.0, (double)std::min<int64_t>(8, runs) / split) / 7.6e6;
}

// pgemm's persistent kernel, in tiles of the height it takes
double ppp_us(int M, int N, int K, bool fp32) {
  return ppp_us_at(M, N, K, ppp_height(M, N, K)) * (fp32 ? 1.04 : 1.0);
}

enum { MG_ACT = 0, MG_SLABS = 1, MG_WHOLE = 2 };

// the fastest tile and split.  Splits are powers of two, so that rows multiplied in batches of different sizes are
// mostly added up in the same order; 2 more for the launch that adds an activation's slabs up, 3 more (`alone`) for slices
// of 8 stages or fewer, over before their ring is full: 1507 rows of 512 x 1024 in 4 slices 17.9, whole 12.3; 339 of
// 1536 x 4096 in 8 22.2, in 4 19.4.  Beyond 3 rounds of workgroups nothing was measured to be faster than pgemm.
double mgemm_best(int M, int N, int K, int kind, bool split_ok, bool alone, int& bm, int& split, int rounds = 3) {
  double best = 1e30;
  for (int b = 128; b <= 256; b += 32) {
    if ((int64_t)((M + b - 1) / b) * ((N + MG_BN - 1) / MG_BN) > rounds * MG_CUS) continue;
    for (int s = 1; s <= (split_ok ? 8 : 1) && s * 64 <= K; s *= 2) {
      const double t = mgemm_us(M, N, K, b, s, kind != MG_ACT) + (s > 1 && kind == MG_ACT ? 2.0 : 0.0) +
                       (s > 1 && alone && K <= 512 * s ? 3.0 : 0.0);
      if (t < best) best = t, bm = b, split = s;
    }
  }
  return best;
}

// cfc_prompt_plan's choice and its us
double prompt_best(int M, int N, int K, int kind, int* plan) {
  plan[0] = plan[1] = plan[2] = 0;
  const int64_t weights = (int64_t)N * K;
  int bm = 0, split = 0;
  if (M <= 128 || N < 64 || K < 64 || (int64_t)M * K * 2 >= (1ll << 32) || weights * 2 >= (1ll << 32))
    return ppp_us(M, N, K, kind != MG_ACT);
  double all = mgemm_best(M, N, K, kind, kind != MG_WHOLE, true, bm, split);
  if (weights <= 1 << 23 && M <= (weights > 1 << 22 ? 256 : 640)) return all;       // the decode GEMM, within 10 %
  const int tn = (N + 255) / 256, tm = (M + 255) / 256;
  double best = M < 256 ? 1e29 : ppp_us(M, N, K, kind != MG_ACT);
  if ((int64_t)tm * tn >= MG_PGEMM_TILES) all = std::max(all, mgemm_x_us(M, N, K, split));
  if (all < best) best = all, plan[1] = bm, plan[2] = split;
  const int rounds = (int)((int64_t)tm * tn / MG_CUS), head = rounds ? (int)((int64_t)MG_CUS * rounds / tn) * 256 : 0;
  if (head > 0 && head < M && K >= 128) {
    // behind another launch its own start is hidden, and W waits in the 256 MB cache for a row tile or two if what the head read and
    // wrote fits there as well, nearly (1 to 128 rows of 28672 x 4096 behind 512 40 to 49 us, alone 58; 80 of 16384 x 4096 behind 1024
    // 28, alone 42, behind 7168 46)
    double rest = mgemm_best(M - head, N, K, kind, kind == MG_ACT, false, bm, split) - 3.0;
    if (M - head <= 256 && 2 * (weights + (int64_t)head * (N + K)) <= 280ll << 20) rest *= 0.8;
    const double both = ppp_us(head, N, K, kind != MG_ACT) + rest;
    // (by a hundredth in runs of 1.2 ms and longer, where the model is no nearer: 14 000 and 15 760 rows of 28672 x 4096 take the same either way)
    if (both < (1.0 - 0.01 * std::min(1.0, best / 1200.0)) * best) best = both, plan[0] = head, plan[1] = bm, plan[2] = split;
  }
  return best;
}

}  // namespace

// The model misses the fastest of the heights, this kernel alone and a head with its rest by 0.2 % on average of 550 sizes measured (257 to
// 15 049 rows of 1024 .. 28672 x 2048 .. 14336), and by 9 % at most.
// A prompt product's plan: plan = {head, bm, split}: `head` rows (as many as whole rounds of 256 x 256 tiles have) on pgemm's
// persistent kernel, in tiles of the height it takes, and the others here; {0, 0, 0}: all on the decode GEMM or pgemm.  kind 0: an activation (an epilogue,
// or what adds the slabs up), 1: fp32 slabs for a consumer that adds them up (with a head: one), 2: one fp32 result.
//   * up to 128 rows, and 256 (640) of 2^23 (2^22) weights or fewer: the decode GEMM (129 .. 256 rows, 2^23 weights: 17
//     against 18; 2^21: 14 against 15 at 220 rows, 16 against 17 at 512, but 18.6 against 18.3 at 700);
//   * all here where pgemm's tiles leave the chip idle: 4096 x 4096 up to 1866 rows (62 against 65; 2072: 78 against 65),
//     28672 x 4096 up to 256 (68 against 87; 285: 82 against 76 in tiles of 192 rows);
//     nor where X would be brought into every L2 for a few columns each (mgemm_x_us): 1024 x 4096 up to 7000 rows;
//   * the rows beyond pgemm's last whole round here: 4096 x 14336 of 4500 rows 438 -> 367, 4096 x 4096 136 -> 124, 28672 x
//     4096 of 560 138 -> 125 (of 1344 not: 242 and 264).
CFC_API int cfc_prompt_plan(int M, int N, int K, int kind, int* plan) {
  prompt_best(M, N, K, kind, plan);
  return 0;
}

// us of a product by its plan
CFC_API double cfc_prompt_us(int M, int N, int K, int kind) {
  int plan[3];
  return M < 1 || N < 1 || K < 1 ? 0.0 : prompt_best(M, N, K, kind, plan);
}

// Rows per workgroup of cfc_mgemm_joint and its us; 0 where it does not fit or takes more than six rounds of workgroups
// (five products of 4096 x 4096: 2300 rows 400 -> 360, 2569 rows 404 -> 427).
CFC_API int cfc_joint_plan(int M, int N, int K, int* bm, double* us) {
  int split = 0;
  *bm = 0;
  *us = 1e30;
  if (M > 128 && N >= 128 && K >= 64 && (int64_t)M * K * 2 < (1ll << 32) && (int64_t)N * K * 2 < (1ll << 32))
    *us = mgemm_best(M, N, K, MG_ACT, false, false, *bm, split, 6);
  return 0;
}

// epi as cfc_pgemm's (0 bf16, 3 SwiGLU, 4 fp32, 6 squared relu) or 5, the clamped GLU with its constants; out: row stride
// ldo, or (fp32) slabs [split][M][N].  bm: 128, 160 .. 256 rows per workgroup.  W packed for bn = 16 wnw.
CFC_API int cfc_mgemm(const void* x, const void* w, void* out, int M, int N, int K, int epi, int ldo, int bm, int split,
                      int wnw, float limit, float alpha, float beta, float cubic, hipStream_t stream) {
  if (M < 1 || N < 64 || K < 64 || K % 64 || N % 64 || split < 1 || split > K / 64 || (split > 1 && epi != PG_F32) ||
      wnw < 1 || N % (16 * wnw) || (uint64_t)M * K * 2 >= (1ull << 32) || (uint64_t)N * K * 2 >= (1ull << 32) ||
      (epi != PG_F32 && (ldo % 4 || ldo < (pg_gated(epi) ? N / 2 : N))) || ((uintptr_t)out & (epi == PG_F32 ? 15 : 7)) ||
      (int64_t)((M + 127) / 128) * ((N + 127) / 128) * split > (1 << 30))
    return (int)hipErrorInvalidValue;
  PgGlu gp;
  gp.limit = limit; gp.alpha = alpha; gp.beta = beta; gp.cubic = cubic;
  switch (epi) {
    case PG_BF16: return mgemm_launch<PG_BF16>(x, w, out, M, N, K, ldo, bm, split, wnw, gp, stream);
    case PG_SWIGLU: return mgemm_launch<PG_SWIGLU>(x, w, out, M, N, K, ldo, bm, split, wnw, gp, stream);
    case PG_F32: return mgemm_launch<PG_F32>(x, w, out, M, N, K, ldo, bm, split, wnw, gp, stream);
    case PG_GLU: return mgemm_launch<PG_GLU>(x, w, out, M, N, K, ldo, bm, split, wnw, gp, stream);
    case PG_RELU2: return mgemm_launch<PG_RELU2>(x, w, out, M, N, K, ldo, bm, split, wnw, gp, stream);
    default: return (int)hipErrorInvalidValue;
  }
}

// Activations [M][N] (row stride ldo) of x [inputs][M][K], columns 128 t .. of W (packed for bn = 128) multiplying input
// in_of[t]: several products of a layer in one launch.
CFC_API int cfc_mgemm_joint(const void* x, const void* w, void* out, int M, int N, int K, int ldo, int bm, const int32_t* in_of,
                            hipStream_t stream) {
  if (M < 1 || N < MG_BN || N % MG_BN || K < 64 || K % 64 || !in_of || (uint64_t)M * K * 2 >= (1ull << 32) ||
      (uint64_t)N * K * 2 >= (1ull << 32) || ldo % 4 || ldo < N || ((uintptr_t)out & 7) ||
      (int64_t)((M + 127) / 128) * (N / MG_BN) > (1 << 30))
    return (int)hipErrorInvalidValue;
  return mgemm_launch<PG_BF16>(x, w, out, M, N, K, ldo, bm, 1, MG_BN / 16, PgGlu{}, stream, in_of);
}
