// Hyper-connections: a residual stream of several copies x_1 .. x_S per token, 32-bit, [T][S][W].  One kernel stands between
// two sublayers, one row per workgroup:
//
//   y    the finished sublayer's result, the sum of a product's fp32 slabs
//   x_t  = sum_s mix[s][t] x_s + out[t] y, all from the old ones
//   u    = sum_s in[s] x_s of the new ones: what the next sublayer reads (in null: the plain sum)
//
// and an ending: u and its 1 / rms (a prompt's rows, ahead of their convolution), the normed row u / rms(u) w as an
// activation, or (decode) the normed row h as h + conv(h) over time, its earlier inputs in a slot per sequence.  Without y
// (the first sublayer) the streams stay as they are; with a stream stride of 0 they are all the same row.
#include "rows.h"

namespace {

enum { HN_RSTD = 0, HN_NORM = 1, HN_CONV = 2 };

struct HyperArgs {
  const float* x;              // [T] rows of stride ldx, streams lds apart
  int64_t ldx, lds;
  float* x_out;                // [T][S][W], null: not stored (may be x)
  const float* y; int split;   // slabs [split][T][W] or null
  const float* mix; const float* out; const float* in;
  const float* w;              // [W] the norm's multiplier
  float eps;
  const int32_t* rows;         // row of the b-th workgroup (null: b); normed outputs are at b
  int T, W, S;
  float* u; float* rstd;       // HN_RSTD
  const float* cw; int taps;   // HN_CONV: [taps][W]
  const int32_t* positions; const int32_t* slots;
  float* tail; int ring;       // [slots][ring][W], position p at p % ring
};

// SM >= S copies in registers; a thread holds NV vectors of V channels.  ROWS: FEW_ROWS at most, all that a row needs asked for
// ahead (90 VGPRs), or more: two workgroups of 1024 a CU (46; 2400 rows of 4096 in 4 streams 63.9 -> 58.5 us; smaller workgroups are
// enough to a CU either way, 700 rows of 1024 in 4 streams 6.1 ahead, 6.6 without), or past the caches
template <typename ACT, int V, int SM, int NV, int BT, int ROWS>
__global__ void __launch_bounds__(BT) hyper_norm_kernel(HyperArgs a, int mode, ACT* __restrict__ h) {
  constexpr bool NT = ROWS == ROWS_PAST;
  __shared__ float red[16];
  __shared__ float mx[SM * SM + 2 * SM];       // mix [from][to], out, in
  const int b = blockIdx.x, t = a.rows ? a.rows[b] : b, W = a.W, S = a.S;
  const float* xr = a.x + t * a.ldx;
  // All that a row's first vectors need is asked for before anything is waited for, what waits for an index last (5 rows of
  // 4096 in 4 streams: 6.9 -> 6.2 us, of which 300 KB a row through one CU take most).
  constexpr bool ONE = NV == 1 && SM <= 4 && ROWS == ROWS_FEW;     // else the registers are wanted for more vectors or streams
  constexpr int MX = SM * SM + 2 * SM;
  static_assert(!ONE || MX <= BT, "");
  float mv = 0.f;
  auto weight = [&](int i) {                   // past S: 0
    const int s = i / SM, k = i % SM;
    if (k >= S) return 0.f;
    if (s < SM) return s >= S ? 0.f : a.y ? a.mix[s * S + k] : s == k ? 1.f : 0.f;
    if (s == SM) return a.y ? a.out[k] : 0.f;
    return a.in ? a.in[k] : 1.f;
  };
  if constexpr (ONE) {
    if (threadIdx.x < MX) mv = weight(threadIdx.x);
  } else {
    for (int i = threadIdx.x; i < MX; i += BT) mx[i] = weight(i);
  }
  constexpr int PRE = NV == 1 && V == 4 && ROWS == ROWS_FEW ? 3 : 0;
  const int back = a.taps - 1;
  const bool ahead = PRE > 0 && back <= PRE;
  const int c0 = min((int)threadIdx.x * V, W - V);
  Vec<V> u[NV], x[SM], y = zerov<V>(), past[PRE ? PRE : 1], cw[PRE ? PRE + 1 : 1], gain;
  Slabs<V, (ROWS == ROWS_FEW || NV > 1 || SM > 4 ? 8 : 4), ONE, NT> slabs;
  float ss = 0.f;
  auto ask = [&](int c) {
#pragma unroll
    for (int s = 0; s < SM; ++s) x[s] = ldv<V, NT>(xr + min(s, S - 1) * a.lds + c);
    if (!a.y) return;
    y = zerov<V>();
    slabs.ask(a.y, a.split, (int64_t)a.T * W, (size_t)t * W + c);
    if constexpr (!ONE) slabs.add(y, a.y, a.split, (int64_t)a.T * W, (size_t)t * W + c);
  };
  if constexpr (ONE) ask(c0);
  if (NV == 1 && V == 4 && SM <= 4 && mode != HN_RSTD) gain = ldv<V>(a.w + c0);
  if constexpr (PRE > 0) {
    if (mode == HN_CONV && ahead)
#pragma unroll
      for (int d = 0; d <= PRE; ++d) cw[d] = ldv<V>(a.cw + (size_t)max(back - d, 0) * W + c0);
  }
  const int pos = mode == HN_CONV ? a.positions[b] : 0;
  float* tail = mode == HN_CONV && back > 0 ? a.tail + (size_t)a.slots[b] * a.ring * W : nullptr;
  if constexpr (PRE > 0)
    if (mode == HN_CONV && ahead)
#pragma unroll
      for (int d = 1; d <= PRE; ++d) past[d - 1] = d <= back && d <= pos ? ldv<V>(tail + (size_t)((pos - d) % a.ring) * W + c0) : zerov<V>();
  if constexpr (!ONE) ask(c0);
  if (ONE && threadIdx.x < MX) mx[threadIdx.x] = mv;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = (k * BT + threadIdx.x) * V;
    u[k] = zerov<V>();
    if (c >= W) continue;
    if (k) ask(c);
    if (a.y) {
      if constexpr (ONE) slabs.add(y, a.y, a.split, (int64_t)a.T * W, (size_t)t * W + c);
#pragma unroll
      for (int q = 0; q < SM; ++q) {
        if (q >= S) break;
        Vec<V> n;
#pragma unroll
        for (int e = 0; e < V; ++e) n.v[e] = mx[SM * SM + q] * y.v[e];
#pragma unroll
        for (int s = 0; s < SM; ++s)
#pragma unroll
          for (int e = 0; e < V; ++e) n.v[e] += mx[s * SM + q] * x[s].v[e];
        if (a.x_out) stv<V, NT>(a.x_out + ((size_t)t * S + q) * W + c, n);
#pragma unroll
        for (int e = 0; e < V; ++e) u[k].v[e] += mx[SM * SM + SM + q] * n.v[e];
      }
    } else {
#pragma unroll
      for (int s = 0; s < SM; ++s)
#pragma unroll
        for (int e = 0; e < V; ++e) u[k].v[e] += mx[SM * SM + SM + s] * x[s].v[e];
    }
#pragma unroll
    for (int e = 0; e < V; ++e) ss += u[k].v[e] * u[k].v[e];
  }
  const float r = 1.f / sqrtf(block_sum<NV == 1 ? 16 : 1>(ss, red) / (float)W + a.eps);
  if (mode == HN_RSTD) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = (k * BT + threadIdx.x) * V;
      if (c < W) stv<V>(a.u + (size_t)t * W + c, u[k]);
    }
    if (threadIdx.x == 0) a.rstd[t] = r;
    return;
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = (k * BT + threadIdx.x) * V;
    if (c >= W) continue;
    Vec<V> g, n;
    if constexpr (NV == 1 && V == 4 && SM <= 4) g = gain;
    else g = ldv<V>(a.w + c);
#pragma unroll
    for (int e = 0; e < V; ++e) n.v[e] = u[k].v[e] * r * g.v[e];
    if (mode == HN_CONV) {
      const Vec<V> own = n;
      if (ahead) {
        if constexpr (PRE > 0) {
#pragma unroll
          for (int e = 0; e < V; ++e) n.v[e] += cw[0].v[e] * own.v[e];
#pragma unroll
          for (int d = 1; d <= PRE; ++d)
            if (d <= back)
#pragma unroll
              for (int e = 0; e < V; ++e) n.v[e] += cw[d].v[e] * past[d - 1].v[e];
        }
      } else {
        for (int d = 0; d <= back && d <= pos; ++d) {
          const Vec<V> o = d ? ldv<V>(tail + (size_t)((pos - d) % a.ring) * W + c) : own;
          const Vec<V> wd = ldv<V>(a.cw + (size_t)(back - d) * W + c);
#pragma unroll
          for (int e = 0; e < V; ++e) n.v[e] += wd.v[e] * o.v[e];
        }
      }
      if (back > 0) stv<V>(tail + (size_t)(pos % a.ring) * W + c, own);
    }
    stv<V>(h + (size_t)b * W + c, n);
  }
}

constexpr int64_t HYPER_PAST_BYTES = 512ll << 20;      // of all streams

template <typename ACT, int V, int SM>
int hyper_go(hipStream_t s, int n, const HyperArgs& a, int mode, void* h) {
  const int vecs = (a.W + V - 1) / V;
  // past the caches: several streams stay there longer.  us of 4 x 4096 to fp32 and to bf16 rows, before, two workgroups a CU, and past the
  // caches: 14 000 rows 342, 336, 307 and 352, 347, 333; 4800 rows 105, 103, 104 and 115, 109, 118
#define HN_GO(NV, BT, ROWS) hyper_norm_kernel<ACT, V, SM, NV, BT, ROWS><<<n, BT, 0, s>>>(a, mode, (ACT*)h)
#define GO(NV, BT)                                                                                                   \
  do {                                                                                                               \
    constexpr bool one = V == 4 && NV == 1, past = V == 4 && SM <= 4 && NV <= 4;                                     \
    if (one && (SM > 4 || n <= FEW_ROWS || BT < 1024)) HN_GO(NV, BT, (one ? ROWS_FEW : ROWS_SOME));                  \
    else if (past && 4ll * n * a.S * a.W > HYPER_PAST_BYTES) HN_GO(NV, BT, (past ? ROWS_PAST : ROWS_SOME));            \
    else HN_GO(NV, BT, ROWS_SOME);                                                                                   \
  } while (0)
  if (vecs <= 64) GO(1, 64);
  else if (vecs <= 256) GO(1, 256);
  else if (vecs <= 512) GO(1, 512);
  else if (vecs <= 1024) GO(1, 1024);
  else if (vecs <= 4096) GO(4, 1024);
  else if (vecs <= 16384) GO(16, 1024);
  else return -4;
#undef GO
#undef HN_GO
  return CFC_CHECK_LAUNCH();
}

constexpr int HYPER_MAX = 16;

}  // namespace

// mode 0: u and rstd; 1: normed rows into h [n][W]; 2: decoded rows, normed and convolved.  f32: h is fp32 (else bf16).
// y null: no update (mix, out unused); x_out null: streams not stored; rows null: row b of T (modes 1)
CFC_API int cfc_hyper_norm(int mode, int f32, int n, const int32_t* rows, const float* x, int64_t ldx, int64_t lds, float* x_out,
                           const float* y, int split, const float* mix, const float* out, const float* in, const float* w,
                           float eps, int T, int W, int S, float* u, float* rstd, const float* cw, int taps,
                           const int32_t* positions, const int32_t* slots, float* tail, int ring, void* h, hipStream_t stream) {
  if (n <= 0) return 0;
  if (T < 1 || W < 1 || S < 1 || S > HYPER_MAX || !x || (!rows && n > T)) return -1;
  if (y && (split < 1 || !mix || !out)) return -2;
  if (mode == HN_RSTD ? (!u || !rstd) : (!h || !w)) return -2;
  if (mode == HN_CONV && (rows || !cw || taps < 1 || !positions || (taps > 1 && (!slots || !tail || ring < taps - 1)))) return -3;
  if (mode < HN_RSTD || mode > HN_CONV || (mode != HN_NORM && rows)) return -3;
  const HyperArgs a{x, ldx, lds, x_out, y, split, mix, out, in, w, eps, rows, T, W, S, u, rstd, cw, taps, positions, slots, tail,
                    ring > 0 ? ring : 1};
  const bool v4 = W % 4 == 0 && ldx % 4 == 0 && lds % 4 == 0;
#define HG(ACT)                                                             \
  return !v4 ? hyper_go<ACT, 1, HYPER_MAX>(stream, n, a, mode, h)           \
             : S <= 4 ? hyper_go<ACT, 4, 4>(stream, n, a, mode, h) : hyper_go<ACT, 4, HYPER_MAX>(stream, n, a, mode, h)
  if (f32) HG(float);
  HG(uint16_t);
#undef HG
}
