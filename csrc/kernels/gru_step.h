// One token of the minimal gated recurrence (gru.hip): its gates, and a row's step, in a launch of its own or beside the
// rows of an attention that reads the same product (qkv.hip).
#pragma once
#include "recur.h"

namespace {

struct GruCols { const void* p; int split; int64_t ld, plane; };      // split 0: activations, else fp32 slabs

// decay 1 - z and contribution z c of one token.  With t = exp(pre_z): 1 - z = 1 / (1 + t) and z = t / (1 + t), neither
// the other's difference from 1, so that small ones keep their digits; sigmoid(min(u, 0)) is 1/2 where u >= 0
template <typename ACT>
__device__ __forceinline__ void gru_gates(float pz, float u, float& a, float& b) {
  const float t = exp_of<ACT>(fminf(pz, 60.f)), v = exp_of<ACT>(fminf(u, 0.f));
  a = over1<ACT>(t);
  b = t * a * (fmaxf(u, 0.f) + v * over1<ACT>(v));
}

template <typename ACT>
__device__ __forceinline__ float silu(float g) { return g * over1<ACT>(exp_of<ACT>(fminf(-g, 60.f))); }

struct GruStep {
  GruCols z, u, g;
  const float* bz; const float* bx;
  const int32_t* slots; const int32_t* ctx_lens;
  int W;
  float* state;                // [slots][W]
  void* out; int64_t ldo;
  float oscale;
};

// V channels from c on of row b, one token of its sequence
template <typename ACT, int V>
__device__ __forceinline__ void gru_step_row(const GruStep& s, int b, int c) {
  if (c >= s.W) return;
  // all at once; the state last, as it waits for its index (32 rows of 4096: 6.3 -> 4.9 us)
  ColsIn<ACT, V> zi, ui, gi;
  zi.ask(s.z.p, s.z.split, s.z.plane, b * s.z.ld + c);
  ui.ask(s.u.p, s.u.split, s.u.plane, b * s.u.ld + c);
  gi.ask(s.g.p, s.g.split, s.g.plane, b * s.g.ld + c);
  const Vec<V> vz = ldv<V>(s.bz + c), vx = ldv<V>(s.bx + c);
  float* sp = s.state + (size_t)s.slots[b] * s.W + c;
  Vec<V> S = s.ctx_lens[b] > 1 ? ldv<V>(sp) : zerov<V>();
  const Vec<V> zv = zi.get(s.z.p, s.z.split, s.z.plane, b * s.z.ld + c), uv = ui.get(s.u.p, s.u.split, s.u.plane, b * s.u.ld + c);
  const Vec<V> gv = gi.get(s.g.p, s.g.split, s.g.plane, b * s.g.ld + c);
  Vec<V> o;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    float a, k;
    gru_gates<ACT>(zv.v[e] + vz.v[e], uv.v[e] + vx.v[e], a, k);
    S.v[e] = a * S.v[e] + k;
    o.v[e] = S.v[e] * silu<ACT>(gv.v[e]) * s.oscale;
  }
  stv<V>(sp, S);
  stv<V>(reinterpret_cast<ACT*>(s.out) + b * s.ldo + c, o);
}

// vectors of four where every operand's rows allow them
inline bool gru_vec(const GruCols* a, int n, int W, int f32, const void* out, int64_t ldo) {
  bool v = W % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)out & (f32 ? 15 : 7)) == 0;
  for (int i = 0; i < n; ++i)
    v = v && a[i].ld % 4 == 0 && a[i].plane % 4 == 0 && ((uintptr_t)a[i].p & (a[i].split == 0 && !f32 ? 7 : 15)) == 0;
  return v;
}

}  // namespace
