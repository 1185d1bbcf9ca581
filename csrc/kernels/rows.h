// Row kernels' shared parts (one workgroup per row of a 32-bit stream, channels in vectors of V per thread): vector
// loads and stores of activations (bf16 bits or float), sums of fp32 k-slice slabs, launch shapes.
#pragma once
#include "common.h"

namespace {

__device__ __forceinline__ float ld1(const uint16_t* p) { return bf2f(*p); }
__device__ __forceinline__ float ld1(const float* p) { return *p; }

template <int V> struct Vec { float v[V]; };

// NT: past the caches (nontemporal), as far as vectors of four go
typedef float row_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t row_u2 __attribute__((ext_vector_type(2)));
template <int V, bool NT = false>
__device__ __forceinline__ Vec<V> ldv(const float* p) {
  Vec<V> r;
  if constexpr (V == 4 && NT) {
    const row_f4 f = __builtin_nontemporal_load(reinterpret_cast<const row_f4*>(p));
    r.v[0] = f.x; r.v[1] = f.y; r.v[2] = f.z; r.v[3] = f.w;
  } else if constexpr (V == 4) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    r.v[0] = f.x; r.v[1] = f.y; r.v[2] = f.z; r.v[3] = f.w;
  } else {
    r.v[0] = *p;
  }
  return r;
}
template <int V, bool NT = false>
__device__ __forceinline__ Vec<V> ldv(const uint16_t* p) {
  Vec<V> r;
  if constexpr (V == 4) {
    uint2 u;
    if constexpr (NT) {
      const row_u2 n = __builtin_nontemporal_load(reinterpret_cast<const row_u2*>(p));
      u = make_uint2(n.x, n.y);
    } else {
      u = *reinterpret_cast<const uint2*>(p);
    }
    r.v[0] = __uint_as_float(u.x << 16); r.v[1] = __uint_as_float(u.x & 0xffff0000u);
    r.v[2] = __uint_as_float(u.y << 16); r.v[3] = __uint_as_float(u.y & 0xffff0000u);
  } else {
    r.v[0] = bf2f(*p);
  }
  return r;
}
template <int V, bool NT = false>
__device__ __forceinline__ void stv(float* p, const Vec<V>& r) {
  if constexpr (V == 4 && NT) __builtin_nontemporal_store(row_f4{r.v[0], r.v[1], r.v[2], r.v[3]}, reinterpret_cast<row_f4*>(p));
  else if constexpr (V == 4) *reinterpret_cast<float4*>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
  else *p = r.v[0];
}
template <int V, bool NT = false>
__device__ __forceinline__ void stv(uint16_t* p, const Vec<V>& r) {
  if constexpr (V == 4 && NT) __builtin_nontemporal_store(row_u2{pack2bf(r.v[0], r.v[1]), pack2bf(r.v[2], r.v[3])}, reinterpret_cast<row_u2*>(p));
  else if constexpr (V == 4) *reinterpret_cast<uint2*>(p) = make_uint2(pack2bf(r.v[0], r.v[1]), pack2bf(r.v[2], r.v[3]));
  else *p = f2bf(r.v[0]);
}
template <int V>
__device__ __forceinline__ Vec<V> zerov() {
  Vec<V> r;
#pragma unroll
  for (int e = 0; e < V; ++e) r.v[e] = 0.f;
  return r;
}

// y += slabs of row offset `off`, F in flight (past the last: re-read, not added)
template <int V, int F = 8, bool NT = false>
__device__ __forceinline__ void add_slabs(Vec<V>& y, const float* p, int split, int64_t plane, size_t off, int first = 0) {
  if (split == 1) {
    const Vec<V> a = ldv<V, NT>(p + off);
#pragma unroll
    for (int e = 0; e < V; ++e) y.v[e] += a.v[e];
    return;
  }
  for (int p0 = first; p0 < split; p0 += F) {
    Vec<V> a[F];
#pragma unroll
    for (int u = 0; u < F; ++u) a[u] = ldv<V, NT>(p + (size_t)min(p0 + u, split - 1) * plane + off);
#pragma unroll
    for (int u = 0; u < F; ++u)
      if (p0 + u < split)
#pragma unroll
        for (int e = 0; e < V; ++e) y.v[e] += a[u].v[e];
  }
}

// The same sum in two steps, in its order: the first F slabs are asked for, and added where the sum is needed.  No load waits
// for another: a loop over the slabs made all that was asked for before it arrive first, and a row that one workgroup works
// on pays a trip to memory, 0.7 us, for each such wait.  Only where a thread has one vector (AHEAD): rows of more want their
// registers for these, and asking ahead was slower (5 rows of 8192 gated 6.5 -> 8.5 us, of 20480 34 -> 43).
template <int V, int F = 8, bool AHEAD = true, bool NT = false>
struct Slabs {
  Vec<V> a[AHEAD ? F : 1];
  __device__ __forceinline__ void ask(const float* p, int split, int64_t plane, size_t off) {
    if constexpr (AHEAD) {
      a[0] = ldv<V, NT>(p + off);
      if (split == 1) return;
#pragma unroll
      for (int u = 1; u < F; ++u) a[u] = u < split ? ldv<V, NT>(p + u * plane + off) : zerov<V>();
    }
  }
  __device__ __forceinline__ void add(Vec<V>& y, const float* p, int split, int64_t plane, size_t off) const {
    if constexpr (AHEAD) {
#pragma unroll
      for (int e = 0; e < V; ++e) y.v[e] += a[0].v[e];
      if (split == 1) return;
#pragma unroll
      for (int u = 1; u < F; ++u)
        if (u < split)
#pragma unroll
          for (int e = 0; e < V; ++e) y.v[e] += a[u].v[e];
      add_slabs<V, F, NT>(y, p, split, plane, off, F);
    } else {
      add_slabs<V, F, NT>(y, p, split, plane, off);
    }
  }
};

// both steps at once
template <int V, int F, bool AHEAD, bool NT = false>
__device__ __forceinline__ void sum_slabs(Vec<V>& y, const float* p, int split, int64_t plane, size_t off) {
  Slabs<V, F, AHEAD, NT> s;
  s.ask(p, split, plane, off);
  s.add(y, p, split, plane, off);
}

// V columns of a product that leaves activations (split 0) or fp32 slabs, in the same two steps.
template <typename ACT, int V, int F = 8, bool AHEAD = true>
struct ColsIn {
  Slabs<V, F, AHEAD> s;
  __device__ __forceinline__ void ask(const void* p, int split, int64_t plane, int64_t o) {
    if constexpr (AHEAD) {
      if (split == 0) s.a[0] = ldv<V>(reinterpret_cast<const ACT*>(p) + o);
      else s.ask(reinterpret_cast<const float*>(p), split, plane, (size_t)o);
    }
  }
  __device__ __forceinline__ Vec<V> get(const void* p, int split, int64_t plane, int64_t o) const {
    if (split == 0) {
      if constexpr (AHEAD) return s.a[0];
      else return ldv<V>(reinterpret_cast<const ACT*>(p) + o);
    }
    Vec<V> y = zerov<V>();
    s.add(y, reinterpret_cast<const float*>(p), split, plane, (size_t)o);
    return y;
  }
};

}  // namespace

// Up to so many rows, no more than there are CUs, a row's time is its trips to memory; of more, what the registers let a CU hold.
constexpr int FEW_ROWS = 256;

// What a kernel keeps in mind of its number of rows: ROWS_FEW, and ROWS_PAST of so many that their stream no longer waits in the
// caches (256 MB) for its next use: it is read and written past them, and what others read next is not pushed out.  A row kernel
// has 10 to 12 bytes a value, x's 4, 4 of a product's and 2 for each of its 16-bit rows: from 88 MB of x they do not all stay (us of
// branch_norm / gated_norm on the same rows again and again, through the caches and past them: 4800 rows of 4096, 75 MB, 47 and 55 / 50
// and 60; 9600, 150 MB, 104 and 103 / 117 and 110).
enum { ROWS_SOME = 0, ROWS_FEW = 1, ROWS_PAST = 2 };
constexpr int64_t PAST_BYTES = 88ll << 20;      // of one stream

// NV, BT for rows of W channels in vectors of V
#define ROW_SHAPES(GO, vecs)           \
  if (vecs <= 64) GO(1, 64);           \
  else if (vecs <= 256) GO(1, 256);    \
  else if (vecs <= 512) GO(1, 512);    \
  else if (vecs <= 1024) GO(1, 1024);  \
  else if (vecs <= 4096) GO(4, 1024);  \
  else if (vecs <= 16384) GO(16, 1024); \
  else return -4
