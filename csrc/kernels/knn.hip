// Vector-search kernels: HBM-resident flat index scan + exact top-k, and the encoder's
// pooling/normalisation epilogue.
//
// Replaces the reference's vector-store hot paths: InMemoryVectorStore's python cosine loop
// (adapters/copilot_vectorstore/copilot_vectorstore/inmemory.py:106-119), FAISS IndexFlatL2 /
// IVFFlat (faiss_store.py:101-111,214) and Qdrant query_points (qdrant_store.py:371).
//
//   * cfc_knn_scan: scores[q][n] = <x_n, q>  (or -||x_n - q||^2) for <= 16 queries, one pass over
//     the bf16 index with MFMA 16x16x32 (queries are the B columns, index rows the A operand: from
//     the caches straight to registers, from memory in whole runs by way of LDS), and every block of
//     rows' best score beside them.
//   * cfc_topk_select: exact sorted top-k of scores with their block maxima: the k-th best block
//     maximum bounds the k-th best score from below, so only the blocks that reach it are looked at.
//   * cfc_knn_maxima, cfc_knn_blocks: the scan of many rows, which stores the best score of every 16 rows
//     alone, and the scores of the k blocks that the k best of these name.
//   * cfc_ivf_topk: scan and top-k of (query, probed list, chunk) work items from a device list-offset
//     table in one launch: each workgroup scores its chunk into LDS and selects the k best there;
//     the candidates are merged by cfc_topk_select.
//   * cfc_l2_normalize: rows -> unit length (+ fp32 norms), used on insert for cosine.
//   * cfc_pool: masked mean / CLS pooling over varlen sequences (+ optional L2 normalise):
//     the SentenceTransformer Pooling+Normalize modules.
#include "lds_ring.h"

namespace {

__device__ __forceinline__ bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ uint32_t f2key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key2f(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Sixteen rows' scores against all queries: X streams straight into the A operand, the queries are the B columns; a lane
// holds four rows' scores (4 (lane >> 4) ..) of query lane & 15.
template <int KC>  // KC = D / 32 MFMA k-steps
struct KnnRows {
  const uint16_t* X;
  int N;
  const float* xnorm2;       // optional: scores are -(x^2 + q^2 - 2 x q)
  const uint8_t* alive;      // optional row mask: scores of other rows are -inf
  bf16x8_t qf[KC];
  float qn;

  __device__ __forceinline__ void queries(const uint16_t* Q, const float* qnorm2, int nq) {
    const int col = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const bool qv = col < nq;
    const uint16_t* qr = Q + (size_t)(qv ? col : 0) * (KC * 32);
#pragma unroll
    for (int c = 0; c < KC; ++c)
      qf[c] = as_bf16x8(qv ? *reinterpret_cast<const uint4*>(qr + 32 * c + 8 * g) : make_uint4(0, 0, 0, 0));
    qn = (qnorm2 && qv) ? qnorm2[col] : 0.f;
  }
  // from what KnnFloats::put left in LDS
  __device__ __forceinline__ void queries(const char* lds, const float* n2, int nq, int row_bytes) {
    const int col = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const bool qv = col < nq;
    const char* qr = lds + (qv ? col : 0) * row_bytes;
#pragma unroll
    for (int c = 0; c < KC; ++c)
      qf[c] = as_bf16x8(qv ? *reinterpret_cast<const uint4*>(qr + 64 * c + 16 * g) : make_uint4(0, 0, 0, 0));
    qn = qv ? n2[col] : 0.f;
  }
  __device__ __forceinline__ void load(uint4* a, int r0) const {
    const int col = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const uint16_t* xr = X + (size_t)min(r0 + col, N - 1) * (KC * 32);
#pragma unroll
    for (int c = 0; c < KC; ++c) a[c] = *reinterpret_cast<const uint4*>(xr + 32 * c + 8 * g);
  }
  __device__ __forceinline__ f32x4_t score(const uint4* a, int r0) const {
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KC; ++c) v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[c]), qf[c], v, 0, 0, 0);
    return finish(v, r0);
  }
  // scores of the products
  __device__ __forceinline__ f32x4_t finish(f32x4_t v, int r0) const {
    const int rb = r0 + 4 * ((threadIdx.x & 63) >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = min(rb + i, N - 1);
      if (xnorm2) v[i] = -(xnorm2[row] + qn - 2.f * v[i]);
      if (alive && !alive[row]) v[i] = -INFINITY;
    }
    return v;
  }
  // The same from LDS: what word() brought there for the rows r0 ..
  __device__ __forceinline__ f32x4_t finish(f32x4_t v, int r0, const char* at) const {
    const int g = (threadIdx.x & 63) >> 4, rb = r0 + 4 * g;
    if (xnorm2) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(at + 16 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = -(x[i] + qn - 2.f * v[i]);
    }
    if (alive) {
      const uint4 a = *reinterpret_cast<const uint4*>(at + 64 + 16 * g);
      const uint32_t m[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!((m[i] >> (8 * ((uintptr_t)(alive + min(rb + i, N - 1)) & 3))) & 255)) v[i] = -INFINITY;
    }
    return v;
  }
  // lanes 0 .. 15: the norms of rows r0 .., 16 .. 31: the words that hold their bytes of the mask (of one that is not there, the
  // other's; the lanes after them alike)
  __device__ __forceinline__ const void* word(int r0) const {
    const int lane = threadIdx.x & 63, row = min(r0 + (lane & 15), N - 1);
    const bool mask = alive && (!xnorm2 || (lane & 16));
    return mask ? (const void*)((uintptr_t)(alive + row) & ~(uintptr_t)3) : (const void*)(xnorm2 + row);
  }
  // Largest key of the rows that there are, in all lanes of a query.
  __device__ __forceinline__ uint32_t best(const f32x4_t& v, int r0) const {
    const int rb = r0 + 4 * ((threadIdx.x & 63) >> 4);
    uint32_t m = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (rb + i < N) m = max(m, f2key(v[i]));
    m = max(m, (uint32_t)__shfl_xor((int)m, 16, 64));
    return max(m, (uint32_t)__shfl_xor((int)m, 32, 64));
  }
};

// Queries of floats to LDS, as l2_normalize_kernel takes them to memory, a wave a query, to the bit: the workgroups of a round each do
// so beside their first rows' way from memory, and a search has a launch less (us: 1 query of 20 k rows of 384 17.0 -> 14.3, of 27 k of
// 768 19.4 -> 16.3, 4 queries of 27 k of 384 17.8 -> 15.6, 1 of 1M 136 -> 133.7, 16 163 -> 159.6).  Asked for before the rows are, by four
// waves; their wait is one for the first rows, too, as that ahead of the first use of queries in bf16 is (taken to LDS before a row is asked
// for: 1.000 of the time, 20 k to 1M rows).  FROWS queries at most, for which there is room beside the rings.
template <int KC>
struct KnnFloats {
  static constexpr int FROWS = KC <= 16 ? 16 : 8, ROW = KC * 64 + 16, NV = (KC * 4 + 63) / 64, BYTES = FROWS * ROW;
  uint4 v[FROWS / 4][NV][2];
  __device__ __forceinline__ void ask(const float* q, int nq) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < FROWS / 4; ++i)
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const uint4* src = reinterpret_cast<const uint4*>(q + (size_t)min(w + 4 * i, nq - 1) * (KC * 32)) + 2 * min(lane + 64 * j, KC * 4 - 1);
        v[i][j][0] = src[0];
        v[i][j][1] = src[1];
      }
  }
  __device__ __forceinline__ void put(char* lds, float* n2, int nq, bool unit) const {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < FROWS / 4; ++i) {
      if (w + 4 * i >= nq) break;
      uint4 b[NV];
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const uint4 x = v[i][j][0], y = v[i][j][1];
        b[j] = make_uint4(pack2bf(__uint_as_float(x.x), __uint_as_float(x.y)), pack2bf(__uint_as_float(x.z), __uint_as_float(x.w)),
                          pack2bf(__uint_as_float(y.x), __uint_as_float(y.y)), pack2bf(__uint_as_float(y.z), __uint_as_float(y.w)));
        float f[8];
        unpack8(b[j], f);
        if (lane + 64 * j < KC * 4)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
      }
      ss = wave_sum(ss);
      if (lane == 0) n2[w + 4 * i] = ss;
      const float inv = ss > 0.f ? rsqrtf(ss) : 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        float f[8];
        unpack8(b[j], f);
        if (unit) {
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] *= inv;
        }
        if (lane + 64 * j < KC * 4) *reinterpret_cast<uint4*>(lds + (w + 4 * i) * ROW + 16 * (lane + 64 * j)) = pack8(f);
      }
    }
  }
};

// One wave scores a block of B rows (16, 32 or 64) against all queries.  Every lane holds four rows' scores of one query;
// they are stored as they lie and their largest key goes to bmax [nq][nb].  Nothing is selected here, so the pass is a plain
// stream over X: 1M x 384 bf16 with one query in 131 us (5.9 TB/s) where scoring 2048-row chunks into LDS and selecting in
// them took 172 us (4.5 TB/s; 489 workgroups, two on most CUs and one on the rest, the selecting wave alone at each one's end).
// MAXIMA: only the best score of every 16 rows is stored, to out [nq][ld] (B = 64).  A wave takes every gridDim-th block.
// FQ: the queries are floats, taken to unit length if `unit` (KC <= 16).
template <int KC, bool MAXIMA, bool FQ = false>
__global__ void __launch_bounds__(256) knn_scan_kernel(const uint16_t* __restrict__ X, const void* __restrict__ Q, int N,
                                                       int nq, const float* __restrict__ xnorm2,
                                                       const float* __restrict__ qnorm2, const uint8_t* __restrict__ alive,
                                                       float* __restrict__ out, size_t ld, uint32_t* __restrict__ bmax, int nb,
                                                       int B, bool unit) {
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const bool qv = col < nq;
  KnnRows<KC> rows{X, N, xnorm2, alive};
  uint4 a[KC <= 16 ? 2 : 1][KC];
  if constexpr (FQ) {
    static_assert(KC <= 16, "");
    __shared__ __attribute__((aligned(16))) char qs[KnnFloats<KC>::BYTES];
    __shared__ float n2[KnnFloats<KC>::FROWS];
    KnnFloats<KC> f;
    f.ask((const float*)Q, nq);
    rows.load(a[0], min((int)(blockIdx.x * 4 + (threadIdx.x >> 6)), nb - 1) * B);
    f.put(qs, n2, nq, unit);
    __syncthreads();
    rows.queries(qs, n2, nq, KnnFloats<KC>::ROW);
  } else {
    rows.queries((const uint16_t*)Q, qnorm2, nq);
  }
  bool first = FQ;
  const bool vec = (ld & 3) == 0 && ((uintptr_t)out & 15) == 0;
  for (int blk = blockIdx.x * 4 + (threadIdx.x >> 6); blk < nb; blk += gridDim.x * 4) {
    const int lo = blk * B, hi = min(N, lo + B);
    uint32_t best = 0u;
    auto take = [&](const uint4* a, int r0) {
      const f32x4_t v = rows.score(a, r0);
      const uint32_t m = rows.best(v, r0);
      if constexpr (MAXIMA) {
        if (r0 - lo == 16 * g) best = m;            // group g's
      } else {
        best = max(best, m);
        const int rb = r0 + 4 * g;
        if (!qv) return;
        float* o = out + col * ld + rb;
        if (rb + 3 < N && vec) {
          *reinterpret_cast<f32x4_t*>(o) = v;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (rb + i < N) o[i] = v[i];
        }
      }
    };
    if constexpr (KC <= 16) {          // the next 16 rows in flight under these (144 -> 131 us); wider rows fill the registers alone
      if (!first) rows.load(a[0], lo);
      first = false;
      for (int r0 = lo; r0 < hi; r0 += 32) {
        if (r0 + 16 < hi) rows.load(a[1], r0 + 16);
        take(a[0], r0);
        if (r0 + 32 < hi) rows.load(a[0], r0 + 32);
        if (r0 + 16 < hi) take(a[1], r0 + 16);
      }
    } else {
      for (int r0 = lo; r0 < hi; r0 += 16) {
        rows.load(a[0], r0);
        take(a[0], r0);
      }
    }
    if constexpr (MAXIMA) {
      if (qv && lo + 16 * g < hi) out[col * ld + 4 * blk + g] = key2f(best);
    } else if (bmax && g == 0 && qv) {
      bmax[(size_t)col * nb + blk] = best;
    }
  }
}

// The same scan for rows that come from memory.  A fragment's sixteen rows give 64 bytes each to a load, and memory serves
// that at 6.2 TB/s; whole runs, marked as read once, at 6.8 (768 MB of 16 x 768 bytes: 122 us, 129 marked; in runs 124, 112
// marked).  So rows go to LDS first, by LDS-DMA in pieces of 1 KB, a ring of R units per wave: 16 rows of KU k-steps.  Chunk c
// of row r lies at c ^ (r & 15) of its row's sixteen (through the pieces' source addresses), and sixteen rows' reads
// touch all banks.  No barrier: each wave waits for its own pieces alone.  Workgroups of one round, whose waves' streams
// run on from block to block.  Norms and the mask come with the rows, a word a lane: loads to registers, which hipcc knows nothing else to be
// in flight beside, waited for all units that had been asked for (us of squared distances / masked / both, fragments from memory, such
// loads, this: 1M rows of 512, 4 queries 219 / 217 / 229, 232 / 227 / 254, 182 / 181 / 181; 2M of 256 217 / 215 / 239, 235 / 240 / 271, 184 /
// 187 / 189; 1M of 384 164 / 162 / 178, this 134 / 134 / 135).
// us with the selection, fragments from memory -> this: 1M rows of 384 148 -> 132 (of 16 queries 181 -> 166), 3M 413 -> 374;
// of 768 values, whose fragments fill the registers alone, 500 k 165 -> 131, 100 k 38 -> 33, 5000 16.9 -> 15.7, of 1024 141 k 64 -> 56.
template <int KC>
struct KnnUnit {
  static constexpr int KU = KC <= 16 ? KC : KC % 12 == 0 ? 12 : KC % 16 == 0 ? 16 : KC % 8 == 0 ? 8 : 4;      // k-steps of a unit, and KB
  static constexpr int R = KU > 12 ? 2 : KU > 8 ? 3 : 4, NU = KC / KU;
  static_assert(KC % KU == 0 && KU % 4 == 0 && 4 * R * KU <= 160, "");
};

// WORDS: there are norms or a mask.  FQ: the queries are floats, as above
template <int KC, bool MAXIMA, bool WORDS, bool FQ>
__device__ __forceinline__ void knn_stream(const uint16_t* __restrict__ X, const void* __restrict__ Q, int N, int nq,
                                           const float* __restrict__ xnorm2, const float* __restrict__ qnorm2,
                                           const uint8_t* __restrict__ alive, float* __restrict__ out, size_t ld,
                                           uint32_t* __restrict__ bmax, int nb, int B, bool unit) {
  constexpr int KU = KnnUnit<KC>::KU, R = KnnUnit<KC>::R, NU = KnnUnit<KC>::NU, UB = KU * 1024;
  __shared__ __attribute__((aligned(16))) char kn_smem[4 * R * (UB + (WORDS ? 256 : 0))];      // rings, then those of norms and masks
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), stride = gridDim.x * 4;
  const bool qv = col < nq;
  KnnRows<KC> rows{X, N, xnorm2, alive};
  KnnFloats<KC> f;
  if constexpr (FQ) f.ask((const float*)Q, nq);
  else rows.queries((const uint16_t*)Q, qnorm2, nq);
  const bool vec = (ld & 3) == 0 && ((uintptr_t)out & 15) == 0;
  int blk = blockIdx.x * 4 + w;
  if (!FQ && blk >= nb) return;
  const char* ring = kn_smem + w * (R * UB);
  const uint32_t lds0 = lds_at(ring);
  const char* words = kn_smem + 4 * R * UB + w * (R * 256);
  const uint32_t words0 = lds_at(words);
  uint32_t voff[KU];
#pragma unroll
  for (int i = 0; i < KU; ++i) {
    const int p = 64 * i + lane, r = p / (4 * KU), c = p % (4 * KU);
    voff[i] = (uint32_t)(r * (KC * 64) + ((c & ~15) | ((c ^ r) & 15)) * 16);
  }
  // ---- what is asked for: unit iu of the 16 rows from ir0 of block iblk
  int iblk = blk, ir0 = blk * B, iu = 0, fill = 0, wfill = 0;
  auto issue = [&]() {
    if (iblk >= nb) return;
    if (WORDS && iu == 0) {
      ring_word_at(rows.word(ir0), words0 + wfill * 256);
      wfill = wfill + 1 == R ? 0 : wfill + 1;
    }
    const char* src = reinterpret_cast<const char*>(X) + (size_t)ir0 * (KC * 64) + iu * (KU * 64);
    if (ir0 + 16 <= N) {
#pragma unroll
      for (int i = 0; i < KU; ++i) ring_piece<true>(voff[i], src, lds0 + fill * UB + i * 1024);
    } else {                                          // past the last row: that one again
#pragma unroll
      for (int i = 0; i < KU; ++i) {
        const int r = (64 * i + lane) / (4 * KU);
        ring_piece<true>(voff[i] - (uint32_t)(max(0, ir0 + r - (N - 1)) * (KC * 64)), src, lds0 + fill * UB + i * 1024);
      }
    }
    fill = fill + 1 == R ? 0 : fill + 1;
    if (++iu == NU) {
      iu = 0;
      ir0 += 16;
      if (ir0 >= min(N, iblk * B + B)) {
        iblk += stride;
        ir0 = iblk * B;
      }
    }
  };
#pragma unroll
  for (int i = 0; i < R - 1; ++i) issue();
  if constexpr (FQ) {
    __shared__ __attribute__((aligned(16))) char qs[KnnFloats<KC>::BYTES];
    __shared__ float n2[KnnFloats<KC>::FROWS];
    f.put(qs, n2, nq, unit);
    __syncthreads();
    rows.queries(qs, n2, nq, KnnFloats<KC>::ROW);
  }
  int slot = 0, wslot = 0;
  for (; blk < nb; blk += stride) {
    const int lo = blk * B, hi = min(N, lo + B);
    uint32_t best = 0u;
    for (int r0 = lo; r0 < hi; r0 += 16) {
      f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        // this unit's pieces (scores stored since count too: it waits for no less), and the reads of the one before, whose
        // place the next one takes
        constexpr int LATER = KU * (R - 2);
        if (iblk >= nb) ring_wait<0>();
        else if (NU == 1 && WORDS) ring_wait<LATER + R - 2>();       // (more units a row: a word of the next rows, too, now and then)
        else ring_wait<LATER>();
        issue();
        const char* img = ring + slot * UB + col * (KU * 64);
#pragma unroll
        for (int c = 0; c < KU; ++c) {
          const int ch = 4 * c + g;
          const uint4 a = *reinterpret_cast<const uint4*>(img + ((ch & ~15) | ((ch ^ col) & 15)) * 16);
          v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), rows.qf[u * KU + c], v, 0, 0, 0);
        }
        slot = slot + 1 == R ? 0 : slot + 1;
      }
      if constexpr (WORDS) {
        v = rows.finish(v, r0, words + wslot * 256);
        wslot = wslot + 1 == R ? 0 : wslot + 1;
      }
      const uint32_t m = rows.best(v, r0);
      if constexpr (MAXIMA) {
        if (r0 - lo == 16 * g) best = m;            // group g's
      } else {
        best = max(best, m);
        const int rb = r0 + 4 * g;
        if (qv) {
          float* o = out + col * ld + rb;
          if (rb + 3 < N && vec) {
            *reinterpret_cast<f32x4_t*>(o) = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (rb + i < N) o[i] = v[i];
          }
        }
      }
    }
    if constexpr (MAXIMA) {
      if (qv && lo + 16 * g < hi) out[col * ld + 4 * blk + g] = key2f(best);
    } else if (bmax && g == 0 && qv) {
      bmax[(size_t)col * nb + blk] = best;
    }
  }
}

template <int KC, bool MAXIMA, bool WORDS>
__global__ void __launch_bounds__(256, 1) knn_stream_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ Q, int N,
                                                            int nq, const float* __restrict__ xnorm2,
                                                            const float* __restrict__ qnorm2, const uint8_t* __restrict__ alive,
                                                            float* __restrict__ out, size_t ld, uint32_t* __restrict__ bmax, int nb,
                                                            int B) {
  knn_stream<KC, MAXIMA, WORDS, false>(X, Q, N, nq, xnorm2, qnorm2, alive, out, ld, bmax, nb, B, false);
}

template <int KC, bool WORDS>
__global__ void __launch_bounds__(256, 1) knn_stream_floats_kernel(const uint16_t* __restrict__ X, const float* __restrict__ Q, int N,
                                                                   int nq, const float* __restrict__ xnorm2,
                                                                   const uint8_t* __restrict__ alive, float* __restrict__ out,
                                                                   size_t ld, uint32_t* __restrict__ bmax, int nb, int B, bool unit) {
  knn_stream<KC, false, WORDS, true>(X, Q, N, nq, xnorm2, nullptr, alive, out, ld, bmax, nb, B, unit);
}

// The scores of `kb` blocks of 16 rows per query (blocks [nq][kb], in any order) into out [nq][16 kb] and their rows into
// ids, blocks in rising order, with their largest keys in bmax [nq][kb]; past the last row the lowest NaN.  A wave per block.
template <int KC>
__global__ void __launch_bounds__(256) knn_blocks_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ Q, int N,
                                                         int nq, const float* __restrict__ xnorm2,
                                                         const float* __restrict__ qnorm2, const uint8_t* __restrict__ alive,
                                                         const int64_t* __restrict__ blocks, int kb, int64_t row0,
                                                         float* __restrict__ out, int64_t* __restrict__ ids,
                                                         uint32_t* __restrict__ bmax) {
  const int lane = threadIdx.x & 63, j = blockIdx.x * 4 + (threadIdx.x >> 6), q = blockIdx.y;
  if (j >= kb) return;
  const int64_t mine = blocks[(size_t)q * kb + j];
  const int r0 = (int)mine * 16, rb = r0 + 4 * (lane >> 4);
  KnnRows<KC> rows{X, N, xnorm2, alive};
  rows.queries(Q, qnorm2, nq);
  uint4 a[KC];
  rows.load(a, r0);
  int rank = 0;
  for (int i = lane; i < (kb + 63) / 64 * 64; i += 64) rank += __popcll(__ballot(i < kb && blocks[(size_t)q * kb + min(i, kb - 1)] < mine));
  const f32x4_t v = rows.score(a, r0);
  const uint32_t m = rows.best(v, r0);
  if ((lane & 15) != q) return;
  const size_t to = (size_t)q * kb + rank;
  if (lane < 16) bmax[to] = m;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = 4 * (lane >> 4) + i;
    out[16 * to + at] = rb + i < N ? v[i] : key2f(0u);
    ids[16 * to + at] = rb + i < N ? row0 + rb + i : -1;
  }
}

// ------------------------------------------------------------------ exact top-k
// Largest key of every B consecutive scores: one wave per block, grid (ceil(nb / 4), nq).
__global__ void __launch_bounds__(256) block_max_kernel(const float* __restrict__ in, int n, size_t ld, int B, uint32_t* __restrict__ bmax,
                                                        int nb) {
  const int lane = threadIdx.x & 63, blk = blockIdx.x * 4 + (threadIdx.x >> 6), qi = blockIdx.y;
  if (blk >= nb) return;
  const float* src = in + (size_t)qi * ld;
  const int hi = (int)min((long)n, (long)(blk + 1) * B);
  uint32_t best = 0u;
  for (int i = blk * B + lane; i < hi; i += 64) best = max(best, f2key(src[i]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = max(best, (uint32_t)__shfl_xor((int)best, o, 64));
  if (lane == 0) bmax[(size_t)qi * nb + blk] = best;
}

constexpr int SEL_THREADS = 1024, SEL_WAVES = SEL_THREADS / 64;
constexpr int SEL_BLOCKS = 16384;      // most blocks of a workgroup (16 maxima per thread)
constexpr int SEL_WIDEST = 64;         // most rows of a block: more scores than these hold go in segments
constexpr int SEL_CAP = 8192;          // candidates held
constexpr int SEL_STEP = 4096;         // scores looked at between two looks at the candidates' number
constexpr int SEL_K = 2048;            // most winners: SEL_K + SEL_STEP <= SEL_CAP

// Sum over the workgroup of a wave-uniform count: one barrier a call, the two halves of `red` in turn.
__device__ __forceinline__ int sel_count(int c, int (*red)[SEL_WAVES], int& turn) {
  if ((threadIdx.x & 63) == 0) red[turn][threadIdx.x >> 6] = c;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int i = 0; i < SEL_WAVES; ++i) t += red[turn][i];
  turn ^= 1;
  return t;
}

// The candidates cut to their kk largest (cnt > kk; all differ, as each holds its row); what all of those reach is returned.
// Any bound that exactly kk of them reach will do, so the bitwise search begins below the bits that all candidates share
// (of equal scores, the upper half) and ends where the count fits.
__device__ __forceinline__ uint64_t sel_cut(uint64_t* cand, int cnt, int kk, int (*red)[SEL_WAVES], int& turn, int* s_n,
                                            uint64_t (*bits)[SEL_WAVES]) {
  const int tid = threadIdx.x, lane = tid & 63;
  uint64_t e[SEL_CAP / SEL_THREADS], all = ~0ull, any = 0ull;
#pragma unroll
  for (int j = 0; j < SEL_CAP / SEL_THREADS; ++j) {
    const bool in = tid + j * SEL_THREADS < cnt;
    e[j] = in ? cand[tid + j * SEL_THREADS] : 0ull;
    any |= e[j];
    if (in) all &= e[j];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    all &= (uint64_t)__shfl_xor((unsigned long long)all, o, 64);
    any |= (uint64_t)__shfl_xor((unsigned long long)any, o, 64);
  }
  if (lane == 0) { bits[0][tid >> 6] = all; bits[1][tid >> 6] = any; }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SEL_WAVES; ++i) { all &= bits[0][i]; any |= bits[1][i]; }
  const int top = 63 - __clzll((long long)(all ^ any));     // they differ: two candidates or more
  uint64_t thr = top == 63 ? 0ull : any >> (top + 1) << (top + 1);
  for (int b = top; b >= 0; --b) {
    const uint64_t t = thr | (1ull << b);
    int c = 0;
#pragma unroll
    for (int j = 0; j < SEL_CAP / SEL_THREADS; ++j) c += __popcll(__ballot(e[j] >= t));
    c = sel_count(c, red, turn);
    if (c >= kk) thr = t;
    if (c == kk) break;
  }
  if (tid == 0) *s_n = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SEL_CAP / SEL_THREADS; ++j) {
    const bool p = e[j] != 0ull && e[j] >= thr;
    const uint64_t m = __ballot(p);
    int at = 0;
    if (lane == 0 && m) at = atomicAdd(s_n, __popcll(m));
    at = __shfl(at, 0, 64) + __popcll(m & ((1ull << lane) - 1ull));
    if (p) cand[at] = e[j];
  }
  __syncthreads();
  return thr;
}

// Sorted top-k of a query's n scores, one workgroup per query.  Largest first, the lower row first among
// equals.  bmax [nq][nb] holds the largest key of every B rows.  At least k blocks hold a score at or
// above the k-th best maximum, so no lower score is among the k best: the scores of the blocks that reach
// this bound (about k of them) are read, those at or above it kept, cut to k and ranked.  Where many blocks' maxima equal
// the bound (equal scores, or all but a few masked), the first of them do, as many as are missing: each holds a score of
// that value, at a lower row than any later block's.  Once cut, the k kept bound what may still come.  (300 of 1M: equal
// scores 48 us where looking at every block that reaches the bound took 5075, all but 100 masked 86 where it took 5586,
// others as before, 32; the radix passes 258, 189 and 176.)
// A chain of short steps: 13 us for 150 of 1M scores, where three rounds of radix histograms in LDS over
// 2048-row chunks' winners and a library sort took 120.
// ids (row stride ld, optional): what the rows are called; else row0 + row.
// grid (queries, segments): workgroup y selects from `seg` of the n scores, a whole number of blocks of B, into
// out [query][y].  One workgroup brings in 25 B/ns: more than 2^20 scores are shared out, and their winners selected from
// again (us for 2048 of 20M in one, here: 983, 320; rising scores 4435, 510; the radix passes 634 and 808).
__global__ void __launch_bounds__(SEL_THREADS) topk_select_kernel(const float* __restrict__ in, int n, size_t ld, int B, int seg,
                                                                  const uint32_t* __restrict__ bmax, int nb, int k,
                                                                  const int64_t* __restrict__ ids, int64_t row0,
                                                                  float* __restrict__ out_v, int64_t* __restrict__ out_i) {
  __shared__ uint64_t cand[SEL_CAP];
  __shared__ uint16_t list[SEL_BLOCKS];
  __shared__ int red[2][SEL_WAVES], s_n, s_list;
  __shared__ uint32_t s_lo[SEL_WAVES], s_hi[SEL_WAVES];
  __shared__ uint64_t bits[2][SEL_WAVES];
  __shared__ uint16_t ties[SEL_BLOCKS / SEL_THREADS][SEL_WAVES];
  const int tid = threadIdx.x, lane = tid & 63, qi = blockIdx.x;
  const uint64_t below = (1ull << lane) - 1ull;
  const int lb = 31 - __clz(B);                      // B is a power of two
  {
    const size_t first = (size_t)blockIdx.y * seg;
    in += qi * ld + first;
    if (ids) ids += qi * ld + first;
    row0 += first;
    bmax += (size_t)qi * nb + (first >> lb);
    out_v += ((size_t)qi * gridDim.y + blockIdx.y) * k;
    out_i += ((size_t)qi * gridDim.y + blockIdx.y) * k;
    n = (int)min((size_t)seg, n - first);
    nb = ((n - 1) >> lb) + 1;
  }
  int turn = 0;
  uint32_t key[SEL_BLOCKS / SEL_THREADS];
#pragma unroll
  for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
    const int i = tid + j * SEL_THREADS;
    key[j] = i < nb ? bmax[i] : 0u;
  }
  // a bound that k blocks reach, and not many more (none: every block is looked at); the search begins
  // below the bits that all maxima share
  uint32_t thr = 0;
  int reach = nb;                                    // blocks that do
  const int most = k + k / 4;
  auto blocks_at = [&](uint32_t t) {
    int c = 0;
#pragma unroll
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) c += __popcll(__ballot(key[j] >= t));
    return c;
  };
  if (nb >= SEL_THREADS && k <= SEL_THREADS / 4) {
    // What k threads' best blocks reach will do if not many more blocks do: few of the k best share one of 1024 threads, of 256
    // about 40 do, which `most` leaves room for; of more it would not.  One wave looks at the threads' best, without a barrier
    // a bit (15 625 blocks, k 150: 6.2 -> 3.9 us; 1 250 blocks, k 20: 4.4 -> 2.9).
    uint32_t best = 0u;
#pragma unroll
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) best = max(best, key[j]);
    uint32_t* bests = reinterpret_cast<uint32_t*>(cand);
    bests[tid] = best;
    __syncthreads();
    if (tid < 64) {
      uint32_t e[SEL_WAVES], lo = ~0u, hi = 0u;
#pragma unroll
      for (int j = 0; j < SEL_WAVES; ++j) {
        e[j] = bests[64 * j + lane];
        lo = min(lo, e[j]);
        hi = max(hi, e[j]);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
      }
      uint32_t t = hi;
      if (lo != hi) {
        const int top = 31 - __clz(lo ^ hi);
        t = top == 31 ? 0u : hi >> (top + 1) << (top + 1);
        for (int b = top; b >= 0; --b) {
          const uint32_t x = t | (1u << b);
          int c = 0;
#pragma unroll
          for (int j = 0; j < SEL_WAVES; ++j) c += __popcll(__ballot(e[j] >= x));
          if (c >= k) t = x;
          if (c >= k && c <= k + k / 16) break;
        }
      }
      if (lane == 0) s_lo[0] = t;
    }
    __syncthreads();
    thr = s_lo[0];
    reach = sel_count(blocks_at(thr), red, turn);
  }
  if (nb > k && reach > most) {
    uint32_t lo = ~0u, hi = 0u;
#pragma unroll
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
      if (tid + j * SEL_THREADS < nb) lo = min(lo, key[j]);
      hi = max(hi, key[j]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
      hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
    }
    __syncthreads();
    if (lane == 0) { s_lo[tid >> 6] = lo; s_hi[tid >> 6] = hi; }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SEL_WAVES; ++i) { lo = min(lo, s_lo[i]); hi = max(hi, s_hi[i]); }
    reach = nb;
    if (lo == hi) {
      thr = hi;
    } else {
      const int top = 31 - __clz(lo ^ hi);
      thr = top == 31 ? 0u : hi >> (top + 1) << (top + 1);
      for (int b = top; b >= 0; --b) {
        const uint32_t t = thr | (1u << b);
        const int c = sel_count(blocks_at(t), red, turn);
        if (c >= k) thr = t, reach = c;
        if (c >= k && c <= most) break;
      }
    }
  }
  if (nb > k && reach > most) {                      // thr is the k-th best maximum itself; seldom so: read again, not unrolled
    int c = 0;
#pragma unroll 1
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
      const int i = tid + j * SEL_THREADS;
      const uint32_t x = i < nb ? bmax[i] : 0u;
      const uint64_t m = __ballot(i < nb && x == thr);
      if (lane == 0) ties[j][tid >> 6] = (uint16_t)__popcll(m);
      c += __popcll(__ballot(x > thr));
    }
    const int missing = k - sel_count(c, red, turn);
    uint32_t drop = 0;                               // bit j: block j of this thread is not looked at
    int before = 0;                                  // ties in lower blocks
#pragma unroll 1
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
      const int at = tid + j * SEL_THREADS;
      const bool tie = at < nb && bmax[at] == thr;
      int mine = before + __popcll(__ballot(tie) & below);
#pragma unroll 1
      for (int i = 0; i < SEL_WAVES; ++i) {
        if (i < tid >> 6) mine += ties[j][i];
        before += ties[j][i];
      }
      if (tie && mine >= missing) drop |= 1u << j;
    }
#pragma unroll
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) key[j] = drop >> j & 1 ? 0u : key[j];
  }
  if (tid == 0) { s_n = 0; s_list = 0; }
  __syncthreads();
  {
    uint64_t m[SEL_BLOCKS / SEL_THREADS];
    int mine = 0;
#pragma unroll
    for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
      m[j] = __ballot(tid + j * SEL_THREADS < nb && key[j] >= thr);
      mine += __popcll(m[j]);
    }
    if (mine) {
      int at = 0;
      if (lane == 0) at = atomicAdd(&s_list, mine);
      at = __shfl(at, 0, 64);
#pragma unroll
      for (int j = 0; j < SEL_BLOCKS / SEL_THREADS; ++j) {
        if (m[j] >> lane & 1) list[at + __popcll(m[j] & below)] = (uint16_t)(tid + j * SEL_THREADS);
        at += __popcll(m[j]);
      }
    }
  }
  __syncthreads();
  const long total = (long)s_list << lb;             // scores to look at, four neighbours per thread
  const float* src = in;
  const bool vec = ((uintptr_t)in & 15) == 0;
  auto place = [&](long at) { return at < total ? ((int)list[at >> lb] << lb) + (int)(at & (B - 1)) : n; };
  auto load = [&](int row) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (vec && row + 3 < n) {
      x = *reinterpret_cast<const float4*>(src + row);
    } else {
      if (row < n) x.x = src[row];
      if (row + 1 < n) x.y = src[row + 1];
      if (row + 2 < n) x.z = src[row + 2];
      if (row + 3 < n) x.w = src[row + 3];
    }
    return x;
  };
  int row = place(4 * tid);
  float4 x = load(row);
  uint64_t floor = (uint64_t)thr << 32;               // no lower candidate is among the k best
  for (long s0 = 0; s0 < total; s0 += SEL_STEP) {
    const int row1 = place(s0 + SEL_STEP + 4 * tid);
    const float4 x1 = load(row1);                     // the next step's, under this one's work
    const float v[4] = {x.x, x.y, x.z, x.w};
    uint64_t e[4], m[4];
    int mine = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      e[u] = ((uint64_t)f2key(v[u]) << 32) | (0xffffffffu - (uint32_t)(row + u));
      m[u] = __ballot(row + u < n && e[u] >= floor);
      mine += __popcll(m[u]);
    }
    if (mine) {
      int at = 0;
      if (lane == 0) at = atomicAdd(&s_n, mine);
      at = __shfl(at, 0, 64);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (m[u] >> lane & 1) cand[at + __popcll(m[u] & below)] = e[u];
        at += __popcll(m[u]);
      }
    }
    row = row1;
    x = x1;
    __syncthreads();
    const int cnt = s_n;
    __syncthreads();
    // the next step might not fit; at the end, no more than the ranking takes.  One place for both: twice in the way, the cut's
    // code costs every call 0.6 us
    if (cnt > (s0 + SEL_STEP < total ? SEL_CAP - SEL_STEP : max(k, SEL_THREADS))) floor = sel_cut(cand, cnt, k, red, turn, &s_n, bits);
  }
  const int cnt = s_n;                                // at least min(k, n)
  const int share = cnt <= SEL_THREADS / 4 ? 2 : 0;   // few candidates: four threads count for one (173 of them: 3.1 -> 1.6 us)
  for (int i = tid >> share; i < cnt; i += SEL_THREADS >> share) {
    const uint64_t e = cand[i];
    int rank = 0;
    if (!share) {                                     // a loop of its own: in steps of 1 << share its reads were one by one (150 best of 1000: 44 us, so 34)
#pragma unroll 4
      for (int j = 0; j < cnt; ++j) rank += cand[j] > e;
    } else {
#pragma unroll 4
      for (int j = tid & 3; j < cnt; j += 4) rank += cand[j] > e;
      rank += __shfl_xor(rank, 1, 64);
      rank += __shfl_xor(rank, 2, 64);
    }
    if (rank >= k || (tid & ((1 << share) - 1))) continue;
    const uint32_t r = 0xffffffffu - (uint32_t)e;
    out_v[rank] = key2f((uint32_t)(e >> 32));
    out_i[rank] = ids ? ids[r] : row0 + r;
  }
}

// ------------------------------------------------------------------ IVF: fused scan + top-k
constexpr int KT_ROWS = 1024;   // rows per workgroup chunk (scores [nqb][KT_ROWS] fp32 in LDS)

// Wave-level exact top-k of sc[0..len) (LDS, len <= KT_ROWS): every lane holds 16 keys in
// registers (row lane + 64 j); the k-th largest key is found bit by bit, MSB first, from wave-wide
// counts of keys >= the candidate (32 rounds of 16 compare-ballot-popcounts, all in SGPRs/VALU) --
// no LDS: a radix histogram's atomics serialise here because one chunk's scores share their top
// key bytes, and a shuffle-tree sum pays an LDS round trip per level.
// Writes exactly k slots (ov/oi; -inf / -1 padding when len < k).
template <int ROWS>
__device__ __forceinline__ void wave_topk(const float* sc, int len, int k, int64_t row0, float* ov, int64_t* oi) {
  const int lane = threadIdx.x & 63;
  const int kk = min(k, len);
  uint32_t key[ROWS / 64];
#pragma unroll
  for (int j = 0; j < ROWS / 64; ++j) {
    const int i = lane + 64 * j;
    key[j] = i < len ? f2key(sc[i]) : 0u;
  }
  uint32_t thr = 0;
  if (kk > 0) {
    for (int b = 31; b >= 0; --b) {
      const uint32_t cand = thr | (1u << b);
      int c = 0;
#pragma unroll
      for (int j = 0; j < ROWS / 64; ++j) c += __popcll(__ballot(key[j] >= cand));
      if (c >= kk) thr = cand;                 // wave-uniform decision
    }
  }
  int gt = 0;
#pragma unroll
  for (int j = 0; j < ROWS / 64; ++j) gt += __popcll(__ballot(key[j] > thr));
  const uint32_t n_gt = (uint32_t)gt;
  const uint32_t need = (uint32_t)kk - n_gt;   // keys == thr to take (>= 1 when kk > 0)
  uint32_t base_gt = 0, base_eq = 0;
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int j = 0; j < ROWS / 64; ++j) {
    const int i = lane + 64 * j;
    const bool g = kk > 0 && i < len && key[j] > thr, e = kk > 0 && i < len && key[j] == thr;
    const uint64_t bg = __ballot(g), be = __ballot(e);
    int slot = -1;
    if (g) slot = (int)(base_gt + __popcll(bg & below));
    else if (e) {
      const uint32_t q = base_eq + __popcll(be & below);
      if (q < need) slot = (int)(n_gt + q);
    }
    if (slot >= 0) {
      ov[slot] = key2f(key[j]);
      oi[slot] = row0 + i;
    }
    base_gt += __popcll(bg);
    base_eq += __popcll(be);
  }
  for (int s2 = kk + lane; s2 < k; s2 += 64) { ov[s2] = -INFINITY; oi[s2] = -1; }
}

// Work item = a chunk of <= KT_ROWS consecutive rows of a probed list and its query: blockIdx.x =
// (q * nprobe + j) * maxc + c -> list probe[q][j], its chunk c.  out_v/out_i: [nq][nslots][k].
template <int KC>
__global__ void __launch_bounds__(256) ivf_topk_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ Q,
                                                       const float* __restrict__ xnorm2,
                                                       const float* __restrict__ qnorm2,
                                                       const uint8_t* __restrict__ alive, int k,
                                                       const int32_t* __restrict__ probe, int nprobe, int maxc,
                                                       const int64_t* __restrict__ list_off, int nslots,
                                                       float* __restrict__ out_v, int64_t* __restrict__ out_i) {
  constexpr int D = KC * 32, ROWS = KT_ROWS, nqb = 1;
  __shared__ float sc[ROWS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qc = blockIdx.x % maxc, qj = blockIdx.x / maxc;
  const int q0 = qj / nprobe, slot = (qj % nprobe) * maxc + qc, l = probe[qj];
  const int lo = (int)list_off[l] + qc * ROWS, hi = min((int)list_off[l + 1], lo + ROWS);
  const int len = max(0, hi - lo);
  if (len > 0) {
    const int col = lane & 15, g = lane >> 4;
    const bool qv = col < nqb;
    bf16x8_t qf[KC];
    const uint16_t* qr = Q + (size_t)(q0 + (qv ? col : 0)) * D;
#pragma unroll
    for (int c = 0; c < KC; ++c)
      qf[c] = as_bf16x8(qv ? *reinterpret_cast<const uint4*>(qr + 32 * c + 8 * g) : make_uint4(0, 0, 0, 0));
    const float qn = (qnorm2 && qv) ? qnorm2[q0 + col] : 0.f;
    const int ngroups = (len + 15) / 16;
    for (int grp = w; grp < ngroups; grp += 4) {
      const int r0 = lo + grp * 16;
      const int r = min(r0 + col, hi - 1);
      const uint16_t* xr = X + (size_t)r * D;
      uint4 a[KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) a[c] = *reinterpret_cast<const uint4*>(xr + 32 * c + 8 * g);
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[c]), qf[c], acc, 0, 0, 0);
      if (qv) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = r0 + 4 * g + i;
          if (row < hi) {
            float v = acc[i];
            if (xnorm2) v = -(xnorm2[row] + qn - 2.f * v);
            if (alive && !alive[row]) v = -INFINITY;
            sc[row - lo] = v;
          }
        }
      }
    }
  }
  __syncthreads();
  if (w == 0) {
    const size_t o = ((size_t)q0 * nslots + slot) * k;
    wave_topk<ROWS>(sc, len, k, lo, out_v + o, out_i + o);
  }
}

// Rows of bf16, or of floats that are rounded to bf16 first (queries: a launch that took them there alone was 4 us of a
// search of a million rows in 154), to unit length; `as_is`: only rounded.
template <typename T>
__global__ void __launch_bounds__(256) l2_normalize_kernel(uint16_t* __restrict__ out, const T* __restrict__ in,
                                                           float* __restrict__ norms2, int dim, bool as_is) {
  __shared__ float red[16];
  const int row = blockIdx.x;
  const int nvec = dim / 8;
  const uint4* src = reinterpret_cast<const uint4*>(in + (size_t)row * dim);
  auto load = [&](int c) {
    if constexpr (sizeof(T) == 2) {
      return src[c];
    } else {
      const uint4 a = src[2 * c], b = src[2 * c + 1];
      return make_uint4(pack2bf(__uint_as_float(a.x), __uint_as_float(a.y)), pack2bf(__uint_as_float(a.z), __uint_as_float(a.w)),
                        pack2bf(__uint_as_float(b.x), __uint_as_float(b.y)), pack2bf(__uint_as_float(b.z), __uint_as_float(b.w)));
    }
  };
  float ss = 0.f;
  for (int c = threadIdx.x; c < nvec; c += blockDim.x) {
    float v[8];
    unpack8(load(c), v);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += v[j] * v[j];
  }
  ss = block_sum(ss, red);
  if (norms2 && threadIdx.x == 0) norms2[row] = ss;
  const float inv = as_is ? 1.f : ss > 0.f ? rsqrtf(ss) : 0.f;
  if (!out) return;
  uint4* dst = reinterpret_cast<uint4*>(out + (size_t)row * dim);
  for (int c = threadIdx.x; c < nvec; c += blockDim.x) {
    float v[8];
    unpack8(load(c), v);
    if (!as_is) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= inv;
    }
    dst[c] = pack8(v);
  }
}

// grid = nseq, block = 256. mode 0: masked mean over the sequence's tokens; 1: CLS (first
// token); 2: unmasked mean over a fixed padded length (HF provider parity,
// huggingface_provider.py:101) -- identical to 0 for packed varlen input.
// A thread sums V neighbouring columns of every R-th token, R = 256 / (dim / V) groups of rows beside each
// other, four tokens' loads in flight: 365 texts of 180 tokens x 384 in 14 us, where a thread per column and
// one two-byte load after the other took 184.
template <int V>
__global__ void __launch_bounds__(256) pool_kernel(float* __restrict__ out_f32, uint16_t* __restrict__ out_bf16,
                                                   const uint16_t* __restrict__ hidden,
                                                   const int32_t* __restrict__ cu_seqlens, int dim, int mode,
                                                   int normalize) {
  __shared__ float red[16];
  extern __shared__ __attribute__((aligned(16))) float acc[];  // [R][dim] floats
  const int s = blockIdx.x;
  const int beg = cu_seqlens[s], len = cu_seqlens[s + 1] - beg;
  const int cnt = mode == 1 ? min(len, 1) : len;
  const int nvec = dim / V, R = max(1, 256 / nvec);
  const uint16_t* src = hidden + (size_t)beg * dim;
  for (int id = threadIdx.x; id < R * nvec; id += 256) {
    const int r = id / nvec, c = id - r * nvec;
    float sum[V];
#pragma unroll
    for (int j = 0; j < V; ++j) sum[j] = 0.f;
    for (int t = r; t < cnt; t += 4 * R) {
      if constexpr (V == 8) {
        uint4 x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const uint4*>(src + (size_t)min(t + u * R, cnt - 1) * dim + 8 * c);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float f[8];
          unpack8(x[u], f);
#pragma unroll
          for (int j = 0; j < 8; ++j) sum[j] += t + u * R < cnt ? f[j] : 0.f;
        }
      } else {
        for (int u = 0; u < 4; ++u)
          if (t + u * R < cnt) sum[0] += bf2f(src[(size_t)(t + u * R) * dim + c]);
      }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) acc[r * dim + V * c + j] = sum[j];
  }
  __syncthreads();
  float ss = 0.f;
  for (int d = threadIdx.x; d < dim; d += 256) {
    float v = 0.f;
    for (int r = 0; r < R; ++r) v += acc[r * dim + d];
    v = cnt > 0 ? v / (float)cnt : 0.f;
    acc[d] = v;                       // this thread's column alone
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float inv = (normalize && ss > 0.f) ? rsqrtf(ss) : 1.f;
  for (int d = threadIdx.x; d < dim; d += 256) {
    const float v = acc[d] * inv;
    if (out_f32) out_f32[(size_t)s * dim + d] = v;
    if (out_bf16) out_bf16[(size_t)s * dim + d] = f2bf(v);
  }
}

}  // namespace

#define KNN_DIMS(KS)    \
  switch (dim / 32) {   \
    case 4: KS(4);      /* 128 */ \
    case 8: KS(8);      /* 256 */ \
    case 12: KS(12);    /* 384 (MiniLM, bge-small) */ \
    case 16: KS(16);    /* 512 */ \
    case 24: KS(24);    /* 768 (bge-base, mpnet) */ \
    case 32: KS(32);    /* 1024 (bge-large) */ \
    default: return -2; \
  }

// Rows per block for the top-k of n scores: as small as the select kernel's number of blocks allows.
CFC_API int cfc_topk_block(int n) {
  int b = 16;
  while (b < SEL_WIDEST && (long)b * SEL_BLOCKS < n) b *= 2;
  return b;
}

// Scores per workgroup of the select kernel: all n, or equal shares of whole blocks.
CFC_API int cfc_topk_segment(int n) {
  constexpr int most = SEL_BLOCKS * SEL_WIDEST;
  if (n <= most) return n;
  const int parts = (n - 1) / most + 1;
  return ((n - 1) / parts / SEL_WIDEST + 1) * SEL_WIDEST;
}

// Where rows of up to 512 values come from the 256 MB that the chip caches, workgroups of one round (two a CU) take all
// blocks, and no last round is nearly empty: 50 k rows of 384 9.8 -> 8.6 us, 100 k of 16 queries 21.8 -> 16.5, 200 k 28.4
// -> 24.7; 300 k 36.2 -> 38.2 (from memory a workgroup per four blocks reads faster).
constexpr long KNN_ROUND_BYTES = 160l << 20;
constexpr int KNN_ROUND = 512;
// More than the cache holds goes by knn_stream_kernel, which marks rows as read once (MB of 384 values, us: 230 46 -> 48, 260
// 50 -> 52, 290 58.5 -> 56.5, 330 69 -> 63; of 256 270 56.5 -> 55, 300 58 -> 58.6, 400 84 -> 74), and all rows of more than 512
// values; rows of 128, a quarter of a unit each, do not (200 MB 44 -> 65, 400 97 -> 127).
constexpr long KNN_STREAM_BYTES = 288l << 20;
constexpr int KNN_CUS = 256;
// LDS-DMA's sources are whole sixteens of bytes; rows that lie otherwise come to registers
bool knn_aligned(const void* X) { return ((uintptr_t)X & 15) == 0; }

#define KNN_ARGS(OUT, B) (const uint16_t*)X, (const uint16_t*)Q, N, nq, xnorm2, qnorm2, alive, OUT, (size_t)ld, B

// floats: where Q holds floats the scan takes them itself, if its workgroups are no more than a round (each takes the queries to LDS) and
// these fit beside the rings; where it does not, *floats is cleared and nothing launched
static int knn_scan_go(const void* X, const void* Q, int N, int nq, int dim, const float* xnorm2, const float* qnorm2,
                       const uint8_t* alive, float* out, long ld, uint32_t* bmax, long room, hipStream_t stream, bool* floats, bool unit) {
  if (nq < 1 || nq > 16 || dim % 32 != 0 || N <= 0 || ld < N) return -1;
  const int B = cfc_topk_block(N), nb = (N - 1) / B + 1;
  if (bmax && (long)nq * nb > room) return -1;
  const int all = (nb + 3) / 4;
  const long bytes = (long)N * dim * 2;
#define ST(KC, W)                                                                                                                      \
  if (floats) knn_stream_floats_kernel<KC, W><<<min(all, KNN_CUS), 256, 0, stream>>>((const uint16_t*)X, (const float*)Q, N, nq, xnorm2, \
                                                                                     alive, out, (size_t)ld, bmax, nb, B, unit);        \
  else knn_stream_kernel<KC, false, W><<<min(all, KNN_CUS), 256, 0, stream>>>(KNN_ARGS(out, bmax), nb, B)
#define SC(KC, F) knn_scan_kernel<KC, false, F><<<grid, 256, 0, stream>>>(KNN_ARGS(out, bmax), nb, B, unit)
#define KS(KC)                                                                                         \
  {                                                                                                    \
    if constexpr (KC > 4)                                                                              \
      if (knn_aligned(X) && (KC > 16 || bytes > KNN_STREAM_BYTES)) {                                   \
        if (floats && nq > KnnFloats<KC>::FROWS) { *floats = false; return 0; }                        \
        if (xnorm2 || alive) { ST(KC, true); }                                                         \
        else { ST(KC, false); }                                                                        \
        break;                                                                                         \
      }                                                                                                \
    const int grid = KC <= 16 && bytes <= KNN_ROUND_BYTES ? min(all, KNN_ROUND) : all;                 \
    if constexpr (KC <= 16)                                                                            \
      if (floats && grid <= KNN_ROUND) { SC(KC, true); break; }                                        \
    if (floats) { *floats = false; return 0; }                                                         \
    SC(KC, false);                                                                                     \
    break;                                                                                             \
  }
  KNN_DIMS(KS)
#undef KS
#undef SC
#undef ST
  return CFC_CHECK_LAUNCH();
}

// Scores of rows [0, N) of X for nq queries into out [nq][ld], and the largest key of every cfc_topk_block(N) rows into
// bmax [nq][blocks] (null: not wanted), which has room for `room` of them.
CFC_API int cfc_knn_scan(const void* X, const void* Q, int N, int nq, int dim, const float* xnorm2, const float* qnorm2,
                         const uint8_t* alive, float* out, long ld, uint32_t* bmax, long room, hipStream_t stream) {
  return knn_scan_go(X, Q, N, nq, dim, xnorm2, qnorm2, alive, out, ld, bmax, room, stream, nullptr, false);
}

// The best score of every 16 rows of [0, N) of X for nq queries, into out [nq][ld].
CFC_API int cfc_knn_maxima(const void* X, const void* Q, int N, int nq, int dim, const float* xnorm2, const float* qnorm2,
                           const uint8_t* alive, float* out, long ld, hipStream_t stream) {
  if (nq < 1 || nq > 16 || dim % 32 != 0 || N <= 0 || ld < (N - 1) / 16 + 1) return -1;
  const int nb = (N - 1) / 64 + 1, all = (nb + 3) / 4;
#define KS(KC)                                                                                                              \
  if constexpr (KC > 4)                                                                                                     \
    if (knn_aligned(X)) {                                                                                                   \
      if (xnorm2 || alive) knn_stream_kernel<KC, true, true><<<min(all, KNN_CUS), 256, 0, stream>>>(KNN_ARGS(out, nullptr), nb, 64); \
      else knn_stream_kernel<KC, true, false><<<min(all, KNN_CUS), 256, 0, stream>>>(KNN_ARGS(out, nullptr), nb, 64);       \
      break;                                                                                                                \
    }                                                                                                                       \
  knn_scan_kernel<KC, true><<<all, 256, 0, stream>>>(KNN_ARGS(out, nullptr), nb, 64, false);                                       \
  break
  KNN_DIMS(KS)
#undef KS
#undef KNN_ARGS
  return CFC_CHECK_LAUNCH();
}

// Scores of kb blocks of 16 rows per query, for a cfc_topk_select over 16 kb: see knn_blocks_kernel.  Every block starts
// below N.
CFC_API int cfc_knn_blocks(const void* X, const void* Q, int N, int nq, int dim, const float* xnorm2, const float* qnorm2,
                           const uint8_t* alive, const int64_t* blocks, int kb, long row0, float* out, int64_t* ids,
                           uint32_t* bmax, hipStream_t stream) {
  if (nq < 1 || nq > 16 || dim % 32 != 0 || N <= 0 || kb < 1 || kb > (N - 1) / 16 + 1) return -1;
#define KS(KC) knn_blocks_kernel<KC><<<dim3((kb + 3) / 4, nq), 256, 0, stream>>>((const uint16_t*)X, (const uint16_t*)Q, N, nq, \
      xnorm2, qnorm2, alive, blocks, kb, row0, out, ids, bmax); break
  KNN_DIMS(KS)
#undef KS
  return CFC_CHECK_LAUNCH();
}

// Sorted top-k of every segment of in [nq][n] (row stride ld) -> out [nq][segments][k], k no more than a segment has.
// bmax [nq][ceil(n / B)], B = cfc_topk_block(n), with room for `room` maxima: those from cfc_knn_scan, or (fill) workspace
// that is filled here.
CFC_API int cfc_topk_select(const float* in, const int64_t* ids, int nq, int n, long ld, int k, uint32_t* bmax, long room,
                            int fill, long row0, float* out_v, int64_t* out_i, hipStream_t stream) {
  if (nq < 1 || n < 1 || k <= 0 || k > SEL_K || ld < n) return -1;
  const int B = cfc_topk_block(n), nb = (n - 1) / B + 1, seg = cfc_topk_segment(n), parts = (n - 1) / seg + 1;
  if ((long)nq * nb > room || k > n - (parts - 1) * seg) return -1;
  if (fill) block_max_kernel<<<dim3((nb + 3) / 4, nq), 256, 0, stream>>>(in, n, (size_t)ld, B, bmax, nb);
  topk_select_kernel<<<dim3(nq, parts), SEL_THREADS, 0, stream>>>(in, n, (size_t)ld, B, seg, bmax, nb, k, ids, row0, out_v, out_i);
  return CFC_CHECK_LAUNCH();
}

CFC_API int cfc_l2_normalize(void* out, const void* in, float* norms2, int rows, int dim, hipStream_t stream) {
  if (dim % 8 != 0) return -1;
  if (rows == 0) return 0;
  l2_normalize_kernel<<<rows, dim >= 2048 ? 256 : 64, 0, stream>>>((uint16_t*)out, (const uint16_t*)in, norms2, dim, false);
  return CFC_CHECK_LAUNCH();
}

// Queries of floats [rows][dim] to bf16, of unit length if `unit`, and the squared norms of the rounded ones (all 16-byte aligned).
CFC_API int cfc_knn_queries(void* out, const float* in, float* norms2, int unit, int rows, int dim, hipStream_t stream) {
  if (dim % 8 != 0 || rows < 1) return -1;
  l2_normalize_kernel<<<rows, dim >= 2048 ? 256 : 64, 0, stream>>>((uint16_t*)out, in, norms2, dim, !unit);
  return CFC_CHECK_LAUNCH();
}

// Workspace of cfc_knn_search: block maxima, queries in bf16, their norms and scores of whole fours a row, each at a whole line (scores
// at 16 bytes took 62.7 us for 6 queries of 200 k rows of 768, 61.5 at a line).
struct KnnRoom { int64_t q, n2, scores, bytes, ld, nb; };
static KnnRoom knn_room(int N, int nq, int dim) {
  const int64_t line = 512, ld = ((int64_t)N + 3) / 4 * 4, nb = (N - 1) / cfc_topk_block(N) + 1;
  auto up = [&](int64_t n) { return (n + line - 1) / line * line; };
  KnnRoom r{up(4 * nq * nb), 0, 0, 0, ld, nb};
  r.n2 = r.q + up((int64_t)nq * dim * 2);
  r.scores = r.n2 + up(4 * nq);
  r.bytes = r.scores + 4 * nq * ld;
  return r;
}
CFC_API int64_t cfc_knn_search_bytes(int N, int nq, int dim) { return N < 1 || nq < 1 || dim < 1 ? -1 : knn_room(N, nq, dim).bytes; }

// A flat search of floats q [nq][dim] (16-byte aligned) from end to end by one call, whose host takes as long as the GPU does for an
// index of up to some 100 k rows (20 k rows, 1 query: three calls 27.1 us, this 14.3): queries, scores, the k best of N rows
// that cfc_topk_select takes in one segment.  As cfc_knn_queries, cfc_knn_scan and cfc_topk_select; ws 16-byte aligned.
CFC_API int cfc_knn_search(const void* X, const float* q, int unit, int N, int nq, int dim, const float* xnorm2, const uint8_t* alive,
                           int k, long row0, void* ws, int64_t room, float* out_v, int64_t* out_i, hipStream_t stream) {
  if (nq < 1 || nq > 16 || N < 1 || dim < 1 || cfc_topk_segment(N) < N) return -1;
  const KnnRoom r = knn_room(N, nq, dim);
  if (room < r.bytes) return -1;
  char* const p = (char*)ws;
  float *const n2 = (float*)(p + r.n2), *const scores = (float*)(p + r.scores);
  bool floats = true;
  if (const int e = knn_scan_go(X, q, N, nq, dim, xnorm2, nullptr, alive, scores, r.ld, (uint32_t*)ws, nq * r.nb, stream, &floats, unit))
    return e;
  if (floats) return cfc_topk_select(scores, nullptr, nq, N, r.ld, k, (uint32_t*)ws, nq * r.nb, 0, row0, out_v, out_i, stream);
  if (const int e = cfc_knn_queries(p + r.q, q, n2, unit, nq, dim, stream)) return e;
  if (const int e = cfc_knn_scan(X, p + r.q, N, nq, dim, xnorm2, n2, alive, scores, r.ld, (uint32_t*)ws, nq * r.nb, stream)) return e;
  return cfc_topk_select(scores, nullptr, nq, N, r.ld, k, (uint32_t*)ws, nq * r.nb, 0, row0, out_v, out_i, stream);
}

CFC_API int cfc_pool(float* out_f32, void* out_bf16, const void* hidden, const int32_t* cu_seqlens, int nseq, int dim,
                     int mode, int normalize, hipStream_t stream) {
  if (nseq == 0) return 0;
  const bool vec = dim % 8 == 0 && (uintptr_t)hidden % 16 == 0;
  const int R = max(1, 256 / (vec ? dim / 8 : dim));
#define PL(V) pool_kernel<V><<<nseq, 256, R * dim * sizeof(float), stream>>>(out_f32, (uint16_t*)out_bf16, (const uint16_t*)hidden, \
                                                                           cu_seqlens, dim, mode, normalize)
  if (vec) PL(8);
  else PL(1);
#undef PL
  return CFC_CHECK_LAUNCH();
}

// rows per IVF list chunk (one workgroup each)
CFC_API int cfc_knn_topk_rows() { return KT_ROWS; }

// IVF: probe [nq][nprobe] list ids, list_off [nlist + 1] row offsets (rows grouped by list), maxc =
// max chunks of any list.  One launch of nq * nprobe * maxc workgroups; candidates out
// [nq][nprobe * maxc][k].
CFC_API int cfc_ivf_topk(const void* X, const void* Q, int N, int nq, int dim, const float* xnorm2,
                         const float* qnorm2, const uint8_t* alive, const int32_t* probe, int nprobe,
                         const int64_t* list_off, int maxc, int k, float* out_v, int64_t* out_i, hipStream_t stream) {
  if (nq < 1 || nprobe < 1 || maxc < 1 || dim % 32 != 0 || k < 1 || k > 256) return -1;
  const long blocks = (long)nq * nprobe * maxc;
  if (blocks > (1L << 30)) return -1;
#define KT(KC) ivf_topk_kernel<KC><<<(int)blocks, 256, 0, stream>>>((const uint16_t*)X, (const uint16_t*)Q, xnorm2, qnorm2, alive, k, \
      probe, nprobe, maxc, list_off, nprobe * maxc, out_v, out_i); break
  switch (dim / 32) {
    case 4: KT(4);
    case 8: KT(8);
    case 12: KT(12);
    case 16: KT(16);
    case 24: KT(24);
    case 32: KT(32);
    default: return -2;
  }
#undef KT
  return CFC_CHECK_LAUNCH();
}
