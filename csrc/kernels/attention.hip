// Attention kernels for gfx950 (CDNA4), bf16 in / fp32 accumulate on MFMA 16x16x32.
//
//   * paged decode attention (GQA, split-K over context partitions + LSE combine)
//   * varlen causal prefill attention over the paged KV cache (flash-style online softmax)
//   * varlen bidirectional encoder attention (BERT / MiniLM / BGE, head_dim 32 or 64)
//
// They replace the attention inside the engines the reference drives over HTTP
// (Ollama /api/generate: local_llm_summarizer.py:107; llama.cpp /completion:
// llamacpp_summarizer.py:108) and inside SentenceTransformer.encode
// (sentence_transformer_provider.py:93).  The reference itself has no kernels.
//
// Layout decisions (MI355X-first, not a CUDA translation):
//   * "Swapped" products: S^T = K . Q^T and O^T = V^T . P^T.  With the 16x16x32 C/D map
//     (col = lane&15, row = 4*(lane>>4)+i) every lane then owns ONE query column, so the
//     online-softmax max/sum are lane-local plus two xor-shuffles, and the S^T accumulator is
//     already the P^T B-operand of the next MFMA ("accumulator as the next operand").
//   * KV cache block = 32 tokens = one MFMA k-step.  K is stored [blk][kvh][32][D] (row = key),
//     V is stored TRANSPOSED in slot groups, [blk][kvh][4 groups g][D][8] (common.h kv_v_off), with
//     the keys of each block permuted so that slot 8g+j holds key perm(g,j) = (j<4 ? 4g+j : 16+4g+j-4).
//     That is exactly the key order a lane holds in its S^T registers, so the V^T A-operand is one
//     contiguous 16-byte load per lane (no LDS transpose, no ds_read_tr needed) in both decode
//     (straight from HBM) and prefill; and one decode token's V column dirties 16 cache lines
//     ([D][32] rows: 64), which is what its write costs the step.
//   * LDS tiles are XOR-swizzled for conflict-free ds_read_b128; the swizzles
//     were derived against the gfx950 ds_read_b128 lane groups {0-3,12-15,20-27}, ...
#include "lds_ring.h"
#include <limits.h>
#include <stdlib.h>

#include <type_traits>

namespace {

constexpr int KV_BS = 32;          // tokens per KV-cache block
constexpr float LOG2E = 1.4426950408889634f;
constexpr int DEC_ORDER_ROWS = 128;   // sequences that longest_first orders at most
constexpr int DEC_FUSED_ROWS = 4;     // sequences whose step with its rotation inside takes loads to registers, whatever their lengths
constexpr int DEC_ORDER_FROM = 1024;  // the longest context from which it does

__device__ __forceinline__ bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// P^T fragment for keys [32ks, 32ks+32): {p[2ks][0..3], p[2ks+1][0..3]} as bf16.
__device__ __forceinline__ bf16x8_t pack_p(const f32x4_t& a, const f32x4_t& b) {
  uint4 u;
  u.x = pack2bf(a[0], a[1]); u.y = pack2bf(a[2], a[3]);
  u.z = pack2bf(b[0], b[1]); u.w = pack2bf(b[2], b[3]);
  return as_bf16x8(u);
}

// ------------------------------------------------------------------------------------------
// Paged decode attention.
// grid = (P partitions, Hkv, B); block = 256 (4 waves).  Each wave walks the partition's KV
// blocks with stride 4, K/V fragments straight from HBM into VGPRs
// (no reuse for the LDS to serve), next block prefetched while the current one is in the MFMAs.
// The G = Hq/Hkv query heads of the kv-head share every K/V byte (GQA packing: the G heads are
// the MFMA's B columns).
// ------------------------------------------------------------------------------------------
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// 16-byte KV load; NT = non-temporal (streamed once per step: keep it out of the caches' LRU so the
// shared-prefix blocks and the weights stay resident)
template <bool NT>
__device__ __forceinline__ uint4 kv_load(const uint16_t* p) {
  if constexpr (NT) {
    const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
  } else {
    return *reinterpret_cast<const uint4*>(p);
  }
}

typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

// 8-byte load of 8 fp8 KV values (the FP8 cache's fragment)
template <bool NT>
__device__ __forceinline__ uint2 kv_load8(const uint8_t* p) {
  if constexpr (NT) {
    const u32x2_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p));
    return make_uint2(v.x, v.y);
  } else {
    return *reinterpret_cast<const uint2*>(p);
  }
}

// Raw KV fragment as loaded (bf16: 16 B; fp8: 8 B) and its bf16x8 MFMA operand.  The fp8 ->
// bf16 conversion happens at the MFMA, so a prefetched block's loads stay in flight.
template <bool F8> struct KvFrag { typedef uint4 raw; };
template <> struct KvFrag<true> { typedef uint2 raw; };
__device__ __forceinline__ bf16x8_t kv_operand(uint4 r) { return as_bf16x8(r); }
__device__ __forceinline__ bf16x8_t kv_operand(uint2 r) { return as_bf16x8(fp8x8_to_bf16x8(r)); }

// ROPE: the decode step's RoPE + KV write happens in the prologue (DecRope below): every workgroup
// ropes the G query heads it needs straight from the qkv projection output (bf16, or the decode
// GEMM's fp32 split-K slabs) into LDS, and the workgroup whose KV range holds the sequence's last
// block writes the new key / value into the cache first -- the separate rope_kv launch, its q
// round trip through HBM and its dependency edge disappear.  Same helpers (common.h) as
// rope_kv_kernel, so the cache bytes and q values are identical to the two-kernel path.
// Workgroup barrier that orders LDS only: global loads and stores issued before it stay in flight
// (__syncthreads waits for every outstanding vector-memory operation first).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Element e (0..7) of a bf16x8 fragment replaced by the bf16 bits h (register selects, no scratch).
__device__ __forceinline__ uint4 set_bf16(uint4 v, int e, uint32_t h) {
  const int wi = e >> 1;
  const bool hi = e & 1;
  auto put = [&](uint32_t x, int i) -> uint32_t {
    return i != wi ? x : hi ? ((x & 0xffffu) | (h << 16)) : ((x & 0xffff0000u) | h);
  };
  return make_uint4(put(v.x, 0), put(v.y, 1), put(v.z, 2), put(v.w, 3));
}

// {sequence, its context} of the one that has `rank` others before it, longest contexts first (of equal ones the first
// first): more workgroups than the chip holds at once start as others end, and a long one that starts last is waited for
// alone.  In the order that they have where the contexts are short or differ by no more than `least` sixteenths of the
// longest: the ranking, 0.5 us a workgroup, would be more than it saves.
// `lds`: ORDER_LDS bytes, free again when it returns.
constexpr int ORDER_LDS = (2 * DEC_ORDER_ROWS + 5) * 4;
template <int THREADS>
__device__ __forceinline__ int2 longest_first(const int32_t* __restrict__ ctx_lens, int B, int rank, int least, char* lds) {
  constexpr int SHARES = THREADS / DEC_ORDER_ROWS;    // threads of a sequence, each with a share of the others
  static_assert(SHARES == 1 || SHARES == 2, "");
  int* key = reinterpret_cast<int*>(lds);
  int *before = key + DEC_ORDER_ROWS, *ends = before + DEC_ORDER_ROWS, *found = ends + 4;
  const int t = threadIdx.x, s = t & (DEC_ORDER_ROWS - 1), n = ctx_lens[min(s, B - 1)];
  const int lo = wave_min_int(n), hi = -wave_min_int(-n);
  if (t < DEC_ORDER_ROWS) {
    key[t] = t < B ? (n << 8) + (255 - t) : -1;
    before[t] = 0;
    if ((t & 63) == 0) ends[t >> 5] = lo, ends[(t >> 5) + 1] = hi;
  }
  __syncthreads();
  const int4 e = *reinterpret_cast<const int4*>(ends);
  const int longest = max(e.y, e.w);
  int b = rank;
  if (__builtin_amdgcn_readfirstlane(longest >= DEC_ORDER_FROM && (longest - min(e.x, e.z)) * 16 > least * longest)) {
    const int own = key[s];
    int c = 0;
#pragma unroll 8
    for (int j = 0; j < DEC_ORDER_ROWS / SHARES; j += 4) {
      const int4 k = *reinterpret_cast<const int4*>(key + (t & DEC_ORDER_ROWS) / 2 + j);
      c += (k.x > own) + (k.y > own) + (k.z > own) + (k.w > own);
    }
    if constexpr (SHARES == 1) before[s] = c;
    else atomicAdd(before + s, c);
    __syncthreads();
    if (t < B && before[t] == rank) *found = t;
    __syncthreads();
    b = *found;
  }
  b = __builtin_amdgcn_readfirstlane(b);
  const int ctx = __builtin_amdgcn_readfirstlane(key[b] >> 8);
  __syncthreads();
  return make_int2(b, ctx);
}

struct DecRope {
  const uint16_t* qkv;     // [B, (Hq + 2 Hkv) D] bf16, or nullptr with part
  const float* part;       // [split, B, (Hq + 2 Hkv) D] fp32 split-K slabs
  int split;
  const int32_t* positions;
  const int32_t* slots;    // -1: no cache write
  const float* cos_sin;
  float inv_k, inv_v;
  int probe;               // timing ablations only (cfc_set_decode_rope_probe); 0 in production
};

// One KV block's K fragments (bf16: 8 x 16 B per lane; fp8: 4 x 16 B) and V^T fragments (8) of
// kv-head block `base` (elements), loaded nontemporal (NT) or through the caches.
template <bool NT, bool F8>
__device__ __forceinline__ void dec_load_blk(const void* kc, const void* vc, size_t base, int col, int g, uint4* kk,
                                             typename KvFrag<F8>::raw* vv) {
  constexpr int D = 128;
  if constexpr (F8) {
    const uint8_t* kb = reinterpret_cast<const uint8_t*>(kc) + base;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int pp = 0; pp < 2; ++pp)
        kk[st * 2 + pp] = kv_load<NT>(reinterpret_cast<const uint16_t*>(kb + (16 * st + col) * D + 64 * pp + 16 * g));
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      vv[dt] = kv_load8<NT>(reinterpret_cast<const uint8_t*>(vc) + base + kv_v_off(16 * dt + col, 8 * g, D));
  } else {
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        kk[st * 4 + c] = kv_load<NT>(reinterpret_cast<const uint16_t*>(kc) + base + (16 * st + col) * D + 32 * c + 8 * g);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      vv[dt] = kv_load<NT>(reinterpret_cast<const uint16_t*>(vc) + base + kv_v_off(16 * dt + col, 8 * g, D));
  }
}

// NT: the KV stream is read nontemporal (each block once per step, kept out of the caches' LRU) --
// except the first *shared_blocks blocks of every sequence (shared_blocks: device int, may be null):
// the prefix-cache blocks that every sequence of the batch maps to the SAME physical blocks (system
// prompt + template head, ~10 blocks of a 2.9k-token context).  Those go through L2 / MALL, so the
// 128 sequences' reads of them cost one HBM read instead of 128.
template <int G, bool NT, bool F8 = false, bool ROPE = false>
__global__ void __launch_bounds__(256, F8 ? 2 : 1) paged_decode_kernel(
    const uint16_t* __restrict__ q, const void* __restrict__ kc, const void* __restrict__ vc,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ ctx_lens, float scale_log2, int Hkv,
    int max_blocks, int part_blocks, int P, int window, float v_scale, float* __restrict__ part_o,
    float* __restrict__ part_ml, uint16_t* __restrict__ out, DecRope rp, const int32_t* __restrict__ shared_blocks) {
  // F8: kc / vc hold e4m3 of K / k_scale and V / v_scale; k_scale is folded into scale_log2 by the
  // host, v_scale multiplies the output here
  typedef typename KvFrag<F8>::raw Raw;
  constexpr int D = 128;
  const int p = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int Hq = Hkv * G;
  const int ctx = ctx_lens[b];
  const int nblk = (ctx + KV_BS - 1) / KV_BS;
  // sliding window (window > 0): the query at position ctx-1 sees keys [ctx - window, ctx)
  const int key_lo = window > 0 ? max(0, ctx - window) : 0;
  const int blk_lo = key_lo / KV_BS;
  // part_blocks > 0: fixed-size partitions of the block table; <= 0: the sequence's OWN blocks
  // split into P near-equal ranges (balanced per sequence whatever its length -- no nearly empty
  // tail partitions, and P can stay small, so each workgroup streams a long run of KV)
  const int blk0 = part_blocks > 0 ? max(blk_lo, p * part_blocks)
                                   : blk_lo + share_of(nblk - blk_lo, p, P);
  const int blk1 = part_blocks > 0 ? min(nblk, p * part_blocks + part_blocks)
                                   : blk_lo + share_of(nblk - blk_lo, p + 1, P);

  __shared__ float sm_o[4][D][17];
  __shared__ float sm_m[4][16], sm_l[4][16];

  // Q^T B-operand: lane holds Q[head h*G+col][dq(c) .. +7]; columns >= G are zero.  bf16 cache:
  // dq(c) = 32c + 8g.  FP8 cache: the head dim is visited in the order that lets ONE 16-byte load
  // carry two k-steps of a key row (64 contiguous bytes per row per wave instruction, as the bf16
  // loads have): dq(c) = 64(c >> 1) + 16g + 8(c & 1) -- any d order works as long as Q and K agree.
  __shared__ __attribute__((aligned(16))) uint16_t sm_q[ROPE ? G : 1][D];
  f32x4_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const int32_t* bt = block_tables + (size_t)b * max_blocks;
  const size_t head_stride = (size_t)KV_BS * D;  // elements per (block, kv-head)

  // K fragments: bf16 -> 8 x 16 B (st, c); fp8 -> 4 x 16 B (st, pair p of k-steps 2p, 2p+1)
  constexpr int NK = F8 ? 4 : 8;
  uint4 kr[NK];
  Raw vr[8];
  const int temporal = (NT && shared_blocks != nullptr) ? shared_blocks[0] : 0;   // blocks read cached
  auto load_blk = [&](int bi, uint4* kk, Raw* vv) {
    const size_t base = ((size_t)bt[bi] * Hkv + h) * head_stride;
    if (NT && bi >= temporal) dec_load_blk<NT, F8>(kc, vc, base, col, g, kk, vv);
    else dec_load_blk<false, F8>(kc, vc, base, col, g, kk, vv);
  };
  // K operand of (st, k-step c)
  auto kop = [&](const uint4* kk, int st, int c) -> bf16x8_t {
    if constexpr (F8) {
      const uint4 r = kk[st * 2 + (c >> 1)];
      return kv_operand((c & 1) ? make_uint2(r.z, r.w) : make_uint2(r.x, r.y));
    } else {
      return as_bf16x8(kk[st * 4 + c]);
    }
  };

  // ROPE, bf16 cache (PATCH): the new key / value make no round trip through memory inside the
  // step.  The prologue ropes q and k into LDS and writes the new key's cache row (256 contiguous
  // bytes, whole lines); the wave that streams the sequence's last block patches the new slot's K
  // and V into the fragments it loaded and stores the V^T slot group holding the new key back (16
  // full lines; the write costs the step by lines dirtied, scripts/probe_decode_rope_fused.py).
  // Every wave issues its first block before the prologue, so that block's HBM latency overlaps
  // the slab reads.  FP8 keeps the write-then-read order: the prologue writes K and V and the wave
  // whose first block receives them loads it after the barrier.
  constexpr bool PATCH = ROPE && !F8;
  __shared__ __attribute__((aligned(16))) uint16_t sm_kv[PATCH ? 2 : 1][PATCH ? D : 1];
  const int slot = ROPE ? rp.slots[b] : -1;
  const bool owner = ROPE && slot >= 0 && blk0 <= nblk - 1 && nblk - 1 < blk1;   // holds the new key's block
  int bi = blk0 + w;
  const bool early = ROPE && bi < blk1 && (PATCH || !(owner && bi == nblk - 1));
  if (early) load_blk(bi, kr, vr);
  if constexpr (ROPE) {
    constexpr int NV = D / 16;    // 8-vectors per half-head
    const size_t stride = (size_t)(Hq + 2 * Hkv) * D;
    const size_t row0 = (size_t)b * stride, slab = (size_t)gridDim.z * stride;
    const float* cs = rp.cos_sin + (size_t)rp.positions[b] * (D / 2) * 2;
    const int t = threadIdx.x;
    if (t < (G + 1) * NV) {
      const int hh = t / NV, c = t - hh * NV;   // hh < G: query head h*G + hh; hh == G: key head h
      if (hh < G || owner) {
        uint4 pa, pb;
        rope_rot8(rp.qkv, rp.part, rp.split, slab, row0 + (size_t)(hh < G ? h * G + hh : Hq + h) * D, D / 2, c, cs,
                  pa, pb);
        if (hh < G) {
          *reinterpret_cast<uint4*>(&sm_q[hh][c * 8]) = pa;
          *reinterpret_cast<uint4*>(&sm_q[hh][D / 2 + c * 8]) = pb;
        } else {
          if (!(rp.probe & 1)) kv_write_k<F8>(const_cast<void*>(kc), slot, h, Hkv, D, c, pa, pb, rp.inv_k);
          if constexpr (PATCH) {
            *reinterpret_cast<uint4*>(&sm_kv[0][c * 8]) = pa;
            *reinterpret_cast<uint4*>(&sm_kv[0][D / 2 + c * 8]) = pb;
          }
        }
      }
    } else if (owner && t < (G + 1) * NV + D / 8) {
      const int c = t - (G + 1) * NV;
      float vf[8];
      qkv_load8(rp.qkv, rp.part, rp.split, slab, row0 + (size_t)(Hq + Hkv + h) * D + c * 8, vf);
      if constexpr (PATCH) *reinterpret_cast<uint4*>(&sm_kv[1][c * 8]) = pack8(vf);
      else kv_write_v<F8>(const_cast<void*>(vc), slot, h, Hkv, D, c, pack8(vf), rp.inv_v);
    }
    // workgroup-scope release / acquire: sm_q / sm_kv to every wave and (FP8) the cache stores above
    // to this workgroup's KV loads below (same CU).  PATCH reads nothing back from memory, so its
    // barrier orders LDS only: the early KV loads and the key-row store stay in flight across it.
    if constexpr (PATCH) lds_barrier();
    else __syncthreads();
  }
  bf16x8_t qf[4];
  {
    const bool valid = col < G;
    const uint16_t* qr = ROPE ? &sm_q[valid ? col : 0][0] : q + ((size_t)b * Hq + h * G + (valid ? col : 0)) * D;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int dq = F8 ? 64 * (c >> 1) + 16 * g + 8 * (c & 1) : 32 * c + 8 * g;
      uint4 v = valid ? *reinterpret_cast<const uint4*>(qr + dq) : make_uint4(0, 0, 0, 0);
      qf[c] = as_bf16x8(v);
    }
  }

  if (bi < blk1 && !early) load_blk(bi, kr, vr);
  for (; bi < blk1; bi += 4) {
    uint4 kn[NK];
    Raw vn[8];
    const bool more = bi + 4 < blk1;
    if (more) load_blk(bi + 4, kn, vn);
    if constexpr (PATCH) {
      if (owner && bi == nblk - 1) {
        const int sn = slot % KV_BS;
        // K row sn: lanes col == sn % 16 of fragment half st = sn / 16 hold its d-chunks 32c + 8g
        if (col == (sn & 15)) {
#pragma unroll
          for (int st = 0; st < 2; ++st)
            if (st == (sn >> 4))
#pragma unroll
              for (int c = 0; c < 4; ++c) kr[st * 4 + c] = *reinterpret_cast<const uint4*>(&sm_kv[0][32 * c + 8 * g]);
        }
        // V^T column of key sn: stored at slot position ps = kv_v_slot(sn), i.e. element ps % 8 of
        // the lanes g == ps / 8 (rows d = 16 dt + col)
        const int ps = kv_v_slot(sn);
        if (g == (ps >> 3)) {
#pragma unroll
          for (int dt = 0; dt < 8; ++dt) vr[dt] = set_bf16(vr[dt], ps & 7, sm_kv[1][16 * dt + col]);
        }
        // the new key's slot group of the V^T tile back to the cache: the lanes g == ps / 8 store
        // their 8 x 16-byte pieces, the group's 16 full cache lines
        uint16_t* vt = reinterpret_cast<uint16_t*>(const_cast<void*>(vc)) + ((size_t)bt[bi] * Hkv + h) * head_stride;
        if (g != (ps >> 3)) {
        } else if (rp.probe & 4) {
#pragma unroll
          for (int dt = 0; dt < 8; ++dt) {
            const uint4 v = vr[dt];
            __builtin_nontemporal_store(u32x4_t{v.x, v.y, v.z, v.w},
                                        reinterpret_cast<u32x4_t*>(vt + kv_v_off(16 * dt + col, 8 * g, D)));
          }
        } else if (!(rp.probe & 2)) {
#pragma unroll
          for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<uint4*>(vt + kv_v_off(16 * dt + col, 8 * g, D)) = vr[dt];
        }
      }
    }

    f32x4_t s[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      s[st] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) s[st] = mfma16(kop(kr, st, c), qf[c], s[st]);
    }
    const int key0 = bi * KV_BS;
    float tmax = -INFINITY;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + 16 * st + 4 * g + i;
        float v = s[st][i] * scale_log2;
        v = key < ctx && key >= key_lo ? v : -INFINITY;
        s[st][i] = v;
        tmax = fmaxf(tmax, v);
      }
    tmax = xor16_max(tmax);
    tmax = xor32_max(tmax);
    const float mn = fmaxf(m, tmax);
    const float alpha = exp2f(m - mn);
    float rs = 0.f;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int i = 0; i < 4; ++i) { const float e = exp2f(s[st][i] - mn); s[st][i] = e; rs += e; }
    rs = xor16_sum(rs);
    rs = xor32_sum(rs);
    l = l * alpha + rs;
    m = mn;
    const bf16x8_t pf = pack_p(s[0], s[1]);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      o[dt] *= alpha;
      o[dt] = mfma16(kv_operand(vr[dt]), pf, o[dt]);
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i < NK) kr[i] = kn[i];
        vr[i] = vn[i];
      }
    }
  }

  // Combine the 4 waves through LDS.  Lane (col, g) holds O^T[d = 16dt + 4g + i][col].
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) sm_o[w][16 * dt + 4 * g + i][col] = o[dt][i];
  if (g == 0) { sm_m[w][col] = m; sm_l[w][col] = l; }
  // PATCH: the V^T tile store of the last block stays in flight (a full barrier would wait for its
  // write acknowledgement here, once per workgroup, behind the chip-wide KV read stream)
  if constexpr (PATCH) lds_barrier();
  else __syncthreads();

  for (int idx = threadIdx.x; idx < G * D; idx += 256) {
    const int qh = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, sm_m[ww][qh]);
    float L = 0.f, O = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) {
        const float f = exp2f(sm_m[ww][qh] - M);
        L += sm_l[ww][qh] * f;
        O += sm_o[ww][d][qh] * f;
      }
    }
    const int head = h * G + qh;
    O *= v_scale;
    if (P == 1) {
      out[((size_t)b * Hq + head) * D + d] = f2bf(L > 0.f ? O / L : 0.f);
    } else {
      const size_t pi = ((size_t)b * Hq + head) * P + p;
      part_o[pi * D + d] = O;
      if (d == 0) { part_ml[pi * 2] = M; part_ml[pi * 2 + 1] = L; }
    }
  }
}

// ------------------------------------------------------------------------------------------
// The same attention where keys and values come from memory at its full rate: fragments of K take 64 bytes of a row each,
// which memory serves at 5.8 to 6.3 TB/s, whole runs that are marked as read once at 6.8.  So a wave brings each (block, kv
// head) tile of K and of V, 8 KB each, to LDS by LDS-DMA in pieces of 1 KB, through a ring of T tiles of its own (no barrier:
// it waits for its own pieces).  A tile is read to registers as soon as it is there, and the one T tiles on takes its place.
// Chunk c of K's row r lies at c ^ (r & 15) (through the pieces' source addresses), so that sixteen rows' reads touch all
// banks; V's slot groups lie as in the cache.
// A workgroup of NWV waves has one (partition of a) sequence and kv head, wave w its blocks w, w + NWV, ...
// bf16 cache, queries roped.  ROPE: they are not, and neither are the new keys in the cache, as in paged_decode_kernel (DecRope): what it
// takes of the projection comes ahead of the first waves' tiles, the new key and value replace in LDS what came for them.  us of two decode
// steps of four layers, 32 query and 8 key heads, contexts from 0.8 of the longest, a launch of its own -> this: 5 of 700 851 -> 845, 8 of
// 1500 898 -> 880, 16 of 1000 937 -> 922, 24 of 1500 1018 -> 1001, 32 of 1024 1018 -> 995, of 2600 1256 -> 1230, 64 of 300 1078 -> 1051, 72 of
// 700 1261 -> 1252, 100 of 1200 1686 -> 1671, 128 of 40 1205 -> 1191.  The start is a chain of loads, 4 us, that a CU with two long workgroups does not
// win back: 39 of 4152 1716 -> 1736, 128 of 2617 2648 -> 2653 (Python's ops.kernels.rope_inside knows).
// ------------------------------------------------------------------------------------------
template <int G, int NWV, int T, bool ROPE = false>
__global__ void __launch_bounds__(64 * NWV, T == 2 ? 2 : 1) paged_stream_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ ctx_lens, float scale_log2, int Hkv, int max_blocks,
    int P, int window, float v_scale, float* __restrict__ part_o, float* __restrict__ part_ml, uint16_t* __restrict__ out,
    const int32_t* __restrict__ shared_blocks, int cached, int ordered, DecRope rp) {
  constexpr int D = 128, TILE = KV_BS * D * 2, QB = ROPE ? 0 : (G + 3) / 4 * 1024, RING = T * TILE;
  constexpr bool ORD = NWV == 4 && T == 2;
  __shared__ __attribute__((aligned(16))) char smem[NWV * (RING + QB) + (ROPE ? (G + 2) * D * 2 : 0)];
  uint16_t(*sm_q)[D] = reinterpret_cast<uint16_t(*)[D]>(smem + NWV * (RING + QB)), (*sm_kv)[D] = sm_q + G;      // ROPE: queries, the new key and value
  static_assert(sizeof(smem) <= (T == 2 && NWV == 4 ? 80 : 160) * 1024 && sizeof(smem) >= ORDER_LDS, "four waves: two workgroups a CU");
  const int p = blockIdx.x, h = blockIdx.y;
  int b = blockIdx.z, ctx;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool whole = !(ORD && ordered) && P == 1 && window == 0 && max_blocks > 0;       // the table's blocks: asked for beside the length
  const int spec = whole ? block_tables[(size_t)b * max_blocks + min(w + NWV * lane, max_blocks - 1)] : 0;
  if (ORD && ordered) {
    const int2 s = longest_first<256>(ctx_lens, gridDim.z, blockIdx.z, ordered, smem);
    b = s.x;
    ctx = s.y;
  } else {
    ctx = ctx_lens[b];
  }
  const int col = lane & 15, g = lane >> 4;
  const int Hq = Hkv * G;
  const int nblk = (ctx + KV_BS - 1) / KV_BS;
  const int key_lo = window > 0 ? max(0, ctx - window) : 0, blk_lo = key_lo / KV_BS;
  const int blk0 = blk_lo + share_of(nblk - blk_lo, p, P), blk1 = blk_lo + share_of(nblk - blk_lo, p + 1, P);
  const int32_t* bt = block_tables + (size_t)b * max_blocks;
  const int first = blk0 + w, n = first < blk1 ? (blk1 - 1 - first) / NWV + 1 : 0;        // this wave's blocks
  const int temporal = shared_blocks != nullptr ? max(cached, shared_blocks[0]) : cached;  // blocks read through the caches
  char* mine = smem + w * (RING + QB);
  const uint32_t lds0 = lds_at(mine);
  const uint32_t kvoff = (lane >> 4) * 256u, vvoff = lane * 16u;     // K: a piece has four rows, chunk (lane & 15) ^ row of each
  int ids = whole ? spec : n > 0 ? bt[first + min(lane, n - 1) * NWV] : 0;
  // the block of tile i, asked for in turn, from the lane that has it: a scalar load of its own would be waited for with every
  // read of LDS
  auto id = [&](int i) {
    if (i > 0 && (i & 63) == 0 && i < n) ids = bt[first + min(i + lane, n - 1) * NWV];
    return __builtin_amdgcn_readlane(ids, i & 63);
  };
  // tile 2 i + v: keys (v 0) or values of this wave's block i
  auto issue = [&](int j, int block) {
    const bool key = (j & 1) == 0;
    const char* src = reinterpret_cast<const char*>(key ? kc : vc) + ((size_t)block * Hkv + h) * TILE;
    const uint32_t at = lds0 + (j & (T - 1)) * TILE;
    const bool nt = first + (j >> 1) * NWV >= temporal;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t vo = key ? kvoff + (((lane & 15) ^ ((4 * e + (lane >> 4)) & 15)) << 4) : vvoff;
      if (nt) ring_piece<true>(vo, src + e * 1024, at + e * 1024);
      else ring_piece<false>(vo, src + e * 1024, at + e * 1024);
    }
  };
  f32x4_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  bf16x8_t qf[4];
  const int slot = ROPE ? rp.slots[b] : -1;
  const bool owner = ROPE && slot >= 0 && blk0 <= nblk - 1 && nblk - 1 < blk1;   // holds the new key's block
  const int last = owner ? bt[nblk - 1] : 0;
  if constexpr (ROPE) {
    // by the first waves ahead of their tiles: behind these it would wait for all that the chip asks for at first
    constexpr int NV = D / 16;    // 8-vectors per half-head
    const size_t stride = (size_t)(Hq + 2 * Hkv) * D;
    const size_t row0 = (size_t)b * stride, slab = (size_t)gridDim.z * stride;
    const float* cs = rp.cos_sin + (size_t)rp.positions[b] * (D / 2) * 2;
    for (int t = threadIdx.x; t < (G + 1) * NV + D / 8; t += 64 * NWV) {
      const int hh = t / NV, c = t - hh * NV;      // hh < G: query head h G + hh; hh == G: key head h
      if (hh < G || (hh == G && owner)) {
        uint4 pa, pb;
        rope_rot8(rp.qkv, rp.part, rp.split, slab, row0 + (size_t)(hh < G ? h * G + hh : Hq + h) * D, D / 2, c, cs, pa, pb);
        uint16_t* to = hh < G ? sm_q[hh] : sm_kv[0];
        *reinterpret_cast<uint4*>(to + c * 8) = pa;
        *reinterpret_cast<uint4*>(to + D / 2 + c * 8) = pb;
        if (hh == G) kv_write_k<false>(const_cast<uint16_t*>(kc), slot, h, Hkv, D, c, pa, pb, 1.f);
      } else if (hh > G && owner) {
        const int cv = t - (G + 1) * NV;
        float vv[8];
        qkv_load8(rp.qkv, rp.part, rp.split, slab, row0 + (size_t)(Hq + Hkv + h) * D + cv * 8, vv);
        *reinterpret_cast<uint4*>(&sm_kv[1][cv * 8]) = pack8(vv);
      }
    }
  }
  int ahead = 0;                                   // the block of the tiles T on
  if (n > 0) {
    if constexpr (!ROPE) {
      // the queries' rows first: they are there when the first keys are (past the G heads: the last one's, not used)
      const char* qs = reinterpret_cast<const char*>(q + ((size_t)b * Hq + h * G) * D);
#pragma unroll
      for (int e = 0; e < QB / 1024; ++e)
        ring_piece<false>((uint32_t)min(4 * e + (lane >> 4), G - 1) * 256u + (lane & 15) * 16u, qs, lds0 + RING + e * 1024);
    }
#pragma unroll
    for (int j = 0; j < T; j += 2)
      if (j < 2 * n) {
        const int block = id(j / 2);
        issue(j, block);
        issue(j + 1, block);
      }
    ahead = id(T / 2);
  }
  if constexpr (ROPE) lds_barrier();
  {
    for (int i = 0; i < n; ++i) {
      const int bi = first + i * NWV, next = id(i + 1 + T / 2);
      ring_landed<T, 8>(2 * i, 2 * n);
      if (i == 0) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          qf[c] = col < G ? as_bf16x8(*reinterpret_cast<const uint4*>(ROPE ? reinterpret_cast<const char*>(sm_q[min(col, G - 1)]) + c * 64 + g * 16
                                                                          : mine + RING + min(col, G - 1) * 256 + c * 64 + g * 16))
                          : as_bf16x8(make_uint4(0, 0, 0, 0));
      }
      uint4 kf[2][4];
      char* ki = mine + (2 * i & (T - 1)) * TILE;
      const bool fresh = ROPE && owner && bi == nblk - 1;         // the new key's row replaces what came for it
      if (fresh) {
        if (lane < 16)
          *reinterpret_cast<uint4*>(ki + (slot % KV_BS) * 256 + ((lane ^ (slot & 15)) << 4)) = *reinterpret_cast<const uint4*>(&sm_kv[0][8 * lane]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // by other lanes than read it
      }
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int c = 0; c < 4; ++c) kf[st][c] = *reinterpret_cast<const uint4*>(ki + (16 * st + col) * 256 + (((4 * c + g) ^ col) << 4));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // read: the place is free
      if (i + T / 2 < n) issue(2 * i + T, ahead);
      f32x4_t s[2];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        s[st] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) s[st] = mfma16(as_bf16x8(kf[st][c]), qf[c], s[st]);
      }
      const int key0 = bi * KV_BS;
      float tmax = -INFINITY;
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = key0 + 16 * st + 4 * g + e;
          float v = s[st][e] * scale_log2;
          v = key < ctx && key >= key_lo ? v : -INFINITY;
          s[st][e] = v;
          tmax = fmaxf(tmax, v);
        }
      tmax = xor16_max(tmax);
      tmax = xor32_max(tmax);
      const float mn = fmaxf(m, tmax);
      const float alpha = exp2f(m - mn);
      float rs = 0.f;
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = exp2f(s[st][e] - mn);
          s[st][e] = x;
          rs += x;
        }
      rs = xor16_sum(rs);
      rs = xor32_sum(rs);
      l = l * alpha + rs;
      m = mn;
      const bf16x8_t pf = pack_p(s[0], s[1]);
      ring_landed<T, 8>(2 * i + 1, 2 * n);
      if (fresh) {
        // and its values', whose slot group goes back to the cache, 16 whole lines
        const int ps = kv_v_slot(slot % KV_BS);
        char* vg = mine + ((2 * i + 1) & (T - 1)) * TILE + (ps >> 3) * 2048;
#pragma unroll
        for (int e = 0; e < 2; ++e) *reinterpret_cast<uint16_t*>(vg + (2 * lane + e) * 16 + (ps & 7) * 2) = sm_kv[1][2 * lane + e];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // in another type, and by other lanes, than read
        char* to = reinterpret_cast<char*>(const_cast<uint16_t*>(vc)) + ((size_t)last * Hkv + h) * TILE + (ps >> 3) * 2048;
#pragma unroll
        for (int e = 0; e < 2; ++e)
          *reinterpret_cast<uint4*>(to + e * 1024 + lane * 16) = *reinterpret_cast<const uint4*>(vg + e * 1024 + lane * 16);
      }
      uint4 vf[8];
      const char* vi = mine + ((2 * i + 1) & (T - 1)) * TILE + g * 2048 + col * 16;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) vf[dt] = *reinterpret_cast<const uint4*>(vi + dt * 256);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + T / 2 < n) issue(2 * i + 1 + T, ahead);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        o[dt] *= alpha;
        o[dt] = mfma16(as_bf16x8(vf[dt]), pf, o[dt]);
      }
      ahead = next;
    }
  }

  // lane (col, g) holds O^T[d = 16 dt + 4 g + i][col]
  if constexpr (NWV == 1) {        // one slice
    if (col >= G) return;
    const size_t row = (size_t)b * Hq + h * G + col;
    const float inv = l > 0.f ? v_scale / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[row * D + 16 * dt + 4 * g + i] = f2bf(o[dt][i] * inv);         // out is aligned to its elements only
    return;
  }
  __syncthreads();                                 // every wave's tiles are used up
  float(*sm_o)[D][17] = reinterpret_cast<float(*)[D][17]>(smem);
  float(*sm_ml)[16][2] = reinterpret_cast<float(*)[16][2]>(smem + NWV * D * 17 * 4);
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) sm_o[w][16 * dt + 4 * g + i][col] = o[dt][i];
  if (g == 0) sm_ml[w][col][0] = m, sm_ml[w][col][1] = l;
  __syncthreads();
  for (int idx = threadIdx.x; idx < G * D; idx += 64 * NWV) {
    const int qh = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NWV; ++ww) M = fmaxf(M, sm_ml[ww][qh][0]);
    float L = 0.f, O = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < NWV; ++ww) {
        const float f = exp2f(sm_ml[ww][qh][0] - M);
        L += sm_ml[ww][qh][1] * f;
        O += sm_o[ww][d][qh] * f;
      }
    }
    const size_t row = (size_t)b * Hq + h * G + qh;
    O *= v_scale;
    if (P == 1) {
      out[row * D + d] = f2bf(L > 0.f ? O / L : 0.f);
    } else {
      part_o[(row * P + p) * D + d] = O;
      if (d == 0) { part_ml[(row * P + p) * 2] = M; part_ml[(row * P + p) * 2 + 1] = L; }
    }
  }
}

// Merge of the P partition results of each (sequence, head) row, one wave a row: no barrier and no LDS.  The first sixteen
// partitions (eight a half wave, four columns a lane) are asked for before their weights are known; past the last one that
// one is read again and left out (as zeros: a weight of zero leaves an infinite sum in).  A loop of single loads for the
// remainder paid a trip to memory for each.
// us with the attention before it, one wave's barriers and single loads -> this: 24 sequences of 3 partitions 57.6 -> 54.8,
// 12 of 6 23.3 -> 21.5, 5 of 4 8.5 -> 7.8, one of 44 14.1 -> 12.5 (of 8, whose loads were together before, 0.1).
__global__ void __launch_bounds__(256) decode_combine_kernel(const float* __restrict__ part_o,
                                                             const float* __restrict__ part_ml, int P, int rows,
                                                             uint16_t* __restrict__ out) {
  constexpr int D = 128;
  // a caller's workspace and output need no more than their elements' alignment
  typedef float f32x4_el __attribute__((ext_vector_type(4), aligned(4)));
  typedef float f32x2_el __attribute__((ext_vector_type(2), aligned(4)));
  typedef uint32_t u32x2_el __attribute__((ext_vector_type(2), aligned(2)));
  const int lane = threadIdx.x & 63, half = lane >> 5, c = 4 * (lane & 31);
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= rows) return;
  const size_t base = (size_t)row * P;
  float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
  float L = 0.f, M = -INFINITY;
  for (int c0 = 0; c0 < P; c0 += 64) {      // one pass for P <= 64
    const int np = min(64, P - c0);
    const bool live = lane < np;
    f32x2_el ml = {-INFINITY, 0.f};
    if (live) ml = *reinterpret_cast<const f32x2_el*>(part_ml + (base + c0 + lane) * 2);
    f32x4_el v[8];
    auto ask = [&](int p0) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = *reinterpret_cast<const f32x4_el*>(part_o + (base + c0 + min(p0 + 2 * u + half, np - 1)) * D + c);
    };
    ask(0);
    const float mn = fmaxf(M, wave_max(ml.x)), ref = mn == -INFINITY ? 0.f : mn;
    const float f = exp2f(ml.x - ref), a = exp2f(M - ref);      // partitions without a key: 0
    M = mn;
    L = L * a + wave_sum(f * ml.y);
    O.x *= a; O.y *= a; O.z *= a; O.w *= a;
    for (int p0 = 0; p0 < np; p0 += 16) {
      if (p0) ask(p0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float w0 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), p0 + 2 * u));
        const float w1 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), p0 + 2 * u + 1));
        const float w = half ? w1 : w0;
        const f32x4_el o = p0 + 2 * u + half < np ? v[u] : f32x4_el{0.f, 0.f, 0.f, 0.f};
        O.x += w * o.x; O.y += w * o.y; O.z += w * o.z; O.w += w * o.w;
      }
    }
  }
  O.x = xor32_sum(O.x); O.y = xor32_sum(O.y); O.z = xor32_sum(O.z); O.w = xor32_sum(O.w);
  const float inv = L > 0.f ? 1.f / L : 0.f;
  if (half == 0)
    *reinterpret_cast<u32x2_el*>(out + (size_t)row * D + c) = u32x2_el{pack2bf(O.x * inv, O.y * inv), pack2bf(O.z * inv, O.w * inv)};
}

// ------------------------------------------------------------------------------------------
// Varlen causal prefill over the paged cache (D = 128).
// grid = (n_tiles, Hq); block = 512 = 8 waves x 16 query rows = 128-row query tile.
// Tile t covers query rows [tile_q0[t], +128) of sequence tile_seq[t]; those rows sit at
// positions ctx - q_len + row (chunked prefill / prefix reuse: keys come from the cache).
//   * K tile (64 keys x 128) and V^T tile (2 blocks x 128 x 32) double-buffered in LDS and shared
//     by all 8 waves; register-staged (next tile's loads issue before this tile's MFMAs, LDS
//     writes after); one barrier per tile.
//   * <= 128 VGPRs so two workgroups (16 waves, 4 per SIMD) share a CU: one wave's softmax VALU
//     overlaps another's MFMAs (a 1-wave-per-SIMD build of this loop was VALU-serialised).
//   * VALU trimmed: Q is pre-scaled by softmax_scale*log2(e) once (scores come out of the MFMA
//     in the exp2 domain), the causal mask is applied only on tiles that cross the diagonal, and
//     the O rescale is deferred until the running max grows by > RESCALE_THR (P is
//     then bounded by 2^THR, exact after the final 1/l).
//   * The host orders tiles heaviest-first (most keys) so the causal triangle drains evenly.
// ------------------------------------------------------------------------------------------
constexpr int PF_KT = 64;     // keys per tile
#ifndef CFC_PF_QK_PIPE
#define CFC_PF_QK_PIPE 1
#endif
constexpr int PF_QK_PIPE = CFC_PF_QK_PIPE;
#ifndef CFC_PF_V_EARLY
#define CFC_PF_V_EARLY 1
#endif
constexpr int PF_V_EARLY = CFC_PF_V_EARLY;   // prefill v5: V fragments of the first PF_V_EARLY half-tiles read before the softmax (2: 251 VGPRs, 1 % slower, profiles/r05_ab_prefill_attn_vearly2_rejected.log)
   // prefill v5: K fragments of a half-tile read ahead of its MFMAs
constexpr int PF_WAVES = 8;
constexpr int PF_ROWS = 16 * PF_WAVES;
constexpr float RESCALE_THR = 8.0f;

__device__ __forceinline__ int k_lds_off(int row, int ch) { return row * 256 + ((ch ^ (row & 15)) << 4); }
__device__ __forceinline__ int v_lds_off(int blk, int d, int ch) {
  return blk * 128 * 64 + d * 64 + ((ch ^ (((d >> 3) & 1) << 1)) << 4);
}

template <int MINW>
__global__ void __launch_bounds__(512, MINW) prefill_paged_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens,
    const int32_t* __restrict__ tile_seq, const int32_t* __restrict__ tile_q0, float scale_log2, int Hq, int Hkv,
    int max_blocks, uint16_t* __restrict__ out) {
  constexpr int D = 128;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // LDS: [K buf0 16K][K buf1 16K][V buf0 16K][V buf1 16K]
  const int t = blockIdx.x, hq = blockIdx.y;
  const int G = Hq / Hkv, hk = hq / G;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, tid = threadIdx.x;
  const int col = lane & 15, g = lane >> 4;
  const int s = tile_seq[t], qs = tile_q0[t];
  const int q_begin = cu_q[s], q_len = cu_q[s + 1] - q_begin;
  const int ctx = ctx_lens[s];
  const int pos_base = ctx - q_len;
  const int row_last = min(qs + PF_ROWS - 1, q_len - 1);
  const int kend = pos_base + row_last + 1;  // keys [0, kend) are needed by this tile
  const int ntiles = (kend + PF_KT - 1) / PF_KT;
  const int32_t* bt = block_tables + (size_t)s * max_blocks;

  const int my_row = qs + 16 * w + col;
  const int my_pos = pos_base + my_row;
  const int wave_min_pos = pos_base + qs + 16 * w;
  bf16x8_t qf[4];
  {
    const int rr = min(my_row, q_len - 1);
    const uint16_t* qr = q + ((size_t)(q_begin + rr) * Hq + hq) * D;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float f[8];
      unpack8(*reinterpret_cast<const uint4*>(qr + 32 * c + 8 * g), f);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] *= scale_log2;
      qf[c] = as_bf16x8(pack8(f));
    }
  }

  uint4 kst[2], vst[2];
  auto gload = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int id = tid + 512 * i;
      {  // K: row = id>>4 (key within tile), ch = id&15
        const int row = id >> 4, ch = id & 15, key = kt * PF_KT + row;
        if (key < kend) {
          const int blk = bt[key / KV_BS];
          kst[i] = *reinterpret_cast<const uint4*>(kc + (((size_t)blk * Hkv + hk) * KV_BS + (key % KV_BS)) * D + ch * 8);
        } else {
          kst[i] = make_uint4(0, 0, 0, 0);
        }
      }
      {  // V^T: blk_i = id>>9, d = (id>>2)&127, ch = id&3
        const int bi = id >> 9, d = (id >> 2) & 127, ch = id & 3;
        const int key0 = kt * PF_KT + bi * KV_BS;
        if (key0 < kend) {
          const int blk = bt[key0 / KV_BS];
          vst[i] = *reinterpret_cast<const uint4*>(vc + ((size_t)blk * Hkv + hk) * D * KV_BS + kv_v_off(d, 8 * ch, D));
        } else {
          vst[i] = make_uint4(0, 0, 0, 0);
        }
      }
    }
  };
  auto lwrite = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int id = tid + 512 * i;
      *reinterpret_cast<uint4*>(smem + buf * 16384 + k_lds_off(id >> 4, id & 15)) = kst[i];
      *reinterpret_cast<uint4*>(smem + 32768 + buf * 16384 + v_lds_off(id >> 9, (id >> 2) & 127, id & 3)) = vst[i];
    }
  };

  f32x4_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  gload(0);
  lwrite(0);
  __syncthreads();
  for (int kt = 0; kt < ntiles; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < ntiles;
    if (more) gload(kt + 1);

    const char* kb = smem + cur * 16384;
    const char* vb = smem + 32768 + cur * 16384;
    const int key0 = kt * PF_KT;
    // tiles wholly above this wave's rows (possible only in the last tiles): skip the math
    if (key0 <= wave_min_pos + 15) {
      f32x4_t sc[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        sc[st] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const int row = 16 * st + col;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          sc[st] = mfma16(as_bf16x8(*reinterpret_cast<const uint4*>(kb + k_lds_off(row, 4 * c + g))), qf[c], sc[st]);
      }
      if (key0 + PF_KT - 1 > wave_min_pos) {  // diagonal tile: causal mask
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key0 + 16 * st + 4 * g + i > my_pos) sc[st][i] = -INFINITY;
      }
      float tmax = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                         fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
      tmax = fmaxf(tmax, fmaxf(fmaxf(fmaxf(sc[2][0], sc[2][1]), fmaxf(sc[2][2], sc[2][3])),
                               fmaxf(fmaxf(sc[3][0], sc[3][1]), fmaxf(sc[3][2], sc[3][3]))));
      tmax = xor16_max(tmax);
      tmax = xor32_max(tmax);
      // deferred rescale: keep the old max unless some row of the wave grew by > THR
      if (!__all(tmax - m <= RESCALE_THR)) {
        const float mn = fmaxf(m, tmax);
        const float mref = mn == -INFINITY ? 0.f : mn;
        const float alpha = exp2f(m - mref);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt] *= alpha;
        m = mn;
      }
      const float mref = m == -INFINITY ? 0.f : m;
      float rs = 0.f;
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) { const float e = exp2f(sc[st][i] - mref); sc[st][i] = e; rs += e; }
      rs = xor16_sum(rs);
      rs = xor32_sum(rs);
      l += rs;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8_t pf = pack_p(sc[2 * ks], sc[2 * ks + 1]);
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
          o[dt] = mfma16(as_bf16x8(*reinterpret_cast<const uint4*>(vb + v_lds_off(ks, 16 * dt + col, g))), pf, o[dt]);
      }
    }
    if (more) lwrite(cur ^ 1);
    __syncthreads();
  }

  if (my_row < q_len) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* orow = out + ((size_t)(q_begin + my_row) * Hq + hq) * D;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      uint2 pk;
      pk.x = pack2bf(o[dt][0] * inv, o[dt][1] * inv);
      pk.y = pack2bf(o[dt][2] * inv, o[dt][3] * inv);
      *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * g) = pk;
    }
  }
}

// ------------------------------------------------------------------------------------------
// Prefill v4: 4 waves x 32 query rows on v_mfma_f32_32x32x16_bf16 (128-row tiles, as v3).
//   * S^T = K . Q^T per 32-key half-tile: A = K rows from LDS, B = Q^T from registers (8 k-steps
//     over D = 128).  C/D of 32x32: col = lane & 31 (query), row = 8(i>>2) + 4(lane>>5) + (i&3)
//     (key), so each lane owns one query row's scores for 16 of every 32 keys (the other 16 in
//     lane ^ 32): row max / sum = 31 local ops + one xor-32 shuffle.
//   * O^T = V^T . P^T: the S^T accumulator IS the P^T B-operand (k-step s of a 32-key
//     tile = registers 8s..8s+7, key order 16s + 8(j>>2) + 4h + (j&3)); the V^T LDS image stores
//     each d row's 64 keys in exactly that slot order, so the A fragment is one ds_read_b128.
//     The cache's V^T blocks are in the decode (16x16) slot order; the permutation to the 32x32
//     order is applied while writing the LDS image (two 8-byte stores per 16-byte load).
//   * K / V^T tiles (64 keys) double-buffered in LDS, register-staged (loads for tile t+1 issued
//     before tile t's MFMAs, LDS writes after), one barrier per tile; deferred rescale as in v3.
//   * vs v3 (16x16x32, 16 rows/wave): every LDS fragment byte now feeds twice the FLOPs.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x16_t mfma32(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// V^T image: row d (64 keys = 128 B), 16-byte chunk c at d*128 + ((c ^ (d & 7)) << 4)
__device__ __forceinline__ int v4_off(int d, int c) { return d * 128 + ((c ^ (d & 7)) << 4); }

template <int MINW>
__global__ void __launch_bounds__(256, MINW) prefill_paged_kernel_v4(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens,
    const int32_t* __restrict__ tile_seq, const int32_t* __restrict__ tile_q0, float scale_log2, int Hq, int Hkv,
    int max_blocks, uint16_t* __restrict__ out) {
  constexpr int D = 128;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // LDS: [K buf0 16K][K buf1 16K][V buf0 16K][V buf1 16K]
  const int t = blockIdx.x, hq = blockIdx.y;
  const int G = Hq / Hkv, hk = hq / G;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, tid = threadIdx.x;
  const int l32 = lane & 31, hi = lane >> 5;
  const int s = tile_seq[t], qs = tile_q0[t];
  const int q_begin = cu_q[s], q_len = cu_q[s + 1] - q_begin;
  const int ctx = ctx_lens[s];
  const int pos_base = ctx - q_len;
  const int row_last = min(qs + PF_ROWS - 1, q_len - 1);
  const int kend = pos_base + row_last + 1;
  const int ntiles = (kend + PF_KT - 1) / PF_KT;
  const int32_t* bt = block_tables + (size_t)s * max_blocks;

  const int my_row = qs + 32 * w + l32;
  const int my_pos = pos_base + my_row;
  const int wave_min_pos = pos_base + qs + 32 * w;
  // Q^T B-operand, pre-scaled into the exp2 domain: k-step ks holds Q[row][16ks + 8hi .. +7]
  bf16x8_t qf[8];
  {
    const int rr = min(my_row, q_len - 1);
    const uint16_t* qr = q + ((size_t)(q_begin + rr) * Hq + hq) * D;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      float f[8];
      unpack8(*reinterpret_cast<const uint4*>(qr + 16 * ks + 8 * hi), f);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] *= scale_log2;
      qf[ks] = as_bf16x8(pack8(f));
    }
  }

  // staging: 1024 16-B pieces of K + 1024 of V per tile, 4 + 4 per thread
  uint4 kst[4], vst[4];
  auto gload = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int id = tid + 256 * i;
      {  // K: row = id >> 4 (key in tile), chunk = id & 15
        const int row = id >> 4, ch = id & 15, key = kt * PF_KT + row;
        kst[i] = key < kend ? *reinterpret_cast<const uint4*>(
                                  kc + (((size_t)bt[key / KV_BS] * Hkv + hk) * KV_BS + (key % KV_BS)) * D + ch * 8)
                            : make_uint4(0, 0, 0, 0);
      }
      {  // V^T: block bi = id >> 9, d = (id >> 2) & 127, cache chunk g = id & 3 (slots 8g..8g+7)
        const int bi = id >> 9, d = (id >> 2) & 127, g = id & 3;
        const int key0 = kt * PF_KT + bi * KV_BS;
        vst[i] = key0 < kend ? *reinterpret_cast<const uint4*>(
                                   vc + ((size_t)bt[key0 / KV_BS] * Hkv + hk) * D * KV_BS + kv_v_off(d, 8 * g, D))
                             : make_uint4(0, 0, 0, 0);
      }
    }
  };
  auto lwrite = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int id = tid + 256 * i;
      *reinterpret_cast<uint4*>(smem + buf * 16384 + k_lds_off(id >> 4, id & 15)) = kst[i];
      // cache slots 8g..8g+3 hold keys 4g..4g+3 and 8g+4..8g+7 hold keys 16+4g..16+4g+3; in the
      // 32x32 order key k of a 32-block sits at slot 16(k>>4) + 8((k>>2)&1) + 4((k&15)>>3) + (k&3)
      const int bi = id >> 9, d = (id >> 2) & 127, g = id & 3;
      const int base = 32 * bi + 8 * (g & 1) + 4 * (g >> 1);        // slot of key 4g (s = 0)
      char* vrow = smem + 32768 + buf * 16384;
      const uint2 lo = make_uint2(vst[i].x, vst[i].y), hi2 = make_uint2(vst[i].z, vst[i].w);
      *reinterpret_cast<uint2*>(vrow + v4_off(d, base >> 3) + (base & 7) * 2) = lo;
      *reinterpret_cast<uint2*>(vrow + v4_off(d, (base + 16) >> 3) + ((base + 16) & 7) * 2) = hi2;
    }
  };

  f32x16_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m = -INFINITY, l = 0.f;

  gload(0);
  lwrite(0);
  __syncthreads();
  for (int kt = 0; kt < ntiles; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < ntiles;
    if (more) gload(kt + 1);

    const char* kb = smem + cur * 16384;
    const char* vb = smem + 32768 + cur * 16384;
    const int key0 = kt * PF_KT;
    if (key0 <= wave_min_pos + 31) {
      f32x16_t sc[2];
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[hf][r] = 0.f;
        const int row = 32 * hf + l32;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
          sc[hf] = mfma32(as_bf16x8(*reinterpret_cast<const uint4*>(kb + k_lds_off(row, 2 * ks + hi))), qf[ks], sc[hf]);
      }
      if (key0 + PF_KT - 1 > wave_min_pos) {  // diagonal tile: causal mask
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 32 * hf + 8 * (r >> 2) + 4 * hi + (r & 3) > my_pos) sc[hf][r] = -INFINITY;
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sc[hf][r]);
      tmax = xor32_max(tmax);
      if (!__all(tmax - m <= RESCALE_THR)) {
        const float mn = fmaxf(m, tmax);
        const float mref = mn == -INFINITY ? 0.f : mn;
        const float alpha = exp2f(m - mref);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
        m = mn;
      }
      const float mref = m == -INFINITY ? 0.f : m;
      float rs = 0.f;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int r = 0; r < 16; ++r) { const float e = exp2f(sc[hf][r] - mref); sc[hf][r] = e; rs += e; }
      rs = xor32_sum(rs);
      l += rs;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
          uint4 u;
          u.x = pack2bf(sc[hf][8 * ss + 0], sc[hf][8 * ss + 1]);
          u.y = pack2bf(sc[hf][8 * ss + 2], sc[hf][8 * ss + 3]);
          u.z = pack2bf(sc[hf][8 * ss + 4], sc[hf][8 * ss + 5]);
          u.w = pack2bf(sc[hf][8 * ss + 6], sc[hf][8 * ss + 7]);
          const bf16x8_t pf = as_bf16x8(u);
          const int c = 4 * hf + 2 * ss + hi;     // V^T chunk of slots 32hf + 16ss + 8hi .. +7
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
            o[dt] = mfma32(as_bf16x8(*reinterpret_cast<const uint4*>(vb + v4_off(32 * dt + l32, c))), pf, o[dt]);
        }
    }
    if (more) lwrite(cur ^ 1);
    __syncthreads();
  }

  if (my_row < q_len) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* orow = out + ((size_t)(q_begin + my_row) * Hq + hq) * D;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {   // registers 4rg..4rg+3 = d 32dt + 8rg + 4hi + 0..3
        uint2 pk;
        pk.x = pack2bf(o[dt][4 * rg] * inv, o[dt][4 * rg + 1] * inv);
        pk.y = pack2bf(o[dt][4 * rg + 2] * inv, o[dt][4 * rg + 3] * inv);
        *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * rg + 4 * hi) = pk;
      }
  }
}

// ------------------------------------------------------------------------------------------
// Prefill v5 (default): GQA-packed 8-wave tiles on v_mfma_f32_32x32x16_bf16.
// grid = (n_tiles, Hkv); block = 512 = 8 waves, 2 per SIMD.  A tile is QR = 256 / G query rows of
// ONE sequence for ALL G query heads of kv-head hk: wave w takes head hk*G + (w % G) and rows
// 32 (w / G) .. +31.  Every K/V byte staged in LDS therefore feeds 256 query rows (8 waves), and
// the tile spans only 256/G positions, so at G = 4 the causal diagonal idles 4x fewer rows than a
// 256-row single-head tile would.
//   * LDS per KV tile (64 keys): K 64 x 256 B (16-B chunk c of key r at r*256 + ((c ^ (r&15))<<4))
//     and V^T 128 d-rows x 128 B copied AS STORED in the cache (decode slot order).  The decode
//     order already fits the 32x32 PV: cache chunk g of a 32-key block holds keys {4g..4g+3,
//     16+4g..16+4g+3}, all with key bit 2 == g&1, which is exactly the half-wave (lane>>5) that holds
//     them in the S^T accumulator; so k-step s of half hf uses chunk 4hf + 2s + hi for the A operand
//     and accumulator registers {4s..4s+3, 8+4s..8+4s+3} as the B operand -- one ds_read_b128 and
//     one in-lane pack, no permutation anywhere.  V swizzle c ^ ((d>>1)&7) ^ ((d&1)<<2): the
//     ds_read_b128 lane groups and the 8-lane ds_write_b128 groups are both conflict-free.
//   * register-staged double buffer, one barrier per tile (loads for tile t+1 issued before tile
//     t's MFMAs, LDS writes after); Q pre-scaled into the exp2 domain; deferred rescale
//     (RESCALE_THR); row max / sum across the two half-waves with v_permlane32_swap (no LDS
//     bpermute); per-lane partial row sums combined once at the end; v_exp_f32 / v_cvt_pk_bf16_f32
//     directly; waves 4-7 at static priority 1 (the younger half loses VALU arbitration otherwise).
// ------------------------------------------------------------------------------------------
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}
// value of lane l ^ 32 combined with lane l's own (both halves get the same result)
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// reductions over the 4 lanes l, l^16, l^32, l^48 (one MFMA 16x16 output column): two VALU
// permlane swaps instead of two ds_bpermute round trips
__device__ __forceinline__ float quad_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return pair_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float quad_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return pair_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}
// 64 x 128-byte rows of the second key part: chunk c of row r, swizzled
__device__ __forceinline__ int k2_lds_off(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }
__device__ __forceinline__ int v5_off(int d, int c) { return d * 128 + ((c ^ ((d >> 1) & 7) ^ ((d & 1) << 2)) << 4); }

// EXP: keys and values are not in the paged cache but dense (a latent cache's, expanded for this pass):
// K [tokens][Hkv][128] and V^T [Hkv][128][ldv] with each 32 tokens in the cache's slot order, sequence s
// at tokens tok_base[s] .. (rounded up to 64, zero-filled); outputs leave with row stride ldo.
// RD = 64 (with EXP): a second key part shared by all heads, K2 [tokens][64], with the heads' q2 [rows][H][64];
// a sink per head in the denominator; outputs times sigmoid(gate) (row stride ldg, columns as out).
struct PfExtra {
  int64_t q_ld = 0, q_hs = 0;         // q strides per row and head
  const uint16_t* q2 = nullptr;
  const uint16_t* k2 = nullptr;
  const float* sink = nullptr;
  const uint16_t* gate = nullptr;
  int64_t ldg = 0;
};
// PARTS: gridDim.z workgroups share a tile, each multiplying 1 / gridDim.z of its row groups (every wave still stages
// keys and values): short prompts have fewer tiles than CUs, whose SIMDs' two waves then wait for one another.
template <int G, bool F8 = false, bool EXP = false, int RD = 0, bool PARTS = false>
__global__ void __launch_bounds__(512, 2) prefill_gqa_kernel(
    const uint16_t* __restrict__ q, const void* __restrict__ kc, const void* __restrict__ vc,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens,
    const int32_t* __restrict__ tile_seq, const int32_t* __restrict__ tile_q0, float scale_log2, int Hq, int Hkv,
    int max_blocks, int window, float v_scale, int xcd_local, uint16_t* __restrict__ out,
    const int32_t* __restrict__ tok_base = nullptr, int64_t ldv = 0, int64_t ldo = 0, PfExtra ex = PfExtra{}) {
  // F8: e4m3 caches (K / k_scale folded into scale_log2 by the host, V / v_scale rescaled at the
  // output); tiles are widened to bf16 at the LDS write, so the MFMA loop is the bf16 one
  constexpr int D = 128;
  constexpr int QR = 256 / G;      // query rows per tile
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // LDS: [K buf0 16K][K buf1 16K][V buf0 16K][V buf1 16K]
  // xcd_local: the (tile, kv-head) grid is XCD-remapped so each XCD takes a contiguous run of the
  // kv-head-major order -- with Hkv a multiple of 8 one XCD serves whole kv-heads and its L2 holds
  // only their K/V, instead of every XCD touching every head's K/V
  int t = blockIdx.x, hk = blockIdx.y;
  if (xcd_local) {
    const int lin = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    hk = lin / gridDim.x;
    t = lin - hk * gridDim.x;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, tid = threadIdx.x;
  const int l32 = lane & 31, hi = lane >> 5;
  const int hq = hk * G + (w % G);
  const int rsub = w / G;
  const int s = tile_seq[t], qs = tile_q0[t];
  const int q_begin = cu_q[s], q_len = cu_q[s + 1] - q_begin;
  const int ctx = ctx_lens[s];
  const int pos_base = ctx - q_len;
  const int groups = PARTS ? 8 / G / (int)gridDim.z : 8 / G, group0 = PARTS ? (int)blockIdx.z * groups : 0;
  const bool mine = !PARTS || (rsub >= group0 && rsub < group0 + groups);
  const int first = qs + 32 * group0;               // the rows this workgroup answers for: first ..
  if (PARTS && first >= q_len) return;
  const int row_last = min(first + 32 * groups - 1, q_len - 1);
  const int kend = pos_base + row_last + 1;         // keys [0, kend) are needed by them
  const int ntiles = (kend + PF_KT - 1) / PF_KT;
  // sliding window: row at position p sees keys (p - window, p]; the first row bounds it
  const int kt_begin = window > 0 ? max(0, pos_base + first - window + 1) / PF_KT : 0;
  const int32_t* bt = block_tables + (size_t)s * max_blocks;

  if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 256) __builtin_amdgcn_s_setprio(1);

  const int my_row = qs + 32 * rsub + l32;
  const int my_pos = pos_base + my_row;
  const int wave_min_pos = pos_base + qs + 32 * rsub;
  // Q^T B-operand, pre-scaled: k-step ks holds Q[row][16ks + 8hi .. +7]
  bf16x8_t qf[8], qf2[RD ? RD / 16 : 1];
  {
    const int rr = min(my_row, q_len - 1);
    const uint16_t* qr = RD ? q + (q_begin + rr) * ex.q_ld + hq * ex.q_hs : q + ((size_t)(q_begin + rr) * Hq + hq) * D;
    auto scaled = [&](const uint16_t* p) {
      float f[8];
      unpack8(*reinterpret_cast<const uint4*>(p), f);
      uint4 u;
      u.x = cvt_pk_bf16(f[0] * scale_log2, f[1] * scale_log2);
      u.y = cvt_pk_bf16(f[2] * scale_log2, f[3] * scale_log2);
      u.z = cvt_pk_bf16(f[4] * scale_log2, f[5] * scale_log2);
      u.w = cvt_pk_bf16(f[6] * scale_log2, f[7] * scale_log2);
      return as_bf16x8(u);
    };
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = scaled(qr + 16 * ks + 8 * hi);
    if constexpr (RD) {
      const uint16_t* q2 = ex.q2 + ((size_t)(q_begin + rr) * Hq + hq) * RD;
#pragma unroll
      for (int ks = 0; ks < RD / 16; ++ks) qf2[ks] = scaled(q2 + 16 * ks + 8 * hi);
    }
  }

  // staging: tile kt = cache blocks 2kt, 2kt+1; piece i of a thread is block 2kt+i, bytes 16 tid ..
  // of both its K image [32][128] and its V^T image [128][32] (each 8 KB contiguous).  The block id
  // is workgroup-uniform (scalar load) and the data loads are UNCONDITIONAL (a block past kend
  // re-reads the last needed block; its V is zeroed at the LDS write), so no per-lane select
  // makes the compiler wait for the loads inside the issue sequence -- they stay in flight across
  // the tile's MFMAs.
  const int nb_need = (kend + KV_BS - 1) / KV_BS;
  uint4 ks0, ks1, vs0, vs1, k2s;     // named (not an array): an array here is kept in scratch
  const int64_t tok0 = EXP ? tok_base[s] : 0;
  auto gload = [&](int kt) {
    if constexpr (EXP) {
      const int64_t t0 = tok0 + kt * PF_KT;
      const uint16_t* kp = reinterpret_cast<const uint16_t*>(kc) + ((t0 + (tid >> 4)) * Hkv + hk) * D + 8 * (tid & 15);
      const uint16_t* vp = reinterpret_cast<const uint16_t*>(vc) + ((int64_t)hk * D + (tid >> 3)) * ldv + t0 + 8 * (tid & 7);
      ks0 = *reinterpret_cast<const uint4*>(kp);
      vs0 = *reinterpret_cast<const uint4*>(vp);
      ks1 = *reinterpret_cast<const uint4*>(kp + (int64_t)32 * Hkv * D);
      vs1 = *reinterpret_cast<const uint4*>(vp + 64 * ldv);
      if constexpr (RD) k2s = *reinterpret_cast<const uint4*>(ex.k2 + (t0 + (tid >> 3)) * RD + 8 * (tid & 7));
      return;
    }
    const int b0 = bt[min(2 * kt, nb_need - 1)], b1 = bt[min(2 * kt + 1, nb_need - 1)];
    if constexpr (F8) {
      // 8 KB of K and 8 KB of V per tile: one 16-B piece of each per thread; block = tid >> 8
      const size_t base = ((size_t)(tid >> 8 ? b1 : b0) * Hkv + hk) * (KV_BS * D) + 16 * (tid & 255);
      ks0 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(kc) + base);
      vs0 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(vc) + base);
    } else {
      const size_t base0 = ((size_t)b0 * Hkv + hk) * (KV_BS * D) + 8 * tid;
      const size_t base1 = ((size_t)b1 * Hkv + hk) * (KV_BS * D) + 8 * tid;
      ks0 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(kc) + base0);
      vs0 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(vc) + base0);
      ks1 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(kc) + base1);
      vs1 = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(vc) + base1);
    }
  };
  auto lwrite = [&](int buf, int kt) {
    char* kb = smem + buf * 16384;
    char* vb = smem + 32768 + buf * 16384;
    if constexpr (EXP) {
      *reinterpret_cast<uint4*>(kb + k_lds_off(tid >> 4, tid & 15)) = ks0;
      *reinterpret_cast<uint4*>(kb + k_lds_off((tid >> 4) + 32, tid & 15)) = ks1;
      *reinterpret_cast<uint4*>(vb + v5_off(tid >> 3, tid & 7)) = vs0;
      *reinterpret_cast<uint4*>(vb + v5_off((tid >> 3) + 64, tid & 7)) = vs1;
      if constexpr (RD) *reinterpret_cast<uint4*>(smem + 65536 + buf * 8192 + k2_lds_off(tid >> 3, tid & 7)) = k2s;
      return;
    }
    const bool z0 = kt * PF_KT >= kend, z1 = kt * PF_KT + KV_BS >= kend;
    if constexpr (F8) {
      const int b = tid >> 8, e = tid & 255;
      const int key = (e >> 3) + 32 * b, ch = 2 * (e & 7);          // 16 d values = bf16 chunks ch, ch+1
      *reinterpret_cast<uint4*>(kb + k_lds_off(key, ch)) = fp8x8_to_bf16x8(make_uint2(ks0.x, ks0.y));
      *reinterpret_cast<uint4*>(kb + k_lds_off(key, ch + 1)) = fp8x8_to_bf16x8(make_uint2(ks0.z, ks0.w));
      // 16 bytes of the [4][D][8] tile = slot chunk e >> 6 of rows d, d + 1
      const int d = 2 * (e & 63), c = 4 * b + (e >> 6);
      const bool z = b ? z1 : z0;
      const uint4 zero = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(vb + v5_off(d, c)) = z ? zero : fp8x8_to_bf16x8(make_uint2(vs0.x, vs0.y));
      *reinterpret_cast<uint4*>(vb + v5_off(d + 1, c)) = z ? zero : fp8x8_to_bf16x8(make_uint2(vs0.z, vs0.w));
    } else {
      *reinterpret_cast<uint4*>(kb + k_lds_off(tid >> 4, tid & 15)) = ks0;
      *reinterpret_cast<uint4*>(kb + k_lds_off((tid >> 4) + 32, tid & 15)) = ks1;
      // element 8 tid of the [4][D][8] tile = slot chunk tid >> 7 of row tid & 127
      *reinterpret_cast<uint4*>(vb + v5_off(tid & 127, tid >> 7)) = z0 ? make_uint4(0, 0, 0, 0) : vs0;
      *reinterpret_cast<uint4*>(vb + v5_off(tid & 127, 4 + (tid >> 7))) = z1 ? make_uint4(0, 0, 0, 0) : vs1;
    }
  };

  f32x16_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m = -INFINITY, l = 0.f;   // l: this lane's partial row sum (its 32 of every 64 keys)
  // l in 4 interleaved partial sums: one serial chain of 32 dependent v_add_f32 per tile was
  // on the critical path between the exp2s and the next tile (ISA); summed once at the end
  float lp[4] = {0.f, 0.f, 0.f, 0.f};

  gload(kt_begin);
  lwrite(kt_begin & 1, kt_begin);
  __syncthreads();
  for (int kt = kt_begin; kt < ntiles; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < ntiles;
    if (more) gload(kt + 1);

    const char* kb = smem + cur * 16384;
    const char* vb = smem + 32768 + cur * 16384;
    const int key0 = kt * PF_KT;
    const bool below = window > 0 && key0 + PF_KT - 1 <= wave_min_pos - window;  // all keys out of window
    if (mine && key0 <= wave_min_pos + 31 && !below) {     // else every key of the tile is masked for this wave
      // scores come out of the MFMA already shifted by the running max (the accumulator starts at
      // -m): a tile that needs no rescale goes straight to exp2, without 32 subtractions per lane
      const float mref0 = m == -INFINITY ? 0.f : m;
      f32x16_t sc[2];
      if constexpr (PF_QK_PIPE == 2) {
        // both halves' 16 K fragments in flight before the 16 MFMAs (246 VGPRs; measured equal to
        // one half at a time, profiles/r05_ab_prefill_attn_qkpipe2.log)
        uint4 kf[2][8];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            kf[hf][ks] = *reinterpret_cast<const uint4*>(kb + k_lds_off(32 * hf + l32, 2 * ks + hi));
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[hf][r] = -mref0;
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) sc[hf] = mfma32(as_bf16x8(kf[hf][ks]), qf[ks], sc[hf]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
      } else
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[hf][r] = -mref0;
        const int row = 32 * hf + l32;
        // all 8 K fragments of the half in flight before its MFMA chain (PF_QK_PIPE): left to
        // itself hipcc issued read -> lgkmcnt(0) -> MFMA sixteen times, one LDS round trip each
        if constexpr (PF_QK_PIPE) {
          uint4 kf[8];
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) kf[ks] = *reinterpret_cast<const uint4*>(kb + k_lds_off(row, 2 * ks + hi));
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) sc[hf] = mfma32(as_bf16x8(kf[ks]), qf[ks], sc[hf]);
          if constexpr (RD) {
            uint4 kr[RD / 16];
#pragma unroll
            for (int ks = 0; ks < RD / 16; ++ks)
              kr[ks] = *reinterpret_cast<const uint4*>(smem + 65536 + cur * 8192 + k2_lds_off(row, 2 * ks + hi));
#pragma unroll
            for (int ks = 0; ks < RD / 16; ++ks) sc[hf] = mfma32(as_bf16x8(kr[ks]), qf2[ks], sc[hf]);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 8 + RD / 16, 0);   // the DS reads, then
          __builtin_amdgcn_sched_group_barrier(0x008, 8 + RD / 16, 0);   // the MFMAs (counted lgkmcnt waits)
        } else {
#pragma unroll
          for (int ks = 0; ks < 8; ++ks)
            sc[hf] = mfma32(as_bf16x8(*reinterpret_cast<const uint4*>(kb + k_lds_off(row, 2 * ks + hi))), qf[ks],
                            sc[hf]);
        }
      }
      // the first half's 8 V^T fragments read now, under the softmax's VALU work (PF_V_EARLY)
      uint4 vf0[2][2][4];
      if constexpr (PF_V_EARLY) {
#pragma unroll
        for (int hf = 0; hf < PF_V_EARLY; ++hf)
#pragma unroll
          for (int ss = 0; ss < 2; ++ss)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
              vf0[hf][ss][dt] = *reinterpret_cast<const uint4*>(vb + v5_off(32 * dt + l32, 4 * hf + 2 * ss + hi));
      }
      if (key0 + PF_KT - 1 > wave_min_pos) {  // diagonal tile: causal mask
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 32 * hf + 8 * (r >> 2) + 4 * hi + (r & 3) > my_pos) sc[hf][r] = -INFINITY;
      }
      if (window > 0 && key0 <= wave_min_pos + 31 - window) {  // window edge: keys <= pos - window
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 32 * hf + 8 * (r >> 2) + 4 * hi + (r & 3) <= my_pos - window) sc[hf][r] = -INFINITY;
      }
      // the tile's row max minus mref0: two interleaved v_max3 chains (16 instructions for 32
      // values; the pairwise form compiled to 16 v_max + 8 v_max3)
      float ta = fmaxf(fmaxf(sc[0][0], sc[0][1]), sc[0][2]);
      float tb = fmaxf(fmaxf(sc[1][0], sc[1][1]), sc[1][2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) {
        ta = fmaxf(fmaxf(ta, sc[0][r]), sc[0][r + 1]);
        tb = fmaxf(fmaxf(tb, sc[1][r]), sc[1][r + 1]);
      }
      float tmax = fmaxf(fmaxf(ta, sc[0][15]), fmaxf(tb, sc[1][15]));
      tmax = pair_max(tmax);
      if (!__all(m != -INFINITY && tmax <= RESCALE_THR)) {
        const float mn = fmaxf(m, mref0 + tmax);
        const float alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
#pragma unroll
        for (int u = 0; u < 4; ++u) lp[u] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
        m = mn;
        const float shift = (m == -INFINITY ? 0.f : m) - mref0;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[hf][r] -= shift;
      }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(sc[hf][r]);
          sc[hf][r] = e;
          lp[r & 3] += e;
        }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
          uint4 u;
          u.x = cvt_pk_bf16(sc[hf][4 * ss + 0], sc[hf][4 * ss + 1]);
          u.y = cvt_pk_bf16(sc[hf][4 * ss + 2], sc[hf][4 * ss + 3]);
          u.z = cvt_pk_bf16(sc[hf][8 + 4 * ss + 0], sc[hf][8 + 4 * ss + 1]);
          u.w = cvt_pk_bf16(sc[hf][8 + 4 * ss + 2], sc[hf][8 + 4 * ss + 3]);
          const bf16x8_t pf = as_bf16x8(u);
          const int c = 4 * hf + 2 * ss + hi;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
            o[dt] = mfma32(as_bf16x8(hf < PF_V_EARLY ? vf0[hf][ss][dt]
                                                     : *reinterpret_cast<const uint4*>(vb + v5_off(32 * dt + l32, c))),
                           pf, o[dt]);
        }
    }
    if (more) lwrite(cur ^ 1, kt + 1);
    __syncthreads();
  }

  l = pair_sum((lp[0] + lp[1]) + (lp[2] + lp[3]));
  if (mine && my_row < q_len) {
    float inv = l > 0.f ? v_scale / l : 0.f;
    if constexpr (RD != 0) {
      if (ex.sink) {
        const float sk = ex.sink[hq] * LOG2E, M = fmaxf(m, sk), f = __builtin_amdgcn_exp2f(m - M);
        inv = f / (l * f + __builtin_amdgcn_exp2f(sk - M));
      }
    }
    uint16_t* orow = EXP ? out + (q_begin + my_row) * ldo + hq * D : out + ((size_t)(q_begin + my_row) * Hq + hq) * D;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {   // registers 4rg..4rg+3 = d 32dt + 8rg + 4hi + 0..3
        float y[4] = {o[dt][4 * rg] * inv, o[dt][4 * rg + 1] * inv, o[dt][4 * rg + 2] * inv, o[dt][4 * rg + 3] * inv};
        if constexpr (RD != 0) {
          if (ex.gate) {
            const uint2 gv = *reinterpret_cast<const uint2*>(ex.gate + (q_begin + my_row) * ex.ldg + hq * D + 32 * dt + 8 * rg + 4 * hi);
            const float gz[4] = {__uint_as_float(gv.x << 16), __uint_as_float(gv.x & 0xffff0000u),
                                 __uint_as_float(gv.y << 16), __uint_as_float(gv.y & 0xffff0000u)};
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] *= 1.f / (1.f + __expf(-gz[e]));
          }
        }
        uint2 pk;
        pk.x = cvt_pk_bf16(y[0], y[1]);
        pk.y = cvt_pk_bf16(y[2], y[3]);
        *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * rg + 4 * hi) = pk;
      }
  }
}

// ------------------------------------------------------------------------------------------
// Varlen bidirectional encoder attention (BERT family), D in {32, 64}, S <= 512.
// Input qkv is the fused projection output [T, 3*H*D] (q | k | v, head-major inside each).
// 1-D grid over (query tile, head), XCD-remapped; block = 256 = 4 waves, tile = ENC_ROWS = 256
// query rows (wave w: 16-row groups w, w + 4, .. , ENC_R = 4 of them).  The WHOLE key/value range
// of the sequence is staged once in LDS per block (K row-major, V transposed with the per-32-key
// slot permutation) -- with 256-row tiles a MiniLM sequence (S <= 256) stages its K/V once per
// head instead of once per 64 rows -- then every wave runs the swapped-product online softmax:
// each 32-key K / V fragment is read from LDS once and reused by the wave's 4 row groups.
// Softmax: Q is pre-scaled by scale*log2(e) at load, the key mask runs only on the sequence's
// last (partial) 32-key tile, exponentials are v_exp_f32 (inputs <= 0).
// ------------------------------------------------------------------------------------------
constexpr int ENC_ROWS = 256;          // query rows per workgroup, 16 ENC_R of a wave
constexpr float ENC_NONE = 3.4028235e38f;      // less a maximum that no finite score is below, but finite: a score of -inf keeps its weight of 0

// Vector instructions bound it: 32 keys of 16 rows are 8 exponentials a lane, a quarter of the rate of others, and were some 40
// others, 14 of them for a maximum and a sum across lanes in every step.  Now scores start from the maximum (an MFMA's
// addend), a lane compares and sums its own keys only and the end masks in a copy of the step: some 22 others, 16 VGPRs more,
// so four workgroups a CU where there were five.  Texts of up to 128 tokens have two row groups a wave, and six workgroups.
// us a layer: 365 texts of 180 tokens, 12 heads of 32, 72 -> 61; forwards of 800 texts of 30 in all 953 -> 923, of 100 2868 -> 2784.
template <int D, int ENC_R>
__global__ void __launch_bounds__(256, D == 32 ? (ENC_R == 4 ? 4 : 6) : 2) encoder_attn_kernel(const uint16_t* __restrict__ qkv,
                                                           const int32_t* __restrict__ cu_seqlens,
                                                           const int32_t* __restrict__ tile_seq,
                                                           const int32_t* __restrict__ tile_q0, float scale_log2,
                                                           int H, uint16_t* __restrict__ out) {
  constexpr int NC = D / 8;         // 16-byte chunks per K row
  constexpr int KSTEPS = D / 32;    // MFMA k-steps over head_dim
  constexpr int DT = D / 16;        // 16-wide output column tiles
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // logical block = tile * H + head, XCD-remapped: every (query tile, head) block of a sequence
  // lands on ONE XCD, so the sequence's fused qkv rows (all heads share each 128-B line) are
  // fetched from HBM once into that XCD's L2 instead of once per XCD.
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int t = lb / H, h = lb - t * H;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tid = threadIdx.x;
  const int col = lane & 15, g = lane >> 4;
  const int s = tile_seq[t], qs = tile_q0[t];
  const int beg = cu_seqlens[s], S = cu_seqlens[s + 1] - beg;
  const int Spad = (S + 127) & ~127;       // V^T rows hold Spad slots (multiple of 128 => >=16 chunks)
  const int row_stride = 3 * H * D;
  char* klds = smem;                              // [Spad][D]  bf16, swizzled per 16-row group
  char* vlds = smem + (size_t)Spad * D * 2;       // [D][Spad]  bf16, slot-permuted, swizzled

  // K rows: chunk ch of row r at r*D*2 + ((ch ^ sw(r)) * 16).
  auto koff = [&](int r, int ch) -> int {
    if constexpr (D == 32) return r * 64 + ((ch ^ (((r >> 3) & 1) << 1)) << 4);
    else return r * 128 + ((ch ^ (r & 7)) << 4);
  };
  // V^T element (d, slot): row d has Spad*2 bytes; 16-byte chunk c = slot>>3 swizzled by d&15.
  auto voff_chunk = [&](int d, int c) -> int { return d * Spad * 2 + ((c ^ (d & 15)) << 4); };

  // Q fragments first (pre-scaled), so their loads overlap the K/V staging below
  const int wrow0 = qs + 16 * w;       // wave w: every fourth row group, so that short texts keep all waves at work
  const int ng = min(ENC_R, max(0, (S - wrow0 + 63) >> 6));   // row groups with >= 1 row (wave-uniform)
  bf16x8_t qf[ENC_R][KSTEPS];
#pragma unroll
  for (int rg = 0; rg < ENC_R; ++rg) {
    const int r = min(wrow0 + 64 * rg + col, S - 1);
    const uint16_t* qr = qkv + (size_t)(beg + r) * row_stride + h * D;
#pragma unroll
    for (int c = 0; c < KSTEPS; ++c) {
      float f[8];
      unpack8(*reinterpret_cast<const uint4*>(qr + 32 * c + 8 * g), f);
      uint4 u;
      u.x = pack2bf(f[0] * scale_log2, f[1] * scale_log2);
      u.y = pack2bf(f[2] * scale_log2, f[3] * scale_log2);
      u.z = pack2bf(f[4] * scale_log2, f[5] * scale_log2);
      u.w = pack2bf(f[6] * scale_log2, f[7] * scale_log2);
      qf[rg][c] = as_bf16x8(u);
    }
  }

  // K / V staging: a thread takes one chunk of four consecutive rows of K and of V, all loads ahead of the LDS writes, so one
  // memory round trip covers eight chunks.  Four keys are neighbours in the slot order: V^T takes eight 8-byte writes
  // of four keys where a row at a time took 32 of two bytes.
  for (int id = tid; id < Spad / 4 * NC; id += 256) {
    const int r = id / NC * 4, ch = id % NC;
    uint4 kv[4], vv[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      kv[b] = make_uint4(0, 0, 0, 0);
      vv[b] = make_uint4(0, 0, 0, 0);
      if (r + b < S) {
        const uint16_t* base = qkv + (size_t)(beg + r + b) * row_stride;
        kv[b] = *reinterpret_cast<const uint4*>(base + H * D + h * D + ch * 8);
        vv[b] = *reinterpret_cast<const uint4*>(base + 2 * H * D + h * D + ch * 8);
      }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) *reinterpret_cast<uint4*>(klds + koff(r + b, ch)) = kv[b];
    const int kin = r & 31, slot = (r & ~31) + 8 * ((kin >> 2) & 3) + 4 * (kin >> 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x[4] = {e < 2 ? vv[0].x : e < 4 ? vv[0].y : e < 6 ? vv[0].z : vv[0].w, e < 2 ? vv[1].x : e < 4 ? vv[1].y : e < 6 ? vv[1].z : vv[1].w,
                             e < 2 ? vv[2].x : e < 4 ? vv[2].y : e < 6 ? vv[2].z : vv[2].w, e < 2 ? vv[3].x : e < 4 ? vv[3].y : e < 6 ? vv[3].z : vv[3].w};
      const uint32_t pick = e & 1 ? 0x07060302u : 0x05040100u;     // the upper or the lower halves of two words
      *reinterpret_cast<uint2*>(vlds + voff_chunk(ch * 8 + e, slot >> 3) + (slot & 7) * 2) =
          make_uint2(__builtin_amdgcn_perm(x[1], x[0], pick), __builtin_amdgcn_perm(x[3], x[2], pick));
    }
  }
  __syncthreads();
  if (ng == 0) return;   // no barrier follows

  f32x4_t o[ENC_R][DT];
  float l[ENC_R];                 // a lane's own keys' share of the sums until the end
  f32x4_t ref[ENC_R];             // less the running maxima, what the scores start from: no subtraction is left for later
#pragma unroll
  for (int rg = 0; rg < ENC_R; ++rg) {
    ref[rg] = f32x4_t{ENC_NONE, ENC_NONE, ENC_NONE, ENC_NONE};
    l[rg] = 0.f;
#pragma unroll
    for (int i = 0; i < DT; ++i) o[rg][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  auto keys = [&](int k0, auto last) {
    constexpr bool TAIL = decltype(last)::value;      // fewer than 32 keys
    bf16x8_t kf[2][KSTEPS];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int c = 0; c < KSTEPS; ++c)
        kf[st][c] = as_bf16x8(*reinterpret_cast<const uint4*>(klds + koff(k0 + 16 * st + col, 4 * c + g)));
    bf16x8_t vf[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      vf[dt] = as_bf16x8(*reinterpret_cast<const uint4*>(vlds + voff_chunk(16 * dt + col, (k0 >> 3) + g)));

#pragma unroll
    for (int rg = 0; rg < ENC_R; ++rg) {
      if (rg >= ng) break;
      f32x4_t sc[2];
      auto scores = [&](const f32x4_t& from) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          sc[st] = from;
#pragma unroll
          for (int c = 0; c < KSTEPS; ++c) sc[st] = mfma16(kf[st][c], qf[rg][c], sc[st]);
        }
        if constexpr (TAIL) {
#pragma unroll
          for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (k0 + 16 * st + 4 * g + i >= S) sc[st][i] = -INFINITY;
        }
      };
      // three values an instruction
      auto largest = [&]() {
        const float a = fmaxf(fmaxf(sc[0][0], sc[0][1]), sc[0][2]), b = fmaxf(fmaxf(sc[1][0], sc[1][1]), sc[1][2]);
        return fmaxf(fmaxf(fmaxf(a, sc[0][3]), b), sc[1][3]);
      };
      scores(ref[rg]);
      // The running maximum moves, and O and l with it, only where a score exceeds it by more than RESCALE_THR (as in the
      // prefill kernel); each lane looks at its own keys, so nothing crosses lanes where none does.  Before the first
      // keys it lies below all scores.
      if (!__all(largest() <= RESCALE_THR)) {
        scores(f32x4_t{0.f, 0.f, 0.f, 0.f});
        const float m = -ref[rg][0], mn = fmaxf(m, quad_max(largest()));
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l[rg] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[rg][dt] *= alpha;
        ref[rg] = f32x4_t{-mn, -mn, -mn, -mn};
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[st][i] -= mn;
      }
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[st][i] = __builtin_amdgcn_exp2f(sc[st][i]);
          l[rg] += sc[st][i];
        }
      const bf16x8_t pf = pack_p(sc[0], sc[1]);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[rg][dt] = mfma16(vf[dt], pf, o[rg][dt]);
    }
  };
  int k0 = 0;
  for (; k0 + 32 <= S; k0 += 32) keys(k0, std::false_type{});
  if (k0 < S) keys(k0, std::true_type{});
#pragma unroll
  for (int rg = 0; rg < ENC_R; ++rg) l[rg] = quad_sum(l[rg]);

#pragma unroll
  for (int rg = 0; rg < ENC_R; ++rg) {
    const int my_row = wrow0 + 64 * rg + col;
    if (rg < ng && my_row < S) {
      const float inv = l[rg] > 0.f ? 1.f / l[rg] : 0.f;
      uint16_t* orow = out + ((size_t)(beg + my_row) * H + h) * D;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint2 pk;
        pk.x = pack2bf(o[rg][dt][0] * inv, o[rg][dt][1] * inv);
        pk.y = pack2bf(o[rg][dt][2] * inv, o[rg][dt][3] * inv);
        *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * g) = pk;
      }
    }
  }
}

}  // namespace

// Waves of a workgroup of the paged decode attention of `seen` blocks of a table in P slices, less than zero: those of
// paged_decode_kernel, keys and values straight to registers.  By the ring 128 KB are under way in a CU, in the eight waves of one
// workgroup (four with rings of twice the depth: 24 of 1500 28.1 us against 25.7, 16 of 700 14.5 against 13.8) or the four of each of two (two
// waves with twice the depth: 40 of 1500 52.7 against 49.1, 48 of 300 15.4 against 14.3); two blocks in one wave, which has nothing to merge
// (128 of 60 11.4 -> 9.1).  Up to 64 workgroups in four waves all the same: those of the fused step, whose small batches get the same bits
// either way.
// us of 8 key heads, one slice, straight -> ring: 8 of 2617 keys 50.3 -> 31.4, 24 59.9 -> 42.6, 32 66.2 -> 57.5, 48 97 -> 88, 72 158 -> 131, 90
// 170 -> 157, 128 219 -> 212, from 0.8 of it 198 -> 191; 24 of 700 19.1 -> 14.9; but 12 of 64 4.5 -> 5.1, 192 of 2617 315 -> 330 (more sequences than
// are ordered have 2 GB of cache and more to read from, and what waits in registers is deeper).  With four blocks or fewer to a slice, one a
// wave, a ring has nothing to have under way, and so for very few workgroups of any length: 1 of 400 in 12 slices 7.1 -> 7.7, 5 of 1500 in 24
// 14.5 -> 16.1, 24 of 400 in 12 20.8 -> 25.0, 3 of 2617 in one 38.0 -> 39.7.
constexpr int paged_waves(int64_t wgs, int seen, int P, int max_blocks) {
  if (wgs <= 32 || (wgs <= 256 && seen <= 8) || (P > 1 && (seen + P - 1) / P <= 4)) return -4;
  return wgs <= 64 ? 4 : wgs <= 256 ? 8 : max_blocks > 2 ? 4 : 1;
}

// q: [B, Hq, 128] bf16; caches per layer as documented above; out: [B, Hq, 128] bf16.
// part_o / part_ml: fp32 workspaces of B*Hq*P*128 and B*Hq*P*2 floats (unused when P == 1).
template <bool F8>
static int launch_paged_decode(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                               const int32_t* ctx_lens, int B, int Hq, int Hkv, int head_dim, int max_blocks,
                               int part_blocks, int P, float scale, int window, float v_scale, float* part_o,
                               float* part_ml, void* out, hipStream_t stream, const DecRope* rope = nullptr,
                               const int32_t* shared_blocks = nullptr) {
  if (head_dim != 128 || Hq % Hkv != 0 || B <= 0 || P <= 0 || window < 0) return -1;
  if (rope != nullptr && ((rope->qkv == nullptr) == (rope->part == nullptr) || (rope->part && rope->split < 1) ||
                          !rope->positions || !rope->slots || !rope->cos_sin))
    return -1;
  const DecRope rp = rope ? *rope : DecRope{};
  const int G = Hq / Hkv;
  dim3 grid(P, Hkv, B);
  const float sl2 = scale * LOG2E;
  // Longest first where more workgroups than two a CU wait for a place.  Just above 512 only for contexts that differ by more than
  // seven sixteenths: the few that are left over start when the first end, and those are longer in this order.  us of 8 key heads,
  // one partition, contexts from 0.4 / 0.7 of 2600: 66 sequences 103 -> 92 / 132 -> 127, 72 114 -> 105 / 137 -> (144), 80 130 -> 116 /
  // 143 -> (150), 104 157 -> 138 / 176 -> 165, 128 181 -> 159 / 197 -> 186; of 1100, 128 81 -> 73 / 88 -> 85.  136 and more: 0.95 to 1.08.
  // Tables for less than the shortest that is ordered do not ask (the contexts' extremes take 0.5).
  const int64_t wgs = (int64_t)P * Hkv * B;
  const int ordered = wgs <= 512 || B > DEC_ORDER_ROWS || max_blocks * KV_BS < DEC_ORDER_FROM || max_blocks >= 1 << 17 ? 0 : wgs < 704 ? 7 : 2;
#define DEC_ARGS (const uint16_t*)q, k_cache, v_cache, block_tables, ctx_lens, sl2, Hkv, max_blocks, part_blocks, P, \
    window, v_scale, part_o, part_ml, (uint16_t*)out, rp, shared_blocks
  // Read once, or through the caches.  CFC_DECODE_NT=0/1 forces either; of keys and values that come to registers B=128: 6.5 TB/s
  // read once, 5.9 through the caches, B=8: 3.8, 4.2; runs through LDS are read once
  static const int nt_env = [] { const char* e = getenv("CFC_DECODE_NT"); return e ? atoi(e) : -1; }();
  const bool nt = nt_env >= 0 ? nt_env != 0 : B >= 32;
  if constexpr (!F8) {
    const int seen = window > 0 ? min(max_blocks, (window + 30) / KV_BS + 1) : max_blocks;
    const bool aligned = (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;       // LDS-DMA's sources
    const bool few = rope && (B <= DEC_FUSED_ROWS || rope->probe);
    const int nw = few || part_blocks > 0 || B > DEC_ORDER_ROWS || !aligned ? -4 : paged_waves(wgs, seen, P, max_blocks);
    if (nw > 0) {
#define PDS_R(NWV, T, R)                                                                                                    \
  paged_stream_kernel<GG, NWV, T, R><<<grid, 64 * NWV, 0, stream>>>((const uint16_t*)q, (const uint16_t*)k_cache,            \
      (const uint16_t*)v_cache, block_tables, ctx_lens, sl2, Hkv, max_blocks, P, window, v_scale, part_o, part_ml,           \
      (uint16_t*)out, shared_blocks, nt_env == 0 ? INT_MAX : 0, ordered, rp)
#define PDS_GO(NWV, T)                     \
  {                                        \
    if (rope) PDS_R(NWV, T, true);         \
    else PDS_R(NWV, T, false);             \
  }
#define PDS_CASE(G_)                        \
  case G_: {                                \
    constexpr int GG = G_;                  \
    if (nw == 8) PDS_GO(8, 2)               \
    else if (nw == 1) PDS_GO(1, 4)          \
    else if (wgs <= 64) PDS_GO(4, 4)        \
    else PDS_GO(4, 2)                       \
  } break;
      switch (G) {
        PDS_CASE(1) PDS_CASE(2) PDS_CASE(4) PDS_CASE(8) PDS_CASE(16)
        default: return -3;
      }
#undef PDS_CASE
#undef PDS_GO
#undef PDS_R
      if (P > 1) decode_combine_kernel<<<(Hq * B + 3) / 4, 256, 0, stream>>>(part_o, part_ml, P, Hq * B, (uint16_t*)out);
      return CFC_CHECK_LAUNCH();
    }
  }
#define DEC_CASE(GG) \
  case GG: \
    if (rope) { \
      if (nt) paged_decode_kernel<GG, true, F8, true><<<grid, 256, 0, stream>>>(DEC_ARGS); \
      else paged_decode_kernel<GG, false, F8, true><<<grid, 256, 0, stream>>>(DEC_ARGS); \
    } else { \
      if (nt) paged_decode_kernel<GG, true, F8><<<grid, 256, 0, stream>>>(DEC_ARGS); \
      else paged_decode_kernel<GG, false, F8><<<grid, 256, 0, stream>>>(DEC_ARGS); \
    } \
    break;
  switch (G) {
    DEC_CASE(1) DEC_CASE(2) DEC_CASE(4) DEC_CASE(8) DEC_CASE(16)
    default: return -3;
  }
#undef DEC_CASE
#undef DEC_ARGS
  if (P > 1) decode_combine_kernel<<<(Hq * B + 3) / 4, 256, 0, stream>>>(part_o, part_ml, P, Hq * B, (uint16_t*)out);
  return CFC_CHECK_LAUNCH();
}

// what a launch takes (see paged_waves)
CFC_API int cfc_paged_waves(int64_t wgs, int seen, int P, int max_blocks) {
  return wgs < 1 || P < 1 ? 0 : paged_waves(wgs, seen, P, max_blocks);
}

// q: [B, Hq, 128] bf16; caches per layer as documented above; out: [B, Hq, 128] bf16.
// part_o / part_ml: fp32 workspaces of B*Hq*P*128 and B*Hq*P*2 floats (unused when P == 1).
// shared_blocks (device int32, may be null): leading blocks of every sequence read through the
// caches (the batch's shared prefix blocks), the rest nontemporal.
CFC_API int cfc_paged_decode_attention(const void* q, const void* k_cache, const void* v_cache,
                                       const int32_t* block_tables, const int32_t* ctx_lens, int B, int Hq, int Hkv,
                                       int head_dim, int max_blocks, int part_blocks, int P, float scale, int window,
                                       float* part_o, float* part_ml, void* out, const int32_t* shared_blocks,
                                       hipStream_t stream) {
  return launch_paged_decode<false>(q, k_cache, v_cache, block_tables, ctx_lens, B, Hq, Hkv, head_dim, max_blocks,
                                    part_blocks, P, scale, window, 1.f, part_o, part_ml, out, stream, nullptr,
                                    shared_blocks);
}

// Timing ablations of the fused decode RoPE (scripts/probe_decode_rope_fused.py): bit 1 skips the new
// key's cache row, bit 2 the V^T slot-group store, bit 4 makes that store nontemporal.  Results are wrong
// with bits 1 / 2 set; production never sets it.
static int g_dec_rope_probe = 0;
CFC_API int cfc_set_decode_rope_probe(int bits) {
  g_dec_rope_probe = bits;
  return 0;
}

// Decode attention with the step's RoPE + KV write in its prologue (DecRope).  qkv [B, (Hq+2Hkv)*128]
// bf16 OR part [split, B, (Hq+2Hkv)*128] fp32 slabs (exactly one non-null); positions / slots [B];
// fp8 != 0: e4m3 caches (K / k_scale, V / v_scale).  Writes out [B, Hq, 128]; q never leaves the chip.
CFC_API int cfc_paged_decode_rope_attention(const void* qkv, const float* part, int split, const int32_t* positions,
                                            const int32_t* slots, const float* cos_sin, void* k_cache, void* v_cache,
                                            const int32_t* block_tables, const int32_t* ctx_lens, int B, int Hq,
                                            int Hkv, int head_dim, int max_blocks, int part_blocks, int P, float scale,
                                            int window, int fp8, float k_scale, float v_scale, float* part_o,
                                            float* part_ml, void* out, const int32_t* shared_blocks,
                                            hipStream_t stream) {
  const DecRope rp{(const uint16_t*)qkv, part, split, positions, slots, cos_sin, 1.f / k_scale, 1.f / v_scale,
                   g_dec_rope_probe};
  if (fp8)
    return launch_paged_decode<true>(nullptr, k_cache, v_cache, block_tables, ctx_lens, B, Hq, Hkv, head_dim,
                                     max_blocks, part_blocks, P, scale * k_scale, window, v_scale, part_o, part_ml,
                                     out, stream, &rp, shared_blocks);
  return launch_paged_decode<false>(nullptr, k_cache, v_cache, block_tables, ctx_lens, B, Hq, Hkv, head_dim,
                                    max_blocks, part_blocks, P, scale, window, 1.f, part_o, part_ml, out, stream, &rp,
                                    shared_blocks);
}

// FP8 (e4m3fn) caches holding K / k_scale and V / v_scale
CFC_API int cfc_paged_decode_attention_fp8(const void* q, const void* k_cache, const void* v_cache,
                                           const int32_t* block_tables, const int32_t* ctx_lens, int B, int Hq,
                                           int Hkv, int head_dim, int max_blocks, int part_blocks, int P, float scale,
                                           int window, float k_scale, float v_scale, float* part_o, float* part_ml,
                                           void* out, const int32_t* shared_blocks, hipStream_t stream) {
  return launch_paged_decode<true>(q, k_cache, v_cache, block_tables, ctx_lens, B, Hq, Hkv, head_dim, max_blocks,
                                   part_blocks, P, scale * k_scale, window, v_scale, part_o, part_ml, out, stream,
                                   nullptr, shared_blocks);
}

CFC_API int cfc_prefill_tile_rows() { return PF_ROWS; }

static int prefill_variant() {
  static const int v = [] { const char* e = getenv("CFC_PREFILL_VARIANT"); return e ? atoi(e) : 5; }();
  return v;
}
static int prefill_xcd_local() {
  static const int v = [] { const char* e = getenv("CFC_PREFILL_XCD"); return e ? atoi(e) : 1; }();
  return v;
}

// Query rows per tile the default prefill kernel expects for Hq / Hkv heads (the host tiler's
// granularity): 256 / G on the GQA-packed kernel, else PF_ROWS.
CFC_API int cfc_prefill_rows(int Hq, int Hkv) {
  if (Hkv <= 0 || Hq % Hkv) return PF_ROWS;
  const int G = Hq / Hkv;
  const bool v5 = prefill_variant() == 5 && (G == 1 || G == 2 || G == 4 || G == 8);
  return v5 ? 256 / G : PF_ROWS;
}

CFC_API int cfc_prefill_attention(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                                  const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* tile_seq,
                                  const int32_t* tile_q0, int n_tiles, int tile_rows, int Hq, int Hkv, int head_dim,
                                  int max_blocks, float scale, int window, void* out, hipStream_t stream) {
  if (head_dim != 128 || Hkv <= 0 || Hq % Hkv != 0 || window < 0) return -1;
  if (tile_rows != cfc_prefill_rows(Hq, Hkv)) return -2;     // tiles cut for another kernel
  if (n_tiles <= 0) return 0;
  const size_t lds = 65536;
  const int G = Hq / Hkv;
#define PF_ARGS (const uint16_t*)q, (const uint16_t*)k_cache, (const uint16_t*)v_cache, block_tables, cu_q, ctx_lens, \
    tile_seq, tile_q0, scale * LOG2E, Hq, Hkv, max_blocks, (uint16_t*)out
#define PF5_ARGS (const uint16_t*)q, k_cache, v_cache, block_tables, cu_q, ctx_lens, \
    tile_seq, tile_q0, scale * LOG2E, Hq, Hkv, max_blocks, window, 1.f, prefill_xcd_local(), (uint16_t*)out
  if (tile_rows != PF_ROWS || (G * tile_rows == 256 && prefill_variant() == 5)) {
    // 5: GQA-packed 8-wave kernel (default)
    dim3 grid(n_tiles, Hkv);
    // parts of tiles while no CU gets two (us whole, in 2 parts: 420 rows, 56 workgroups 20.0, 17.1; 900 rows 33.8, 29.8;
    // 200 rows behind 1500 keys 52.6, 41.3; four prompts of up to 200 rows 16.0, 13.7)
    while (n_tiles * Hkv * (int)grid.z * 2 <= 256 && (int)grid.z * 2 <= 8 / G) grid.z *= 2;
    if (grid.z > 1) {
      switch (G) {
        case 1: prefill_gqa_kernel<1, false, false, 0, true><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
        case 2: prefill_gqa_kernel<2, false, false, 0, true><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
        case 4: prefill_gqa_kernel<4, false, false, 0, true><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
        default: return -3;
      }
      return CFC_CHECK_LAUNCH();
    }
    switch (G) {
      case 1: prefill_gqa_kernel<1><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
      case 2: prefill_gqa_kernel<2><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
      case 4: prefill_gqa_kernel<4><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
      case 8: prefill_gqa_kernel<8><<<grid, 512, lds, stream>>>(PF5_ARGS); break;
      default: return -3;
    }
    return CFC_CHECK_LAUNCH();
  }
  if (window > 0) return -4;     // sliding window: GQA-packed kernel only
  // legacy single-head 128-row kernels: 0 = v3 <=128 VGPRs (2 workgroups / CU); 1 = v3 <=256 VGPRs;
  // 2/3 = v4 (32x32 MFMA, 2 / 1 WG per CU)
  const int variant = prefill_variant();
  if (variant == 1) prefill_paged_kernel<2><<<dim3(n_tiles, Hq), 512, lds, stream>>>(PF_ARGS);
  else if (variant == 2) prefill_paged_kernel_v4<2><<<dim3(n_tiles, Hq), 256, lds, stream>>>(PF_ARGS);
  else if (variant == 3) prefill_paged_kernel_v4<1><<<dim3(n_tiles, Hq), 256, lds, stream>>>(PF_ARGS);
  else prefill_paged_kernel<4><<<dim3(n_tiles, Hq), 512, lds, stream>>>(PF_ARGS);
#undef PF_ARGS
#undef PF5_ARGS
  return CFC_CHECK_LAUNCH();
}

// Causal prefill attention over dense K [tokens][H][128] / V^T [H][128][ldv] (prefill_gqa_kernel's EXP
// layout), one kv head per query head, 256-row tiles; out row t, head h at t ldo + 128 h.
CFC_API int cfc_prefill_attention_expanded(const void* q, const void* k, const void* vt, const int32_t* tok_base,
                                           int64_t ldv, const int32_t* cu_q, const int32_t* ctx_lens,
                                           const int32_t* tile_seq, const int32_t* tile_q0, int n_tiles, int H, float scale,
                                           void* out, int64_t ldo, hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if (H < 1 || H > 65535 || ldv % 8 || ldo % 4 || ldo < (int64_t)128 * H || ((uintptr_t)vt & 15) || ((uintptr_t)out & 7)) return -1;
  prefill_gqa_kernel<1, false, true><<<dim3(n_tiles, H), 512, 65536, stream>>>(
      (const uint16_t*)q, k, vt, nullptr, cu_q, ctx_lens, tile_seq, tile_q0, scale * LOG2E, H, H, 0, 0, 1.f,
      prefill_xcd_local(), (uint16_t*)out, tok_base, ldv, ldo);
  return CFC_CHECK_LAUNCH();
}

// The same with a second key part of 64 dimensions shared by all heads (K2 [tokens][64]; q2 [rows][H][64]), a sliding
// window (0: none), a sink per head (may be null) and an output gate (may be null); q row t, head h at
// t q_ld + h q_hs.
CFC_API int cfc_prefill_attention_expanded2(const void* q, int64_t q_ld, int64_t q_hs, const void* q2, const void* k,
                                            const void* k2, const void* vt, const int32_t* tok_base, int64_t ldv,
                                            const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* tile_seq,
                                            const int32_t* tile_q0, int n_tiles, int H, float scale, int window,
                                            const float* sink, const void* gate, int64_t ldg, void* out, int64_t ldo,
                                            hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if (H < 1 || H > 65535 || ldv % 8 || ldo % 4 || ldo < (int64_t)128 * H || ((uintptr_t)vt & 15) || ((uintptr_t)out & 7) ||
      q_ld % 8 || q_hs % 8 || ((uintptr_t)q & 15) || ldg % 4 || ((uintptr_t)gate & 7) || window < 0 || !q2 || !k2)
    return -1;
  PfExtra ex;
  ex.q_ld = q_ld; ex.q_hs = q_hs; ex.q2 = (const uint16_t*)q2; ex.k2 = (const uint16_t*)k2;
  ex.sink = sink; ex.gate = (const uint16_t*)gate; ex.ldg = ldg;
  static bool raised = false;
  if (!raised) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_gqa_kernel<1, false, true, 64>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 65536 + 16384);
    raised = true;
  }
  prefill_gqa_kernel<1, false, true, 64><<<dim3(n_tiles, H), 512, 65536 + 16384, stream>>>(
      (const uint16_t*)q, k, vt, nullptr, cu_q, ctx_lens, tile_seq, tile_q0, scale * LOG2E, H, H, 0, window, 1.f,
      prefill_xcd_local(), (uint16_t*)out, tok_base, ldv, ldo, ex);
  return CFC_CHECK_LAUNCH();
}

// FP8 (e4m3fn) caches holding K / k_scale and V / v_scale; GQA-packed kernel only (G in 1,2,4,8)
CFC_API int cfc_prefill_attention_fp8(const void* q, const void* k_cache, const void* v_cache,
                                      const int32_t* block_tables, const int32_t* cu_q, const int32_t* ctx_lens,
                                      const int32_t* tile_seq, const int32_t* tile_q0, int n_tiles, int tile_rows,
                                      int Hq, int Hkv, int head_dim, int max_blocks, float scale, int window,
                                      float k_scale, float v_scale, void* out, hipStream_t stream) {
  if (head_dim != 128 || Hkv <= 0 || Hq % Hkv != 0 || window < 0) return -1;
  const int G = Hq / Hkv;
  if (!(G == 1 || G == 2 || G == 4 || G == 8) || tile_rows * G != 256) return -2;
  if (n_tiles <= 0) return 0;
  const dim3 grid(n_tiles, Hkv);
#define PF8_ARGS (const uint16_t*)q, k_cache, v_cache, block_tables, cu_q, ctx_lens, tile_seq, tile_q0, \
    scale * k_scale * LOG2E, Hq, Hkv, max_blocks, window, v_scale, prefill_xcd_local(), (uint16_t*)out
  switch (G) {
    case 1: prefill_gqa_kernel<1, true><<<grid, 512, 65536, stream>>>(PF8_ARGS); break;
    case 2: prefill_gqa_kernel<2, true><<<grid, 512, 65536, stream>>>(PF8_ARGS); break;
    case 4: prefill_gqa_kernel<4, true><<<grid, 512, 65536, stream>>>(PF8_ARGS); break;
    default: prefill_gqa_kernel<8, true><<<grid, 512, 65536, stream>>>(PF8_ARGS); break;
  }
#undef PF8_ARGS
  return CFC_CHECK_LAUNCH();
}

CFC_API int cfc_encoder_rows() { return ENC_ROWS; }

CFC_API int cfc_encoder_attention(const void* qkv, const int32_t* cu_seqlens, const int32_t* tile_seq,
                                  const int32_t* tile_q0, int n_tiles, int tile_rows, int H, int head_dim,
                                  int max_seqlen, float scale, void* out, hipStream_t stream) {
  if (tile_rows != ENC_ROWS) return -3;          // tiles cut for another kernel revision
  if (n_tiles <= 0) return 0;
  if (max_seqlen > 512) return -2;
  const int spad = (max_seqlen + 127) & ~127;
  const size_t lds = (size_t)spad * head_dim * 2 * 2;
#define ENC_GO(D, R)                                                                                                   \
  encoder_attn_kernel<D, R><<<dim3(n_tiles * H), 256, lds, stream>>>((const uint16_t*)qkv, cu_seqlens, tile_seq, tile_q0, \
                                                                     scale * LOG2E, H, (uint16_t*)out)
  if (head_dim == 32) {
    if (max_seqlen <= 128) ENC_GO(32, 2);
    else ENC_GO(32, 4);
  } else if (head_dim == 64) {
    if (max_seqlen <= 128) ENC_GO(64, 2);
    else ENC_GO(64, 4);
  } else {
    return -1;
  }
  return CFC_CHECK_LAUNCH();
}
