// Decode GEMM for gfx950 at batch sizes 5..256:  Y[M, N] = X[M, K] . W[N, K]^T  (bf16 in, fp32 acc).
//
// At decode a projection is a weight stream: W (14-235 MB per projection, the whole layer per
// token step) is read exactly once while X (M x K, <= 7 MB) stays in L2.  At M = 128 every weight
// byte carries 128 flops, so each CU must keep ~12 B/clk of W arriving AND run its MFMAs at ~40 %
// of peak.  What the measurements on this chip said (scripts/bench_dgemm.py --ablate):
//   * with the MFMAs removed an LDS-ring kernel was exactly as fast -- the limit is how the W bytes
//     are fetched, not the math;
//   * an LDS-DMA W ring of the workgroup's (4-6 stages in flight per CU) stayed at ~4.1-4.5 TB/s however deep.  (Rings of
//     a wave's own, read once and without barriers, bring keys and index rows at up to 6.8, lds_ring.h: not tried for W.)
// So here W never touches LDS:
//
//   * workgroup = BN/16 compute waves + 2 X-loader waves, tile = ALL M rows (BM = 16/32/64/96/128/256) x BN
//     W rows (BN = 64..128, chosen per shape so ~256 workgroups run: one per CU).  A batch of at most 16 or 32 rows
//     takes a tile of no more: in 64 rows X was half of W's bytes again through the CU, its LDS writes and reads four
//     times W's (us, 64-row tiles -> 16, of 5 rows: 4096 x 4096 9.4 -> 8.0, 6144 x 4096 11.7 -> 10.8, 28672 x 4096
//     38.7 -> 36.8, 4096 x 14336 21.6 -> 20.9; -> 32, of 24 rows: 9.4 -> 8.2, 12.0 -> 11.2, 40.2 -> 38.6, 22.0 -> 21.5).  65 .. 96 rows in 128 paid a third more of
//     X's traffic (two steps of four 7B layers, 81 rows 1093 -> 1040 us, 71 rows 1165 -> 1112);
//   * compute wave w owns 16 W rows and loads its B fragments straight from HBM into a D-stage
//     register ring (D = 8 x 64-deep K stages = 16 KB per wave in flight, the GEMV's depth).  Its
//     only vector-memory instructions are those loads, so hipcc's own counted vmcnt waits are
//     exact and never drain the ring; every load is unconditional (the tail re-reads the last
//     stage) so no branch joins force a vmcnt(0);
//   * X (an L2 hit, shared by all compute waves) is staged by the 2 loader waves with LDS-DMA
//     (`global_load_lds_dwordx4`, written in asm so hipcc orders nothing behind it) into an
//     NSX-slot LDS ring; only the loaders wait on vmcnt for it (counted, in one asm statement with
//     the s_barrier), so the X and W streams never serialise each other through the in-order
//     vmcnt counter;
//   * the X image is lane-linear per DMA piece and XOR-swizzled through the SOURCE address: chunk
//     c of row r at r*128 + ((c ^ (r & 7)) << 4), so the 16-row ds_read_b128 A-fragment reads are
//     bank-conflict free;
//   * split-K over the grid for the small-N projections; blocks are remapped XCD-locally so the
//     blocks of one XCD share a K slice and therefore the same X slice in that XCD's L2;
//   * epilogues: fp32 split-K partials (reduced by the residual + RMSNorm / SwiGLU reduce), bf16,
//     or SwiGLU over gate/up weights interleaved in 8-row groups (each 16-row n-tile = 8 gate +
//     8 up rows, so silu(g) * u is one lane swap away; same bf16 rounding points as
//     GEMM -> silu_mul).
//
// MFMA maps: A = X rows (m on lane & 15, k = 8 * (lane >> 4) + j), B = W rows (n on
// lane & 15, same k); C/D: n = lane & 15, m = 4 * (lane >> 4) + i.
#include <algorithm>

#include "common.h"

namespace {

typedef __attribute__((address_space(3))) void dg_lds_t;
typedef unsigned int dg_u32x4 __attribute__((ext_vector_type(4)));

// X-loader waves per workgroup: fill the workgroup up to 8 waves (2 per SIMD, 256 VGPRs each), at
// least one; two beside seven, though their ring of W is shorter for it (28672 x 4096 of 5 / 32 / 64 / 128 rows, us: 36.4 / 36.7 /
// 38.6 / 50.8 by one, 35.8 / 36.4 / 38.2 / 50.5 by two)
template <int BN>
constexpr int dg_loaders() { return BN / 16 >= 8 ? 1 : 2; }
// DG_PART_WT: the split-K slabs stored write-through (sc1): they reach memory while the kernel
// runs instead of as dirty L2 lines the kernel boundary must write back before the consumer (the
// residual + RMSNorm reduce, rope_kv) may start -- MI355X_MICROARCH "boundary": +B / 6 TB/s behind
// B dirty bytes, 2.8-3.8 us behind 12.6-16.8 MB of fp32 partials.
enum { DG_PART = 0, DG_BF16 = 1, DG_SILU = 2, DG_PART_WT = 3, DG_GLU = 4 };

// constants of the DG_GLU epilogue: min(g, limit) sigmoid(alpha g (1 + cubic g^2)) (clamp(u, +-limit) + beta)
struct DgGlu { float limit = 0.f, alpha = 1.f, beta = 0.f, cubic = 0.f; };

// MX (ablation 64): two X-loader waves and an 8-slot X ring whatever BN -- one loader wave's
// vmcnt window (63 pieces = 3 stages at BM = 128) may cap the X stream of the wide-BN shapes.
template <int BM, int BN, bool MX = false, bool EXPERTS = false>
struct DgShape {
  static constexpr int NW = BN / 16;                  // compute waves
  static constexpr int LOADERS = MX ? 2 : dg_loaders<BN>();
  static constexpr int WAVES = NW + LOADERS;
  static constexpr int MT = BM / 16;                  // m-tiles per compute wave
  // W register ring depth (64-deep stages); 9 waves (BN = 128) leave 168 VGPRs per lane
  static constexpr int D = BM == 256 ? 4 : (WAVES > 8 ? 6 : 8);
  static constexpr int XSTAGE = BM * 128;             // X bytes per 64-deep stage
  static constexpr int XP = BM / 8 / LOADERS;         // 1-KB DMA pieces per loader wave per stage
  // X ring slots; a loader keeps NSX - 2 stages in flight at its wait, and vmcnt counts at most 63 of its pieces.  X on its
  // way takes the place of W on its way: from 64 rows on four slots are faster than more (us of a 7B layer's four products,
  // 48 / 64 / 96 / 128 rows: 6 or 8 slots 81.9 / 83.4 / 91.0 / 104.6, 5 80.1 / 82.1 / 90.2 / 103.7, 4 79.7 / 81.4 / 89.5 / 103.5, 3 of 128 rows 106;
  // of 16 rows 8 slots 75.0, 4 75.5); not of experts' matrices, whose workgroups are several rounds (110 rows of pemolorn, a pass of
  // two steps: 4 slots 1968, more 1949)
  static constexpr int NSX_BASE = MX ? 8 : BM == 256 ? 4 : BM < 64 ? 8 : !EXPERTS ? 4 : BM == 128 ? 6 : 8;    // BM 16, 32: a ring of 16 is no faster
  static constexpr int NSX = (NSX_BASE - 2 <= 63 / XP ? NSX_BASE : 2 + 63 / XP);
};

__device__ __forceinline__ f32x4_t dg_mfma(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                 c, 0, 0, 0);
}

// One 1-KB LDS-DMA piece: lane l's 16 source bytes land at lds_addr + 16 l.  Inline asm, so hipcc
// sees no LDS write to order the compute waves' ds_reads behind; M0 (compiler-reserved) is saved
// and restored inside the statement.
__device__ __forceinline__ void dg_glds16(const void* gsrc, uint32_t lds_addr) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(gsrc), "s"(lds_addr)
               : "memory");
}

// loader waves: s_waitcnt vmcnt(n) + s_barrier as ONE statement (n = DMA pieces still allowed in flight)
template <int N>
__device__ __forceinline__ void dg_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(N) : "memory");
}

template <int P, int MAXA>
__device__ __forceinline__ void dg_wait_ahead(int ahead) {
  if constexpr (MAXA == 0) {
    dg_wait_barrier<0>();
  } else {
    if (ahead >= MAXA) dg_wait_barrier<MAXA * P>();
    else dg_wait_ahead<P, MAXA - 1>(ahead);
  }
}

// compute waves: their W loads stay in flight across the barrier; their LDS reads of the previous
// stage are retired first (hipcc may sink the MFMA that waits for them below an asm statement),
// so the loaders' next DMA into that slot cannot overtake them
__device__ __forceinline__ void dg_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// per-lane part of the offset in voff (one VGPR for the whole ring), the wave-uniform stage part in
// soff (an SGPR)
template <bool NT>
__device__ __forceinline__ uint4 dg_ldw_buf(__amdgpu_buffer_rsrc_t rs, int voff, int soff) {
  const dg_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, NT ? 2 : 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

template <bool NT>
__device__ __forceinline__ uint4 dg_ldw(const uint16_t* p) {
  if constexpr (NT) {
    const dg_u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const dg_u32x4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
  } else {
    return *reinterpret_cast<const uint4*>(p);
  }
}

// ABL: ablation builds for the timing probes only (scripts/bench_dgemm.py --ablate); 0 in production.
//   1 = no X DMA, 2 = no ds_read / MFMA (W loads kept live), 4 = no K-order rotation,
//   16 = X first: the loaders' first X stages enter the CU's memory pipeline before the compute
//   waves' W ring fill (one extra barrier), so the first MFMAs do not wait behind ~96 KB of W;
//   32 = contiguous W pieces: wave w loads fragments 2w, 2w+1 of the stage's 2 NW KB region (one
//   2-KB run per wave) instead of its own group's two 1-KB fragments NW KB apart (wrong sums);
//   64 = two X-loader waves + an 8-slot X ring (DgShape MX);
//   256 = the former tail (re-reads the last stage instead of issuing no loads);
//   128 = no workgroup barrier in the compute waves' stage loop (with 1 only: the loader waves
//   return at once) -- is the per-stage lockstep of the compute waves what slows the W stream?
// PACKED: W in the fragment-packed layout of cfc_dgemm_pack for this BN: tile-major, then 32-deep
// k group, then wave: Wp[N/BN][K/32][BN/16][64][8], so the 16 rows x 32 k of one MFMA B fragment
// are 1 KB contiguous in lane order and a workgroup's whole W slice (BN rows x its K range) is ONE
// contiguous span that its waves read front to back, 2 KB each per stage.  Measured
// (scripts/probes_stream.py, probes_flat.py): row-major fragments (16 rows x 64 B per instruction,
// 8 KB row stride) stream at 3.8-4.2 TB/s however deep the ring; contiguous 1-KB pieces at
// 6.0 TB/s from the same 224-256 workgroups.  Packed loads are buffer loads (32-bit offsets into
// the workgroup's span) so the cache policy can be set: NTW = nontemporal for these once-read
// bytes.
// GRP 1: one matrix per expert, W[experts][N][K] packed one after the other.  grid.y walks the row tiles of a
// batch sorted by expert: tile y multiplies rows y BM .. by matrix tile_expert[y] (negative: no such tile, the
// workgroup leaves), row m of it being row rows[m] of X (rows null: m itself); M counts the sorted rows.
// GRP 2: several inputs, X[inputs][M][K]: the BN rows of W tile n multiply input in_of[n].
struct DgGroup {
  const int32_t* rows = nullptr;
  const int32_t* tile_expert = nullptr;
  const int32_t* in_of = nullptr;
};

// Two workgroups per CU: the down products of a batch of experts are several rounds of short workgroups (16 .. 64 stages),
// whose starts the other one's stream covers; half the ring each, 96 VGPRs, 64 KB of LDS (us of 8 experts of 8192 x 2048:
// 58.7 -> 55.5, 64 rows 59.7 -> 56.8; gate / up, one round of 128 stages: no difference, one workgroup kept)
template <int BM, int EPI, int GRP>
constexpr bool dg_twice() { return BM <= 64 && GRP == 1 && EPI == DG_BF16; }

template <int BM, int BN, int EPI, bool NTW, int ABL = 0, bool PACKED = true, int GRP = 0>
__global__ void __launch_bounds__((64 * DgShape<BM, BN, (ABL & 64) != 0, GRP == 1>::WAVES), (dg_twice<BM, EPI, GRP>() ? 5 : 1))
    dgemm_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, int M, int N, int K, int ntiles,
                 int split, float* __restrict__ part, uint16_t* __restrict__ out, int ldo, DgGlu gp, DgGroup grp) {
  if constexpr (GRP == 1) {
    const int e = __builtin_amdgcn_readfirstlane(grp.tile_expert[blockIdx.y]);
    if (e < 0) return;
    W += (size_t)e * N * K;
  }
  using S = DgShape<BM, BN, (ABL & 64) != 0, GRP == 1>;
  constexpr int NW = S::NW;
  constexpr int D = dg_twice<BM, EPI, GRP>() ? 4 : S::D;
  __shared__ __attribute__((aligned(16))) char smem[S::NSX * S::XSTAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // logical block: the blocks of one XCD take consecutive ids, i.e. (mostly) one K slice
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int ks = lid / ntiles, tile = lid % ntiles;
  const int n0 = tile * BN, m0 = blockIdx.y * BM;
  if constexpr (GRP == 2) X += (size_t)__builtin_amdgcn_readfirstlane(grp.in_of[tile]) * M * K;
  const int nks = K >> 6;
  const int kb = (int)((long)ks * nks / split), ke = (int)((long)(ks + 1) * nks / split);
  const int nst = ke - kb;
  const int kq = lane >> 4;         // 8-element k group within a 32-deep MFMA step
  // K-order rotation: workgroup `lid` walks its K slice starting at stage `rot` and wraps around,
  // so the ~256 concurrent workgroups read different K offsets of their rows at any moment instead
  // of all hitting the same power-of-2-strided address set in lock step (the sum is order-free)
  const int rot = (ABL & 4) ? 0 : (int)((unsigned)lid * 37u % (unsigned)nst);
  auto phys = [&](int s) { s += rot; return s >= nst ? s - nst : s; };

  constexpr bool NOBAR = (ABL & 128) != 0;
  // XT: the MFMA's A operand is the W fragment, B the X fragment (probe 512: the former
  // orientation, X as A, one output element per lane per row -> 4-byte epilogue stores)
  constexpr bool XT = (ABL & 512) == 0;
  static_assert(!NOBAR || (ABL & 1), "no-barrier probe only without the X stream");
  if (w >= NW) {
    if constexpr (NOBAR) return;
    // ---------------- X loader wave, LDS-DMA: rows 8 XP l .. 8 XP (l+1) - 1 of the X stage image
    const int l = w - NW;
    const int prow = lane >> 3, pch = (lane & 7) ^ prow;   // row & 7 == prow for every piece
    const uint16_t* xsrc[S::XP];
#pragma unroll
    for (int i = 0; i < S::XP; ++i) {
      int m = min(m0 + 8 * S::XP * l + 8 * i + prow, M - 1);   // rows past M: results dropped
      if constexpr (GRP == 1)
        if (grp.rows) m = grp.rows[m];
      xsrc[i] = X + (size_t)m * K + (size_t)kb * 64 + 8 * pch;
    }
    const uint32_t lds0 =
        __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(dg_lds_t*)smem + 8 * S::XP * l * 128);
    auto issue = [&](int st, int slot) {
      if constexpr ((ABL & 1) != 0) return;
#pragma unroll
      for (int i = 0; i < S::XP; ++i) dg_glds16(xsrc[i] + phys(st) * 64, lds0 + slot * S::XSTAGE + i * 1024);
    };
#pragma unroll
    for (int p = 0; p < S::NSX - 1; ++p)
      if (p < nst) issue(p, p);
    if constexpr ((ABL & 16) != 0) asm volatile("s_barrier" ::: "memory");
    int slot = 0;
    for (int st = 0; st < nst; ++st) {
      if constexpr ((ABL & 1) != 0) dg_wait_barrier<0>();
      else dg_wait_ahead<S::XP, S::NSX - 2>(nst - 1 - st);
      // the slot read in iteration st-1 is free once every wave passed this barrier
      if (st + S::NSX - 1 < nst) issue(st + S::NSX - 1, slot == 0 ? S::NSX - 1 : slot - 1);
      slot = slot + 1 == S::NSX ? 0 : slot + 1;
    }
    return;
  }

  // ---------------- compute wave w: W rows n0 + 16 w + (lane & 15)
  uint4 ring[D][2];
  // packed: the workgroup's span, tile n0 / BN over all of K (split slices are sub-ranges of it),
  // as a buffer descriptor built from wave-uniform values (no waterfall loops)
  const uint16_t* span = W + (size_t)(n0 / BN) * ((size_t)BN * K);
  const uint32_t span_lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)span);
  const uint32_t span_hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)span >> 32));
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((uintptr_t)span_hi << 32) | span_lo), (short)0, PACKED ? BN * K * 2 : 0, 0x00020000);
  const int wvoff = lane * 16;                                                   // per-lane byte offset
  const int wsoff = __builtin_amdgcn_readfirstlane(((kb * 2) * NW + ((ABL & 32) ? 2 * w : w)) * 1024);
  // row-major: this lane's row and k offset
  const uint16_t* wp = W + (size_t)(n0 + 16 * w + (lane & 15)) * K + (size_t)kb * 64 + 8 * kq;
  // stage s of this lane: the kk = 0 and kk = 1 halves of its B fragments
  auto load_stage = [&](int s, uint4 (&dst)[2]) {
    if constexpr (PACKED) {
      const int so = __builtin_amdgcn_readfirstlane(wsoff + s * 2 * NW * 1024);
      dst[0] = dg_ldw_buf<NTW>(wrs, wvoff, so);
      dst[1] = dg_ldw_buf<NTW>(wrs, wvoff, so + ((ABL & 32) ? 1024 : NW * 1024));
    } else {
      dst[0] = dg_ldw<NTW>(wp + s * 64);
      dst[1] = dg_ldw<NTW>(wp + s * 64 + 32);
    }
  };
  // packed: logical stage s of the slice, or -- past its end -- zeros from an out-of-range buffer
  // offset (no memory access); the condition is wave-uniform, so this is a scalar select, no branch
  auto load_stage_past = [&](int s, uint4 (&dst)[2]) {
    const int so = __builtin_amdgcn_readfirstlane(s < nst ? wsoff + phys(s) * 2 * NW * 1024 : 0x40000000);
    dst[0] = dg_ldw_buf<NTW>(wrs, wvoff, so);
    dst[1] = dg_ldw_buf<NTW>(wrs, wvoff, so + ((ABL & 32) ? 1024 : NW * 1024));
  };
  if constexpr ((ABL & 16) != 0) asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int p = 0; p < D; ++p) {
    if constexpr (PACKED && (ABL & 256) == 0) load_stage_past(p, ring[p]);
    else load_stage(phys(min(p, nst - 1)), ring[p]);
  }
  f32x4_t acc[S::MT];
#pragma unroll
  for (int i = 0; i < S::MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int xoff = (lane & 15) * 128;
  const int sw = lane & 7;
  int xslot = 0;
  auto compute = [&](const uint4 (&b)[2]) {
    if constexpr ((ABL & 2) != 0) {
      asm volatile("" ::"v"(__builtin_bit_cast(dg_u32x4, b[0])), "v"(__builtin_bit_cast(dg_u32x4, b[1])));
    } else {
      const char* ximg = smem + xslot * S::XSTAGE + xoff;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int chunk = ((4 * kk + kq) ^ sw) << 4;
#pragma unroll
        for (int i = 0; i < S::MT; ++i) {
          const uint4 a = *reinterpret_cast<const uint4*>(ximg + i * 16 * 128 + chunk);
          // W fragment as the A operand: the 16 x 16 output tile comes out with four consecutive
          // W rows (output columns) of one X row per lane -> 16-byte epilogue stores
          acc[i] = XT ? dg_mfma(b[kk], a, acc[i]) : dg_mfma(a, b[kk], acc[i]);
        }
      }
    }
    xslot = xslot + 1 == S::NSX ? 0 : xslot + 1;
  };

  // Stage s lives in ring slot s % D; after computing stage s the slot is refilled with stage
  // s + D.  Every load is unconditional (a branch around a load makes hipcc drain the ring at the
  // join), so the last D refills of a slice name stages past its end: on the packed path they are
  // buffer loads at an offset past the descriptor's range, which return zeros without touching
  // memory (it re-read the last stage D times instead: up to half of a small
  // slice's loads, e.g. 8 redundant 2-KB stages per wave of qkv's 16 at split 4).  The ring is never
  // read past the slice (the tail computes only real stages).
  constexpr bool TAIL_RELOAD = (ABL & 256) != 0;    // probe: the former tail, which reads again
  int st = 0;
  // (in a plain loop hipcc makes 2 % more code of it: decode steps of four layers, 16 rows 837 -> 843 us, 64 986 -> 1000)
  auto round = [&]() {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if constexpr (!NOBAR) dg_barrier();   // X stage st+u is in LDS
      compute(ring[u]);
      if constexpr (PACKED && !TAIL_RELOAD) load_stage_past(st + u + D, ring[u]);
      else load_stage(phys(min(st + u + D, nst - 1)), ring[u]);
    }
    st += D;
  };
  while (st + D <= nst) round();
#pragma unroll
  for (int u = 0; u < D; ++u) {
    if (st + u < nst) {
      if constexpr (!NOBAR) dg_barrier();
      compute(ring[u]);
    }
  }

  if constexpr (XT) {
    // ---- epilogue: lane holds X row m0 + 16 i + (lane & 15) at the four consecutive W rows (output
    // columns) n0 + 16 w + 4 (lane >> 4) + r, r = 0..3 -- one 16-byte (fp32) / 8-byte (bf16) store per
    // lane and m-tile, 16 rows x 64 B per wave instruction (the former orientation stored 4 bytes
    // per lane: 4x the store instructions, the epilogue's store-issue tail of a small-N projection)
    const int mr = m0 + (lane & 15);
    const int nq = n0 + 16 * w + 4 * kq;
    if constexpr (EPI == DG_SILU || EPI == DG_GLU) {
      // 8-row interleave: W rows 0-7 of each 16-row group are gate, 8-15 the matching up rows, so the
      // lanes with kq < 2 hold gate rows and lane ^ 32 the up rows of the same output columns.  One
      // VALU lane swap (v_permlane32_swap) of (acc[0], acc[2]) hands every lane a (gate, up) pair --
      // column 0 in lanes kq < 2, column 2 in lanes kq >= 2 -- and one of (acc[1], acc[3]) columns
      // 1 / 3: each lane computes and stores two outputs
      const int oc = (n0 >> 1) + 8 * w + 4 * (kq & 1) + 2 * (kq >> 1);
      auto silu_mul = [&](float gate, float up) {
        if constexpr (EPI == DG_GLU) {
          const float gg = fminf(gate, gp.limit), uu = fminf(fmaxf(up, -gp.limit), gp.limit);
          return gg / (1.f + __expf(-gp.alpha * gg * (1.f + gp.cubic * gg * gg))) * (uu + gp.beta);
        }
        const float gt = bf2f(f2bf(gate)), u = bf2f(f2bf(up));
        return gt / (1.f + __expf(-gt)) * u;
      };
#pragma unroll
      for (int i = 0; i < S::MT; ++i) {
        float g0 = acc[i][0], u0 = acc[i][2], g1 = acc[i][1], u1 = acc[i][3];
        swap32(g0, u0);
        swap32(g1, u1);
        const int m = mr + 16 * i;
        if (m < M) *reinterpret_cast<uint32_t*>(out + (size_t)m * ldo + oc) = pack2bf(silu_mul(g0, u0), silu_mul(g1, u1));
      }
    } else if constexpr (EPI == DG_PART_WT) {
      // write-through (sc1) 16-byte stores through a buffer descriptor of the slab array (the
      // consumer kernel reads them from memory, no dirty lines at the boundary)
      const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)part);
      const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)part >> 32));
      const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(((uintptr_t)hi << 32) | lo), (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int i = 0; i < S::MT; ++i) {
        const int m = mr + 16 * i;
        if (m < M) {
          const dg_u32x4 v = {__float_as_uint(acc[i][0]), __float_as_uint(acc[i][1]), __float_as_uint(acc[i][2]),
                              __float_as_uint(acc[i][3])};
          __builtin_amdgcn_raw_buffer_store_b128(v, prs, (int)((((size_t)ks * M + m) * N + nq) * 4), 0, 16);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < S::MT; ++i) {
        const int m = mr + 16 * i;
        if (m < M) {
          if constexpr (EPI == DG_PART)
            *reinterpret_cast<float4*>(part + ((size_t)ks * M + m) * N + nq) =
                make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
          else
            *reinterpret_cast<uint2*>(out + (size_t)m * ldo + nq) =
                make_uint2(pack2bf(acc[i][0], acc[i][1]), pack2bf(acc[i][2], acc[i][3]));
        }
      }
    }
    return;
  }
  // ---- epilogue (the former orientation): lane holds rows m0 + 16 i + 4 (lane >> 4) + r of W row n
  const int n = n0 + 16 * w + (lane & 15);
  const int mb = m0 + 4 * kq;
  if constexpr (EPI == DG_SILU) {
    // 8-row interleave: lanes 0-7 of each 16 hold gate rows, lanes 8-15 the matching up rows
    const bool gate = (lane & 8) == 0;
    const int oc = (n0 >> 1) + 8 * w + (lane & 7);
#pragma unroll
    for (int i = 0; i < S::MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float up = __shfl_xor(acc[i][r], 8, 64);
        const int m = mb + 16 * i + r;
        if (gate && m < M) {
          const float gt = bf2f(f2bf(acc[i][r])), u = bf2f(f2bf(up));
          out[(size_t)m * ldo + oc] = f2bf(gt / (1.f + __expf(-gt)) * u);
        }
      }
  } else {
#pragma unroll
    for (int i = 0; i < S::MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mb + 16 * i + r;
        if (m < M) {
          if constexpr (EPI == DG_PART) part[((size_t)ks * M + m) * N + n] = acc[i][r];
          else if constexpr (EPI == DG_PART_WT) {    // vector store with sc1 (agent-scope relaxed)
            // the element goes through a scalar temporary: __builtin_bit_cast of the vector element
            // expression acc[i][r] itself compiled to element 0 for every r (hipcc, ROCm 7.2)
            const float v = acc[i][r];
            __hip_atomic_store(reinterpret_cast<uint32_t*>(part + ((size_t)ks * M + m) * N + n), __float_as_uint(v),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          else out[(size_t)m * ldo + n] = f2bf(acc[i][r]);
        }
      }
  }
}

// The same product with the whole packed matrix as ONE run of 64-deep stages, tile after tile, of which each of gridDim.x
// workgroups takes an equal share: for tiles x splits that are no whole number of rounds of 256 workgroups (a joint
// projection of 176 tiles took 10 slices a tile, 7 rounds of short workgroups, to come close).  A workgroup streams W
// without a stop across tile boundaries -- the packed tiles follow one another -- and stores its sums at each: the parts
// of a tile go to slabs 0, 1, .. in the order of their workgroups, the last of them filling the slabs that are left with
// zeros.  One round; `slabs`: the most workgroups that share a tile (cfc_dgemm_stream_slabs), 2 to 4 for the products it is
// planned for, up to K / 64 for few short tiles.  W tile n multiplies input in_of[n] (null: 0).
// us, 22528 x 4096 (185 MB, 31 at 5.9 TB/s): 5 rows 44.6 -> 33.8, 12 rows 40.5 -> 35.3; cfc_dgemm_slab_plan has more.
template <int BM, int BN>
__global__ void __launch_bounds__((64 * DgShape<BM, BN>::WAVES), 1)
    dgemm_stream_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, int M, int N, int K, int slabs,
                        float* __restrict__ part, const int32_t* __restrict__ in_of) {
  using S = DgShape<BM, BN>;
  constexpr int NW = S::NW, D = S::D;
  __shared__ __attribute__((aligned(16))) char smem[S::NSX * S::XSTAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nks = K >> 6, G = gridDim.x, id = xcd_remap(blockIdx.x, G);
  const int64_t U = (int64_t)(N / BN) * nks;
  const int64_t u0 = id * U / G;
  const int nst = (int)((id + 1) * U / G - u0);
  if (nst == 0) return;
  const int tile0 = (int)(u0 / nks), k0 = (int)(u0 % nks);
  const int kq = lane >> 4;

  if (w >= NW) {
    // ---------------- X loader wave (as dgemm_kernel's)
    const int l = w - NW;
    const int prow = lane >> 3, pch = (lane & 7) ^ prow;
    const uint16_t* xsrc[S::XP];
#pragma unroll
    for (int i = 0; i < S::XP; ++i)
      xsrc[i] = X + (size_t)min(8 * S::XP * l + 8 * i + prow, M - 1) * K + 8 * pch;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(dg_lds_t*)smem + 8 * S::XP * l * 128);
    int k = k0, tile = tile0;
    auto input = [&]() { return in_of ? (size_t)__builtin_amdgcn_readfirstlane(in_of[tile]) * M * K : (size_t)0; };
    size_t in = input();
    auto issue = [&](int slot) {
#pragma unroll
      for (int i = 0; i < S::XP; ++i) dg_glds16(xsrc[i] + in + (size_t)k * 64, lds0 + slot * S::XSTAGE + i * 1024);
      if (++k == nks) {
        k = 0;
        if (++tile < N / BN) in = input();
      }
    };
#pragma unroll
    for (int p = 0; p < S::NSX - 1; ++p)
      if (p < nst) issue(p);
    int slot = 0;
    for (int st = 0; st < nst; ++st) {
      dg_wait_ahead<S::XP, S::NSX - 2>(nst - 1 - st);
      if (st + S::NSX - 1 < nst) issue(slot == 0 ? S::NSX - 1 : slot - 1);
      slot = slot + 1 == S::NSX ? 0 : slot + 1;
    }
    return;
  }

  // ---------------- compute wave w: W rows 16 w + (lane & 15) of the current tile
  uint4 ring[D][2];
  // a descriptor of this workgroup's run of stages (2 NW KB each)
  const uint16_t* span = W + (size_t)u0 * BN * 64;
  const uint32_t span_lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)span);
  const uint32_t span_hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)span >> 32));
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(((uintptr_t)span_hi << 32) | span_lo), (short)0, nst * BN * 128, 0x00020000);
  const int wvoff = lane * 16, wsoff = w * 1024;
  // past the run: zeros from an out-of-range offset, no memory access
  auto load_stage = [&](int s, uint4 (&dst)[2]) {
    const int so = __builtin_amdgcn_readfirstlane(s < nst ? wsoff + s * 2 * NW * 1024 : 0x40000000);
    dst[0] = dg_ldw_buf<true>(wrs, wvoff, so);
    dst[1] = dg_ldw_buf<true>(wrs, wvoff, so + NW * 1024);
  };
#pragma unroll
  for (int p = 0; p < D; ++p) load_stage(p, ring[p]);
  f32x4_t acc[S::MT];
#pragma unroll
  for (int i = 0; i < S::MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int xoff = (lane & 15) * 128, sw = lane & 7;
  int xslot = 0, tile = tile0, left = nks - k0;

  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)part);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)part >> 32));
  const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc((void*)(((uintptr_t)hi << 32) | lo), (short)0, 0x7fffffff, 0x00020000);
  auto flush = [&](bool whole) {
    // the workgroup that has the tile's first stage
    const int first = (int)((((int64_t)tile * nks + 1) * G - 1) / U);
    const int at = id - first, end = whole ? slabs : at + 1;
    const int mr = lane & 15, nq = tile * BN + 16 * w + 4 * kq;
    for (int s = at; s < end; ++s)
#pragma unroll
      for (int i = 0; i < S::MT; ++i) {
        const int m = mr + 16 * i;
        if (m < M) {
          const dg_u32x4 v = s == at ? dg_u32x4{__float_as_uint(acc[i][0]), __float_as_uint(acc[i][1]), __float_as_uint(acc[i][2]),
                                                __float_as_uint(acc[i][3])} : dg_u32x4{0u, 0u, 0u, 0u};
          __builtin_amdgcn_raw_buffer_store_b128(v, prs, (int)((((size_t)s * M + m) * N + nq) * 4), 0, 16);
        }
      }
#pragma unroll
    for (int i = 0; i < S::MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    ++tile;
    left = nks;
  };
  auto compute = [&](const uint4 (&b)[2]) {
    const char* ximg = smem + xslot * S::XSTAGE + xoff;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int chunk = ((4 * kk + kq) ^ sw) << 4;
#pragma unroll
      for (int i = 0; i < S::MT; ++i) acc[i] = dg_mfma(b[kk], *reinterpret_cast<const uint4*>(ximg + i * 16 * 128 + chunk), acc[i]);
    }
    xslot = xslot + 1 == S::NSX ? 0 : xslot + 1;
  };
  int st = 0;
  for (; st + D <= nst; st += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      dg_barrier();
      compute(ring[u]);
      load_stage(st + u + D, ring[u]);
      if (--left == 0) flush(true);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u) {
    if (st + u < nst) {
      dg_barrier();
      compute(ring[u]);
      if (--left == 0) flush(true);
    }
  }
  if (left < nks) flush(false);
}

constexpr bool DG_NT = true;    // nontemporal packed weight stream (bench_dgemm --ablate: ~10 % faster)

template <int BM, int BN, bool NTW, int ABL, bool PK>
int dgemm_launch_bn(const void* x, const void* w, int M, int N, int K, int split, int epi, float* part, void* out,
                    int ldo, hipStream_t stream) {
  const int ntiles = N / BN;
  const dim3 grid(ntiles * split, (M + BM - 1) / BM);
  const int threads = 64 * DgShape<BM, BN, (ABL & 64) != 0>::WAVES;
#define DG_ARGS (const uint16_t*)x, (const uint16_t*)w, M, N, K, ntiles, split, part, (uint16_t*)out, ldo, DgGlu{}, DgGroup{}
  switch (epi) {
    case DG_PART: dgemm_kernel<BM, BN, DG_PART, NTW, ABL, PK><<<grid, threads, 0, stream>>>(DG_ARGS); break;
    case DG_PART_WT: dgemm_kernel<BM, BN, DG_PART_WT, NTW, ABL, PK><<<grid, threads, 0, stream>>>(DG_ARGS); break;
    case DG_BF16: dgemm_kernel<BM, BN, DG_BF16, NTW, ABL, PK><<<grid, threads, 0, stream>>>(DG_ARGS); break;
    case DG_SILU: dgemm_kernel<BM, BN, DG_SILU, NTW, ABL, PK><<<grid, threads, 0, stream>>>(DG_ARGS); break;
    default: return -3;
  }
#undef DG_ARGS
  return 0;
}

template <int BM, bool NTW, int ABL, bool PK>
int dgemm_launch_pk(const void* x, const void* w, int M, int N, int K, int split, int epi, int bn, float* part,
                    void* out, int ldo, hipStream_t stream) {
  switch (bn) {
    case 64: return dgemm_launch_bn<BM, 64, NTW, ABL, PK>(x, w, M, N, K, split, epi, part, out, ldo, stream);
    case 96: return dgemm_launch_bn<BM, 96, NTW, ABL, PK>(x, w, M, N, K, split, epi, part, out, ldo, stream);
    case 112: return dgemm_launch_bn<BM, 112, NTW, ABL, PK>(x, w, M, N, K, split, epi, part, out, ldo, stream);
    case 128: return dgemm_launch_bn<BM, 128, NTW, ABL, PK>(x, w, M, N, K, split, epi, part, out, ldo, stream);
    default: return -5;
  }
}

// packed weights stream nontemporal (NTW); row-major ones keep the default policy
template <int BM, int ABL = 0>
int dgemm_launch(const void* x, const void* w, int M, int N, int K, int split, int epi, int bn, int packed,
                 float* part, void* out, int ldo, hipStream_t stream) {
  return packed ? dgemm_launch_pk<BM, DG_NT, ABL, true>(x, w, M, N, K, split, epi, bn, part, out, ldo, stream)
                : dgemm_launch_pk<BM, false, ABL, false>(x, w, M, N, K, split, epi, bn, part, out, ldo, stream);
}

// Fragment-pack a row-major W[N][K] for workgroups of nw = BN/16 waves:
// Wp[t][kg][w][l][j] = W[BN t + 16 w + (l & 15)][32 kg + 8 (l >> 4) + j].  One thread per 16-B piece.
__global__ void dgemm_pack_kernel(const uint16_t* __restrict__ W, uint16_t* __restrict__ Wp, int N, int K, int nw) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total = (size_t)N * K / 8;
  if (i >= total) return;
  const int l = (int)(i & 63);
  const size_t frag = i >> 6;
  const int kgs = K / 32;
  const int w = (int)(frag % nw);
  const size_t t2 = frag / nw;
  const int kg = (int)(t2 % kgs), t = (int)(t2 / kgs);
  const int row = 16 * (t * nw + w) + (l & 15);
  const uint4 v = *reinterpret_cast<const uint4*>(W + (size_t)row * K + 32 * kg + 8 * (l >> 4));
  reinterpret_cast<uint4*>(Wp)[i] = v;
}

int dgemm_check(int M, int N, int K, int split, int epi, int bn, const float* part, const void* out, int ldo) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 64 || split < 1 || split > K / 64) return -1;
  if (bn != 64 && bn != 96 && bn != 112 && bn != 128) return -5;
  if (N % bn) return -1;
  const bool slabs = epi == DG_PART || epi == DG_PART_WT;
  if (!slabs && split != 1) return -2;
  if ((slabs && !part) || (!slabs && !out)) return -2;
  // the epilogue stores 4 consecutive outputs per lane: 16-byte fp32 / 8-byte bf16 aligned rows
  if ((slabs && ((uintptr_t)part & 15)) || (!slabs && (((uintptr_t)out & 7) || ldo % 4))) return -2;
  return 0;
}

}  // namespace

// Which row tile (16 / 32 / 64 / 96 / 128 / 256; 64, 128 or 256 of a row-major W) a batch of M rows runs with (M > 256 loops 256-row tiles over grid.y).
CFC_API int cfc_dgemm_bm(int M) { return M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : M <= 96 ? 96 : M <= 128 ? 128 : 256; }

// epi 0: fp32 split-K partials into part[split][M][N]; 1: bf16 into out (row stride ldo, split 1);
// 2: SwiGLU over 8-row interleaved gate/up W -> bf16 [M, N/2] into out (split 1); 3: as 0 with
// write-through (sc1) slab stores.
// bn (W rows per workgroup) in {64, 96, 112, 128}, N % bn == 0, K % 64 == 0, 1 <= split <= K / 64.
// packed: w is in the fragment-packed layout cfc_dgemm_pack wrote for this same bn (else row-major [N][K]).
CFC_API int cfc_dgemm(const void* x, const void* w, int M, int N, int K, int split, int epi, int bn, int packed,
                      float* part, void* out, int ldo, hipStream_t stream) {
  if (const int e = dgemm_check(M, N, K, split, epi, bn, part, out, ldo)) return e;
  int rc;
  const int bm = cfc_dgemm_bm(M);
  switch (packed ? bm : bm == 96 ? 128 : std::max(64, bm)) {
    case 16: rc = dgemm_launch_pk<16, DG_NT, 0, true>(x, w, M, N, K, split, epi, bn, part, out, ldo, stream); break;
    case 32: rc = dgemm_launch_pk<32, DG_NT, 0, true>(x, w, M, N, K, split, epi, bn, part, out, ldo, stream); break;
    case 96: rc = dgemm_launch_pk<96, DG_NT, 0, true>(x, w, M, N, K, split, epi, bn, part, out, ldo, stream); break;
    case 64: rc = dgemm_launch<64>(x, w, M, N, K, split, epi, bn, packed, part, out, ldo, stream); break;
    case 128: rc = dgemm_launch<128>(x, w, M, N, K, split, epi, bn, packed, part, out, ldo, stream); break;
    default: rc = dgemm_launch<256>(x, w, M, N, K, split, epi, bn, packed, part, out, ldo, stream); break;
  }
  return rc ? rc : CFC_CHECK_LAUNCH();
}

// Row-major W[N][K] bf16 -> the fragment-packed layout for bn-row workgroups (same size; the
// packed weight is only valid with that bn).  N % bn == 0, bn % 16 == 0, K % 64 == 0.
namespace {
template <int BM, int BN>
void dgemm_glu_go(const void* x, const void* w, int M, int N, int K, void* out, int ldo, const DgGlu& gp, hipStream_t stream) {
  dgemm_kernel<BM, BN, DG_GLU, DG_NT, 0, true><<<dim3(N / BN, (M + BM - 1) / BM), 64 * DgShape<BM, BN>::WAVES, 0, stream>>>(
      (const uint16_t*)x, (const uint16_t*)w, M, N, K, N / BN, 1, nullptr, (uint16_t*)out, ldo, gp, DgGroup{});
}
template <int BM>
int dgemm_glu_bn(const void* x, const void* w, int M, int N, int K, int bn, void* out, int ldo, const DgGlu& gp,
                 hipStream_t stream) {
  switch (bn) {
    case 64: dgemm_glu_go<BM, 64>(x, w, M, N, K, out, ldo, gp, stream); return 0;
    case 96: dgemm_glu_go<BM, 96>(x, w, M, N, K, out, ldo, gp, stream); return 0;
    case 112: dgemm_glu_go<BM, 112>(x, w, M, N, K, out, ldo, gp, stream); return 0;
    case 128: dgemm_glu_go<BM, 128>(x, w, M, N, K, out, ldo, gp, stream); return 0;
  }
  return -5;
}
}  // namespace

// Clamped GLU epilogue over packed, 8-row interleaved gate / up weights: out [M, N / 2] (row stride ldo)
CFC_API int cfc_dgemm_glu(const void* x, const void* w, int M, int N, int K, int bn, void* out, int ldo, float limit,
                          float alpha, float beta, float cubic, hipStream_t stream) {
  if (const int e = dgemm_check(M, N, K, 1, DG_GLU, bn, nullptr, out, ldo)) return e;
  DgGlu gp;
  gp.limit = limit; gp.alpha = alpha; gp.beta = beta; gp.cubic = cubic;
  int rc;
  switch (cfc_dgemm_bm(M)) {
    case 16: rc = dgemm_glu_bn<16>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
    case 32: rc = dgemm_glu_bn<32>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
    case 96: rc = dgemm_glu_bn<96>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
    case 64: rc = dgemm_glu_bn<64>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
    case 128: rc = dgemm_glu_bn<128>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
    default: rc = dgemm_glu_bn<256>(x, w, M, N, K, bn, out, ldo, gp, stream); break;
  }
  return rc ? rc : CFC_CHECK_LAUNCH();
}

namespace {
template <int BM, int BN>
void dgemm_group_go(int glu, const void* x, const void* w, int M, int N, int K, void* out, int ldo, const DgGlu& gp,
                    const DgGroup& g, hipStream_t stream) {
  const dim3 grid(N / BN, M / BM);
  constexpr int threads = 64 * DgShape<BM, BN, false, true>::WAVES;
  if (glu)
    dgemm_kernel<BM, BN, DG_GLU, DG_NT, 0, true, 1><<<grid, threads, 0, stream>>>(
        (const uint16_t*)x, (const uint16_t*)w, M, N, K, N / BN, 1, nullptr, (uint16_t*)out, ldo, gp, g);
  else
    dgemm_kernel<BM, BN, DG_BF16, DG_NT, 0, true, 1><<<grid, threads, 0, stream>>>(
        (const uint16_t*)x, (const uint16_t*)w, M, N, K, N / BN, 1, nullptr, (uint16_t*)out, ldo, gp, g);
}
template <int BM>
int dgemm_group_bn(int glu, const void* x, const void* w, int M, int N, int K, int bn, void* out, int ldo, const DgGlu& gp,
                   const DgGroup& g, hipStream_t stream) {
  switch (bn) {
    case 64: dgemm_group_go<BM, 64>(glu, x, w, M, N, K, out, ldo, gp, g, stream); return 0;
    case 128: dgemm_group_go<BM, 128>(glu, x, w, M, N, K, out, ldo, gp, g, stream); return 0;
  }
  return -5;
}
}  // namespace

// Products of rows sorted by expert with W[experts][N][K] (each packed for bn): M sorted rows in tiles of bm = 16, 32, 64 or
// 128, rows / tile_expert as in DgGroup.  bf16 out of row stride ldo: [M][N], or (glu) the clamped GLU of 8-row
// interleaved gate / up rows [M][N / 2]
CFC_API int cfc_dgemm_group(int glu, const void* x, const void* w, int M, int N, int K, int bn, int bm, const int32_t* rows,
                            const int32_t* tile_expert, void* out, int ldo, float limit, float alpha, float beta,
                            hipStream_t stream) {
  if (M == 0) return 0;
  if (const int e = dgemm_check(M, N, K, 1, glu ? DG_GLU : DG_BF16, bn, nullptr, out, ldo)) return e;
  if (!tile_expert || (bm != 16 && bm != 32 && bm != 64 && bm != 128) || M % bm) return -1;
  DgGlu gp;
  gp.limit = limit; gp.alpha = alpha; gp.beta = beta;
  DgGroup g;
  g.rows = rows; g.tile_expert = tile_expert;
  int rc;
  switch (bm) {
    case 16: rc = dgemm_group_bn<16>(glu, x, w, M, N, K, bn, out, ldo, gp, g, stream); break;
    case 32: rc = dgemm_group_bn<32>(glu, x, w, M, N, K, bn, out, ldo, gp, g, stream); break;
    case 64: rc = dgemm_group_bn<64>(glu, x, w, M, N, K, bn, out, ldo, gp, g, stream); break;
    default: rc = dgemm_group_bn<128>(glu, x, w, M, N, K, bn, out, ldo, gp, g, stream); break;
  }
  return rc ? rc : CFC_CHECK_LAUNCH();
}

namespace {
template <int BM>
int dgemm_joint_bn(const void* x, const void* w, int M, int N, int K, int split, int bn, float* part, const DgGroup& g,
                   hipStream_t stream) {
#define DJ(BN)                                                                                                       \
  case BN:                                                                                                           \
    dgemm_kernel<BM, BN, DG_PART_WT, DG_NT, 0, true, 2>                                                              \
        <<<dim3(N / BN * split, (M + BM - 1) / BM), 64 * DgShape<BM, BN>::WAVES, 0, stream>>>(                       \
            (const uint16_t*)x, (const uint16_t*)w, M, N, K, N / BN, split, part, nullptr, 0, DgGlu{}, g);           \
    return 0;
  switch (bn) { DJ(64) DJ(128) }
#undef DJ
  return -5;
}
}  // namespace

// fp32 split-K slabs part[split][M][N] of X[inputs][M][K], the bn rows of W tile n multiplying input in_of[n]
CFC_API int cfc_dgemm_joint(const void* x, const void* w, int M, int N, int K, int split, int bn, const int32_t* in_of,
                            float* part, hipStream_t stream) {
  if (const int e = dgemm_check(M, N, K, split, DG_PART_WT, bn, part, nullptr, N)) return e;
  if (!in_of) return -1;
  DgGroup g;
  g.in_of = in_of;
  int rc;
  switch (cfc_dgemm_bm(M)) {
    case 16: rc = dgemm_joint_bn<16>(x, w, M, N, K, split, bn, part, g, stream); break;
    case 32: rc = dgemm_joint_bn<32>(x, w, M, N, K, split, bn, part, g, stream); break;
    case 96: rc = dgemm_joint_bn<96>(x, w, M, N, K, split, bn, part, g, stream); break;
    case 64: rc = dgemm_joint_bn<64>(x, w, M, N, K, split, bn, part, g, stream); break;
    case 128: rc = dgemm_joint_bn<128>(x, w, M, N, K, split, bn, part, g, stream); break;
    default: rc = dgemm_joint_bn<256>(x, w, M, N, K, split, bn, part, g, stream); break;
  }
  return rc ? rc : CFC_CHECK_LAUNCH();
}

// Slabs of cfc_dgemm_stream: the most workgroups that share one tile.
CFC_API int cfc_dgemm_stream_slabs(int N, int K, int bn) {
  if (N <= 0 || K < 64 || K % 64 || bn <= 0 || N % bn) return -1;
  const int64_t nks = K / 64, U = (int64_t)(N / bn) * nks, G = std::min<int64_t>(256, U);
  int most = 1;
  for (int64_t t = 0; t < N / bn; ++t)
    most = std::max(most, (int)((((t + 1) * nks) * G - 1) / U - ((t * nks + 1) * G - 1) / U) + 1);
  return most;
}

// dgemm_stream_kernel: x [inputs][M][K], M <= 64, W packed for bn = 64 or 128, part [cfc_dgemm_stream_slabs][M][N]
CFC_API int cfc_dgemm_stream(const void* x, const void* w, int M, int N, int K, int bn, const int32_t* in_of, float* part,
                             hipStream_t stream) {
  if (const int e = dgemm_check(M, N, K, 1, DG_PART_WT, bn, part, nullptr, N)) return e;
  const int slabs = cfc_dgemm_stream_slabs(N, K, bn);
  if (M > 64 || (bn != 64 && bn != 128) || (int64_t)slabs * M * N * 4 > 0x7fffffff || (int64_t)N * K * 2 / 256 > 0x3ff00000) return -1;
#define DG_STREAM(BM, BN)                                                                                       \
  dgemm_stream_kernel<BM, BN><<<(int)std::min<int64_t>(256, (int64_t)(N / BN) * (K / 64)), 64 * DgShape<BM, BN>::WAVES, 0, stream>>>((const uint16_t*)x, (const uint16_t*)w, M, \
                                                                              N, K, slabs, part, in_of)
  switch (cfc_dgemm_bm(M) * 1000 + bn) {
    case 16064: DG_STREAM(16, 64); break;
    case 16128: DG_STREAM(16, 128); break;
    case 32064: DG_STREAM(32, 64); break;
    case 32128: DG_STREAM(32, 128); break;
    case 64064: DG_STREAM(64, 64); break;
    default: DG_STREAM(64, 128); break;
  }
#undef DG_STREAM
  return CFC_CHECK_LAUNCH();
}

CFC_API int cfc_dgemm_pack(const void* w, void* wp, int N, int K, int bn, hipStream_t stream) {
  if (N <= 0 || K <= 0 || bn <= 0 || bn % 16 || N % bn || K % 64 || w == wp) return -1;
  const size_t pieces = (size_t)N * K / 8;
  dgemm_pack_kernel<<<(unsigned)((pieces + 255) / 256), 256, 0, stream>>>((const uint16_t*)w, (uint16_t*)wp, N, K,
                                                                           bn / 16);
  return CFC_CHECK_LAUNCH();
}

// Timing probe only (scripts/bench_dgemm.py --ablate): split-K partial GEMM at BM = 128 on a
// packed weight, ablation bits `abl` (1 no X DMA, 2 no MFMA, 4 no K rotation); +8 = default
// (not nontemporal) cache policy on the weight stream.
CFC_API int cfc_dgemm_ablate(const void* x, const void* w, int M, int N, int K, int split, int bn, int abl,
                             float* part, hipStream_t stream) {
  if (M > 128 || (abl & ~1023)) return -1;
  if (const int e = dgemm_check(M, N, K, split, DG_PART, bn, part, nullptr, N)) return e;
  int rc;
  switch (abl) {
#define DG_ABL(A, NT) rc = dgemm_launch_pk<128, NT, A, true>(x, w, M, N, K, split, 0, bn, part, nullptr, 0, stream); break;
    case 0: DG_ABL(0, true)
    case 1: DG_ABL(1, true)
    case 2: DG_ABL(2, true)
    case 3: DG_ABL(3, true)
    case 4: DG_ABL(4, true)
    case 7: DG_ABL(7, true)
    case 8: DG_ABL(0, false)
    case 11: DG_ABL(3, false)
    case 16: DG_ABL(16, true)
    case 32: DG_ABL(32, true)
    case 35: DG_ABL(35, true)
    case 64: DG_ABL(64, true)
    case 96: DG_ABL(96, true)
    case 129: DG_ABL(129, true)
    case 131: DG_ABL(131, true)
    case 256: DG_ABL(256, true)
    case 259: DG_ABL(259, true)
    case 512: DG_ABL(512, true)
#undef DG_ABL
    default: return -3;
  }
  return rc ? rc : CFC_CHECK_LAUNCH();
}

namespace {
constexpr int DG_CUS = 256;                // one workgroup per CU

// us of one launch of dgemm_kernel with its slabs written and read back once: each workgroup streams its W slice from
// HBM at a per-CU rate and re-reads its X slice (all bm rows of its K range: X traffic / W traffic = bm / bn) from L2 at
// a per-CU rate, in ceil(blocks / CUs) rounds (a partial second round doubles the time of the CUs that run it).  Rates
// fitted to sweeps of 64 .. 256 rows; each round after the first costs 1.5 for its start (14336 x 4096, 5 rows: 4 rounds
// of 9 slices 28.7, one of 2 slices 21.6).
double dgemm_us(int M, int N, int K, int bn, int split) {
  constexpr double CU_RATE = 25e3;         // W bytes/us one workgroup streams (6.4 TB/s over 256 CUs)
  constexpr double PART_RATE = 6e6;        // fp32 partial slab traffic
  constexpr double X_RATE = 90e3;          // per-CU L2 -> LDS rate of the X re-reads (ablation: X costs ~12 us of gate/up)
  const int bm = M <= 64 ? 64 : M <= 128 ? 128 : 256;   // the tiles of 16 and 32 rows keep the splits of 64 (no other was faster), 96 those of 128
  const int64_t blocks = (int64_t)(N / bn) * ((M + bm - 1) / bm) * split;
  const double rounds = (double)((blocks + DG_CUS - 1) / DG_CUS);
  double t = rounds * ((double)bn * K * 2 / split / CU_RATE + (double)bm * K * 2 / split / X_RATE) + 1.5 * (rounds - 1.0);
  if (split > 1) t += 2.0 * split * M * N * 4 / PART_RATE;
  return t;
}

// us of dgemm_stream_kernel, as measured for 5 .. 64 rows of 9216 .. 22528 columns (within 8 %): 23.5 B/ns of W per CU,
// a quarter of a percent more per row
double dgemm_stream_us(int M, int N, int K, int bn, int slabs) {
  const double stages = (double)(N / bn) * (K / 64) / DG_CUS;
  return 2.5 + stages * bn * 128 / 23.5e3 * (1.0 + 0.0024 * M) + 2.0 * slabs * M * N * 4 / 6e6;
}

double dgemm_best(int M, int N, int K, int swiglu, int bn, int* cfg) {
  const int widths[4] = {bn ? bn : 128, 112, 96, 64};
  double best = -1.0;
  for (int c = 0; c < (bn ? 1 : 4); ++c) {
    const int w = widths[c];
    if (N % w) continue;
    for (int split = 1; split <= (swiglu ? 1 : K / 64); ++split) {
      const double t = dgemm_us(M, N, K, w, split);
      if (best < 0 || t < best - 1e-6) best = t, cfg[0] = w, cfg[1] = split;
    }
  }
  return best;
}
}  // namespace

// cfg = {W rows per workgroup, split-K} of one projection.  A fused SwiGLU epilogue needs split 1.  bn: the width of a
// packed W, 0 to choose it too.  In C because a prompt asks for every product of its row count (K = 14336: 80 us as a
// Python loop, 1 here).
CFC_API int cfc_dgemm_config(int M, int N, int K, int swiglu, int bn, int* cfg) {
  if (M < 1 || N < 1 || K < 1 || bn < 0) return -1;
  return dgemm_best(M, N, K, swiglu, bn, cfg) < 0 ? -1 : 0;
}

// plan = {slabs, 1 for dgemm_stream_kernel} of a product that leaves fp32 slabs, W packed for bn.  The stream where it
// is 7 % faster or more, which it is where no split makes whole rounds (us, 5 / 64 rows, split -> stream: 22528 x 4096
// 44.6 / 40.2 -> 33.8 / 42.9, 18432 33.4 / 37.2 -> 27.9 / 35.0, 9216 in 64-row tiles 26.5 / 23.3 -> 15.7 / 20.9) and not
// where one does (4096 x 14336: 21.8 / 23.0 -> 22.6 / 27.7; 2048 x 4096 in 64-row tiles is faster in a loop, 7.8 -> 7.3,
// but slower in a layer, 6.9 -> 7.6: each XCD then needs all of the X that was just written, not one K slice of it);
// above 64 rows its workgroups wait for X.  Nor where one slice fills the round: 28672 x 4096, 5 / 16 rows 44.3 / 44.8 ->
// 44.9 / 47.9, of which dgemm_us thinks 3 more.
CFC_API int cfc_dgemm_slab_plan(int M, int N, int K, int bn, int* plan) {
  int cfg[2];
  if (M < 1 || N < 1 || K < 1 || bn < 1) return -1;
  const double t = dgemm_best(M, N, K, 0, bn, cfg);
  if (t < 0) return -1;
  plan[0] = cfg[1], plan[1] = 0;
  if (M > 64 || (bn != 64 && bn != 128) || K % 64 || cfg[1] == 1) return 0;
  const int slabs = cfc_dgemm_stream_slabs(N, K, bn);
  if ((int64_t)slabs * M * N * 4 > 0x7fffffff) return 0;
  if (dgemm_stream_us(M, N, K, bn, slabs) < 0.93 * t) plan[0] = slabs, plan[1] = 1;
  return 0;
}
