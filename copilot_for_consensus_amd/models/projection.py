"""One weight matrix and the products a model takes with it, on the kernel that fits the row count.

Up to 128 rows run on the decode GEMM, thousands on the prefill GEMM's 256 x 256 tiles, what lies between on the GEMM
for a few hundred rows (K.prompt_plan), all three reading one fragment-packed bf16 copy.  (One to four rows, too: with its
tile of 16 rows the decode GEMM takes 29 us where the packed GEMV takes 32 to 38, 20608 x 4096, 4.8 where it takes 5.2 to
8.2, 4096 x 1536; and it gates and clamps in its epilogue.  A narrow matrix of long rows only fills the chip in so many
slabs that their sum takes longer than the product: NARROW_SLABS.)  Shapes those kernels do not take (N or K not a multiple
of 64) and 32-bit weights use the library product.  CPU tensors: torch.
"""
from __future__ import annotations

import os

import torch
import torch.nn.functional as F

from ..ops import kernels as K
from ..ops.cols import Cols
from ..ops.stream import clamped_glu, relu_sq


# One to four rows whose product the decode GEMM would cut into more slabs than this run on the packed GEMV, whose workgroup
# reads longer rows: us of product and sum, one and four rows, GEMM -> GEMV, 64 x 4096 in 64 slabs 10.1 -> 7.1 and 10.3 -> 7.0,
# 256 x 7168 in 64 10.5 -> 7.3 and 11.6 -> 8.3, 576 x 4096 in 28 8.2 -> 7.5 and 8.8 -> 7.5; with 16 the GEMM is ahead, 1024 x 4096 7.1
# and 7.4 where the GEMV takes 7.7 and 7.6.
NARROW_SLABS = 16


class Projection:
    """y = x W^T for W [N, K], sharded by the caller.  bf16 on the GPU: packed when the shape fits."""

    # swiglu: interleaved gate / up rows, tiled for a product without split (its epilogue gates)
    __slots__ = ("w", "packed", "N", "K", "min_tiles")

    def __init__(self, w: torch.Tensor, decode_rows: int = 128, swiglu: bool = False):
        self.N, self.K = w.shape
        self.packed = None
        self.w = w.contiguous()
        # fewer 256 x 256 output tiles than this run on the decode GEMM (DecoderModel.PGEMM_MIN_TILES)
        self.min_tiles = 96
        if self.packs(w, self.N, self.K):
            self.packed = K.pack_dgemm_weight(self.w, swiglu=swiglu, m=decode_rows)
            self.w = None

    @staticmethod
    def packs(w: torch.Tensor, N: int, K: int) -> bool:
        """Whether an [N, K] matrix like ``w`` is packed for the hand-written products."""
        return (w.is_cuda and w.dtype == torch.bfloat16 and N % 64 == 0 and K % 64 == 0
                and os.environ.get("CFC_DECODE_PACKED", "auto") != "0")

    def rowmajor(self) -> torch.Tensor:
        return self.w if self.w is not None else K._rowmajor(self.packed)

    def nbytes(self) -> int:
        return self.packed.nbytes() if self.packed is not None else self.w.numel() * self.w.element_size()

    @classmethod
    def of_packed(cls, packed: "K.PackedWeight"):
        """A projection over (a run of tiles of) a packed matrix."""
        p = cls.__new__(cls)
        p.N, p.K, p.w, p.packed, p.min_tiles = packed.N, packed.K, None, packed, 96
        return p

    def _prefill(self, M: int) -> bool:
        return M >= 256 and -(-M // 256) * -(-self.N // 256) >= self.min_tiles and M * self.K * 2 < 2 ** 32

    def _kernel(self, x, kind: str = "act") -> str:
        if self.packed is None or not x.is_contiguous():
            return "lib"
        if K.prompt_plan(x.shape[0], self.N, self.K, kind):
            return "mgemm"
        if kind != "whole" and 1 <= x.shape[0] <= K.GEMV_MAX_M \
                and K.dgemm_slab_plan(x.shape[0], self.N, self.K, self.packed.bn)[0] > NARROW_SLABS:
            return "gemv"
        return "pgemm" if self._prefill(x.shape[0]) else "dgemm"

    def _prompt(self, x, epi: str, kind: str = "act", **kw):
        return K.prompt_gemm(x, self.packed, epi, K.prompt_plan(x.shape[0], self.N, self.K, kind), **kw)

    def act(self, x: torch.Tensor) -> torch.Tensor:
        """[M, N] in x's dtype."""
        k = self._kernel(x)
        if k == "lib":
            return F.linear(x, self.rowmajor())
        if k == "mgemm":
            return self._prompt(x, "bf16", reduce=K.splitk_reduce)
        if k == "pgemm":
            return K.pgemm(x, self.packed, "bf16", variant="ppp")
        if k == "gemv":
            return K.splitk_reduce(K.gemv_part(x, self.packed))
        return K.dgemm_linear(x, self.packed)

    def few_slabs(self, x: torch.Tensor) -> torch.Tensor | None:
        """The slabs that :meth:`act` would sum for a decode step's rows (None: it sums none), to be consumed before the next product."""
        k = self._kernel(x)
        if k == "gemv":
            return K.gemv_part(x, self.packed)
        if k == "dgemm" and x.is_cuda and K.dgemm_config(x.shape[0], self.N, self.K, bn=self.packed.bn)[1] > 1:
            return K.dgemm_slabs(x, self.packed)
        return None

    def slabs(self, x: torch.Tensor, own: bool = False) -> torch.Tensor:
        """fp32 k-slice slabs [split, M, N] whose sum is the product (unrounded).  They may live in the
        stream's split-K workspace: consume them before the next product, unless they are to be a tensor of
        their ``own``."""
        k = self._kernel(x, "slabs")
        M, out = x.shape[0], None
        if k in ("gemv", "dgemm", "mgemm"):
            split = K.gemv_packed_config(self.N, self.K, self.packed.bn // 16, M)[0] if k == "gemv" else \
                K.dgemm_slab_plan(M, self.N, self.K, self.packed.bn)[0] if k == "dgemm" else \
                K.prompt_plan(M, self.N, self.K, "slabs")[2]
            if own:
                out = torch.empty(split, M, self.N, dtype=torch.float32, device=x.device)
        if k == "mgemm":
            return self._prompt(x, "f32", "slabs", out=out)
        if k == "pgemm":
            return K.pgemm(x, self.packed, "f32", variant="ppp")[None]
        if k == "gemv":
            return K.gemv_part(x, self.packed, out=out)
        if k == "dgemm":
            return K.dgemm_slabs(x, self.packed, out)
        w = self.rowmajor()
        if x.is_cuda and x.dtype == torch.bfloat16:
            return torch.mm(x, w.t(), out_dtype=torch.float32)[None]
        return F.linear(x.float(), w.float())[None]

    def glu(self, x: torch.Tensor, out: torch.Tensor, limit: float, alpha: float, beta: float, cubic: float = 0.0) -> torch.Tensor:
        """W = 8-row interleaved gate / up rows: the clamped GLU of the product into ``out`` [M, N / 2]
        (row-strided), in the product's epilogue where one pass over (packed) W fills the chip."""
        k, M = self._kernel(x), x.shape[0]
        # pgemm's part of it stores 16 bytes
        if k == "mgemm" and (out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0 or out.stride(0) % 4 == 0
                             and out.data_ptr() % 8 == 0 and not K.prompt_plan(M, self.N, self.K)[0]):
            return self._prompt(x, "glu", out=out, glu=(limit, alpha, beta, cubic), reduce=lambda slabs, rows: clamped_glu(
                slabs, rows, limit, alpha, beta, interleaved=True, cubic=cubic))
        if k == "pgemm" and self.K >= 128 and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0:
            return K.pgemm_glu(x, self.packed, out, limit, alpha, beta, cubic)
        if k in ("pgemm", "dgemm") and self.N // self.packed.bn * -(-M // 256) > K.DGEMM_CUS // 2 \
                and out.stride(0) % 4 == 0 and out.data_ptr() % 8 == 0:
            return K.dgemm_glu(x, self.packed, out, limit, alpha, beta, cubic)
        return clamped_glu(self.slabs(x), out, limit, alpha, beta, interleaved=True, cubic=cubic)

    def relu_sq(self, x: torch.Tensor) -> torch.Tensor:
        """relu(product)^2 [M, N] in x's dtype, in the prompt product's epilogue, else with the sum of the slabs."""
        k = self._kernel(x)
        if k == "mgemm":
            return self._prompt(x, "relu2", reduce=lambda slabs, rows: relu_sq(slabs, x.dtype, rows))
        if k == "pgemm" and self.K >= 128:
            return K.pgemm(x, self.packed, "relu2", variant="ppp")
        return relu_sq(self.slabs(x), x.dtype)

    def f32(self, x: torch.Tensor) -> torch.Tensor:
        """[M, N] fp32, a tensor of its own."""
        k = self._kernel(x, "whole")
        if k in ("mgemm", "dgemm"):
            out = torch.empty(1, x.shape[0], self.N, dtype=torch.float32, device=x.device)
            if k == "mgemm":
                return self._prompt(x, "f32", "whole", out=out)[0]
            return K.dgemm(x, self.packed, "part", 1, part=out)[0]
        if k == "pgemm":
            return K.pgemm(x, self.packed, "f32", variant="ppp")
        return self.slabs(x)[0]


class JointProjection:
    """Several matrices of one width read by one layer, each multiplying one of a few inputs [inputs, T, K]: one
    packed matrix (every part padded with zero rows to whole tiles).  A decode step runs them all in one launch, and so
    does a prompt of up to 128 rows; more rows take runs of parts in one launch where that is faster."""

    def __init__(self, parts: list[tuple[torch.Tensor, int]]):
        """parts: (W [N, K], index of its input)."""
        self.sizes = [w.shape[0] for w, _ in parts]
        self.inputs = [i for _, i in parts]
        self.K = parts[0][0].shape[1]
        w0 = parts[0][0]
        self.packed, self.runs = None, {}
        pad, bn = (lambda n: n), 64
        if Projection.packs(w0, 64, self.K):
            total = {b: sum(-(-n // b) * b for n in self.sizes) for b in (64, 128)}
            bn = 128 if total[128] <= 1.03 * total[64] else 64
            pad = (lambda n: -(-n // bn) * bn)
        self.offsets, at = [], 0
        for n in self.sizes:
            self.offsets.append(at)
            at += pad(n)
        self.N = at
        if not Projection.packs(w0, 64, self.K):
            self.parts = [Projection(w) for w, _ in parts]
            return
        full = w0.new_zeros(at, self.K)
        for (w, _), o in zip(parts, self.offsets):
            full[o:o + w.shape[0]] = w
        self.packed = K.pack_dgemm_weight(full, bn=bn)
        ends = self.offsets[1:] + [at]
        self.parts = [Projection.of_packed(K.PackedWeight(self.packed.data[o * self.K:e * self.K], e - o, self.K, bn))
                      for o, e in zip(self.offsets, ends)]
        self.in_of = torch.tensor([i for i, o, e in zip(self.inputs, self.offsets, ends) for _ in range((e - o) // bn)],
                                  dtype=torch.int32, device=w0.device)

    def nbytes(self) -> int:
        return self.packed.nbytes() if self.packed is not None else sum(p.nbytes() for p in self.parts)

    def act(self, j: int, acts: torch.Tensor) -> Cols:
        """Part j's columns as activations."""
        return Cols(self.parts[j].act(acts[self.inputs[j]]), 0, self.sizes[j])

    def slabs(self, j: int, acts: torch.Tensor) -> Cols:
        """Part j's columns in fp32 (a tensor of its own)."""
        return Cols(self.parts[j].slabs(acts[self.inputs[j]], own=True), 0, self.sizes[j])

    def prompt(self, acts: torch.Tensor, slabs: tuple[int, ...] = ()) -> list[Cols]:
        """Every part's columns of a prompt's rows, as activations, or (the parts named in ``slabs``) in fp32.

        Up to 128 rows, where a product is a stream of W: one product and one sum of its slabs, in place of a product and
        a sum for every part.  More rows: runs of parts side by side as one product, whose tiles fill rounds of the chip that
        each part's alone leave part empty (joint_plan).  us, apart -> in one: five inputs' products of 4096 x 4096 134 ->
        40 (130 rows), 158 -> 133 (862); 22528 columns in three parts of one input 106 -> 73 (420), 365 -> 334 (2569)."""
        M, n = acts.shape[1], len(self.sizes)
        if self.packed is None or not acts.is_contiguous() or n == 1:
            return [self.slabs(j, acts) if j in slabs else self.act(j, acts) for j in range(n)]
        if M <= 128:
            c = self.joint(acts)
            y = K.splitk_reduce(c[0].t)
            return [c[j] if j in slabs else Cols(y, self.offsets[j], self.sizes[j]) for j in range(n)]
        out: list = [None] * n
        for first, last, run, in_of in self._runs(slabs):
            at = self.offsets[first]
            widths = tuple(self.parts[j].N for j in range(first, last))
            plan = K.joint_plan(M, widths, self.K, in_of is None) if last - first > 1 else 0
            if plan:
                y = run.act(acts[self.inputs[first]]) if in_of is None else K.mgemm_joint(acts, run.packed, in_of, plan)
                out[first:last] = [Cols(y, self.offsets[j] - at, self.sizes[j]) for j in range(first, last)]
        return [c if c is not None else self.slabs(j, acts) if j in slabs else self.act(j, acts) for j, c in enumerate(out)]

    def _runs(self, slabs: tuple[int, ...]) -> list[tuple]:
        """(first part, one past the last, their columns as one projection, input per 128 of them or None: all the same) of
        the runs of neighbours that leave activations."""
        if slabs not in self.runs:
            ends, runs, j = self.offsets[1:] + [self.N], [], 0
            while j < len(self.sizes):
                first = j
                while j < len(self.sizes) and j not in slabs:
                    j += 1
                one = len(set(self.inputs[first:j])) == 1
                if j - first > 1 and (one or self.packed.bn == 128):
                    o, e, bn = self.offsets[first], ends[j - 1], self.packed.bn
                    run = Projection.of_packed(K.PackedWeight(self.packed.data[o * self.K:e * self.K], e - o, self.K, bn))
                    runs.append((first, j, run, None if one else self.in_of[o // bn:e // bn].contiguous()))
                j = max(j, first + 1)
            self.runs[slabs] = runs
        return self.runs[slabs]

    def joint(self, acts: torch.Tensor) -> list[Cols]:
        """Every part's columns in fp32, of one product (a tensor of its own)."""
        M = acts.shape[1]
        if self.packed is None or not acts.is_contiguous():
            x = [F.linear(acts[i].float(), p.rowmajor().float()) for p, i in zip(self.parts, self.inputs)]
            out = torch.cat(x, 1)[None]            # no padding: the parts lie side by side
        else:
            split = K.dgemm_slab_plan(M, self.N, self.K, self.packed.bn)[0]
            out = torch.empty(split, M, self.N, dtype=torch.float32, device=acts.device)
            K.dgemm_slabs(acts, self.packed, out, self.in_of)
        return [Cols(out, o, n) for o, n in zip(self.offsets, self.sizes)]
