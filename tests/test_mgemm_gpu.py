"""The prompt GEMM for a few hundred rows (mgemm.hip) against 64-bit products, and the rule that takes a product there."""
import pytest
import torch

from copilot_for_consensus_amd._build import KERNELS_LIB
from copilot_for_consensus_amd.models import registry
from copilot_for_consensus_amd.models.projection import Projection
from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops import reference as ref
from copilot_for_consensus_amd.ops._native import kernels_available


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
def test_plan_takes_what_lies_between_the_decode_gemm_and_pgemm():
    for N, Kd in ((6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (1024, 2048), (64, 64)):
        for kind in ("act", "slabs", "whole"):
            assert all(K.prompt_plan(M, N, Kd, kind) is None for M in (1, 5, 128))
            for M in range(129, 20000, 97):
                plan = K.prompt_plan(M, N, Kd, kind)
                if plan:
                    head, bm, split = plan
                    assert 0 <= head < M and head % 256 == 0
                    assert bm in (128, 160, 192, 224, 256) and split in (1, 2, 4, 8) and split * 64 <= Kd
                    assert split == 1 or kind == "act" or kind == "slabs" and head == 0
    assert K.prompt_plan(700, 4096, 4096)[0] == 0 and K.prompt_plan(4500, 4096, 14336)[0] == 4096
    assert K.prompt_plan(4096, 4096, 4096) is None and K.prompt_plan(16384, 28672, 4096) is None
    assert K.prompt_plan(2 ** 19, 64, 4096) is None         # 32-bit DMA offsets


def _data(M, N, Kd, seed, swiglu=False):
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * 0.1).bfloat16()
    return x, w, Projection(w, swiglu=swiglu).packed


def _f32_tol(x, w):
    """Sums of K products in fp32, in any order: K units in the last place of the sum of the magnitudes."""
    return x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


@pytest.mark.gpu
@pytest.mark.parametrize("bm", (128, 160, 192, 224, 256))
@pytest.mark.parametrize("M, N, Kd", [(1, 64, 64), (129, 192, 128), (255, 320, 192), (257, 384, 320), (449, 448, 576),
                                      (300, 1024, 2048)])
def test_slabs_match_the_exact_product(M, N, Kd, bm):
    """Odd rows, half column tiles, fewer stages than the ring has slots and more, uneven slices."""
    x, w, pk = _data(M, N, Kd, M + bm)
    want = x.double() @ w.double().t()
    for split in {1, min(2, Kd // 64), min(3, Kd // 64), min(8, Kd // 64)}:
        out = torch.full((split, M, N), float("nan"), device="cuda")
        K.mgemm(x, pk, "part", bm, split, out)
        assert ((out.double().sum(0) - want).abs() <= _f32_tol(x, w) + 1e-30).all(), (split,)


@pytest.mark.gpu
@pytest.mark.parametrize("bm, M, N, Kd", [(128, 130, 128, 64), (160, 161, 192, 256), (192, 400, 320, 448), (224, 223, 448, 128),
                                          (256, 513, 256, 1024)])
def test_epilogues_round_the_exact_product(bm, M, N, Kd):
    x, w, pk = _data(M, N, Kd, bm, swiglu=True)
    y = K.mgemm(x, pk, "part", bm, 1, torch.empty(1, M, N, device="cuda"))[0]     # the sums the epilogues see
    assert torch.equal(K.mgemm(x, pk, "bf16", bm), y.bfloat16())
    assert torch.equal(K.mgemm(x, pk, "relu2", bm), ref.relu_sq(y).bfloat16())
    g, u = (t.double() for t in y.view(M, N // 16, 2, 8).unbind(2))
    wide = torch.full((M, N // 2 + 24), 7.0, device="cuda", dtype=torch.bfloat16)
    K.mgemm(x, pk, "glu", bm, out=wide[:, 8:8 + N // 2], glu=(3.0, 1.702, 1.0, 0.0))
    want = (g.clamp(max=3.0) * torch.sigmoid(1.702 * g.clamp(max=3.0)) * (u.clamp(-3.0, 3.0) + 1.0)).reshape(M, N // 2)
    got = wide[:, 8:8 + N // 2].double()
    # one rounding to bf16 and, before it, a few of fp32 (1e-5 of the value covers the exponential's)
    assert ((got - want).abs() <= want.abs() * (2.0 ** -8 + 1e-5) + 1e-6).all()
    assert (wide[:, :8] == 7.0).all() and (wide[:, 8 + N // 2:] == 7.0).all()
    g, u = (t.bfloat16().double() for t in y.view(M, N // 16, 2, 8).unbind(2))
    want = (g * torch.sigmoid(g) * u).reshape(M, N // 2)
    assert ((K.mgemm(x, pk, "swiglu", bm).double() - want).abs() <= want.abs() * (2.0 ** -8 + 1e-5) + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", (129, 256, 300, 700, 1500, 4100, 4500, 8400))
def test_projection_agrees_with_the_general_path(M, monkeypatch):
    """Every product of a Projection on mgemm and without it: the same sums to fp32, the same rounding."""
    N, Kd = 4096, 2176
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * 0.1).bfloat16()
    p, tol = Projection(w, swiglu=True), _f32_tol(x, w)

    def all_of():
        out = torch.empty(M, N // 2, device="cuda", dtype=torch.bfloat16)
        slabs = p.slabs(x).double().sum(0)
        own = p.slabs(x, own=True)
        p.act(x)                                       # another product: own slabs stay
        assert torch.equal(own.double().sum(0), slabs)
        rows = torch.full((M, N // 2 + 4), 3.0, device="cuda", dtype=torch.bfloat16)          # rows 8 bytes apart from 16
        glu = p.glu(x, out, 7.0, 1.702, 1.0).double()
        assert ((p.glu(x, rows[:, 4:], 7.0, 1.702, 1.0).double() - glu).abs() <= 2.0 ** -7 * glu.abs() + 80 * tol.max()).all()
        assert (rows[:, :4] == 3.0).all()
        return slabs, p.f32(x).double(), p.act(x).double(), p.relu_sq(x).double(), glu
    assert K.prompt_plan(M, N, Kd) and K.prompt_plan(M, N, Kd)[0] == M // 4096 * 4096
    new = all_of()
    monkeypatch.setattr(K, "prompt_plan", lambda *a: None)
    old = all_of()
    for a, b in zip(new[:2], old[:2]):
        assert ((a - b).abs() <= 2 * tol).all()
    for a, b, slope in zip(new[2:], old[2:], (1.0, 2 * old[0].abs().max(), 40.0)):
        # both round to bf16 once, of values that differ by the sums' error times the epilogue's slope at most
        assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 2 * slope * tol.max()).all()


@pytest.mark.gpu
def test_what_does_not_fit_is_refused():
    x, w, pk = _data(130, 128, 128, 1)
    for bm, split, epi in ((100, 1, "bf16"), (128, 3, "part"), (128, 0, "part"), (128, 2, "bf16")):
        with pytest.raises((RuntimeError, ValueError)):
            K.mgemm(x, pk, epi, bm, split)
    with pytest.raises(ValueError):
        K.mgemm(x[:, :64], pk, "bf16", 128)
    with pytest.raises(ValueError):
        K.mgemm(x, w, "bf16", 128)


@pytest.mark.gpu
@torch.inference_mode()
def test_captured_products_replay():
    x, w, pk = _data(700, 4096, 1024, 5)
    p = Projection(w)
    want = p.act(x)
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        p.act(x)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        y = p.act(x)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("preset", ("vofosun-7b", "zisapel-7b", "pemolorn-7b", "tadolix-7b"))
def test_libraries_of_one_family_hold_every_product(preset):
    """A library built of the sources that a family names has the entry points of every route of a projection."""
    cfg = registry.get_config(preset)
    names = registry.family_of(cfg).model.kernel_sources(cfg, torch.bfloat16)
    text = "".join((KERNELS_LIB.parents[2] / "csrc" / "kernels" / f"{n}.hip").read_text() for n in names)
    for entry in ("cfc_prompt_plan", "cfc_mgemm", "cfc_pgemm", "cfc_pgemm_glu", "cfc_dgemm", "cfc_dgemm_config", "cfc_dgemm_slab_plan",
                  "cfc_dgemm_stream", "cfc_dgemm_joint", "cfc_gemv_packed", "cfc_splitk_reduce", "cfc_clamped_glu"):
        assert entry + "(" in text, entry


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
def test_plan_goes_by_one_model():
    """A rule for one size made others worse: 14 000 rows of 4096 x 4096 in two launches (326 us, one 321); a few
    rows beyond a whole round of 28672 x 4096 are a launch of their own (513 rows 123 us against 133 of all on mgemm)."""
    assert K.prompt_plan(14_000, 4096, 4096, "whole") is None and K.prompt_plan(14_000, 4096, 4096) is None
    assert all(K.prompt_plan(M, 28672, 4096)[0] == 512 for M in (513, 533, 560, 640))
    assert K.prompt_plan(1344, 28672, 4096) is None           # (one launch of 224 rows a tile 242, with a tail 264)
