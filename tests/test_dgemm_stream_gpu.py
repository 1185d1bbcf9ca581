"""The decode GEMM as one run of stages over all tiles (dgemm.hip, dgemm_stream_kernel) against 64-bit products."""
import pytest
import torch

from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops._native import kernels_available


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
def test_plan_streams_where_no_split_makes_whole_rounds():
    assert K.dgemm_slab_plan(5, 22528, 4096, 128) == (3, True) and K.dgemm_slab_plan(24, 18432, 4096, 128)[1]
    for M, N, Kd, bn in ((5, 4096, 14336, 128), (5, 4096, 4096, 64), (64, 28672, 4096, 112), (65, 22528, 4096, 128), (300, 18432, 4096, 128)):
        assert K.dgemm_slab_plan(M, N, Kd, bn) == (K.dgemm_config(M, N, Kd, bn=bn)[1], False)


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
@pytest.mark.parametrize("M", (5, 8, 16, 33, 64))
def test_one_slice_that_fills_the_round_is_no_stream(M):
    assert K.dgemm_config(M, 28672, 4096, bn=128)[1] == 1 and K.dgemm_slab_plan(M, 28672, 4096, 128) == (1, False)


@pytest.mark.gpu
@pytest.mark.parametrize("M", (1, 5, 16, 17, 63, 64))
@pytest.mark.parametrize("N, Kd, bn", [(64, 64, 64), (128, 192, 128), (640, 320, 128), (16384, 64, 64), (38400, 64, 64),
                                       (1920, 2176, 64), (4992, 1088, 128), (22528, 512, 128)])
def test_slabs_match_the_exact_product(monkeypatch, M, N, Kd, bn):
    """One stage in all, one per workgroup, several tiles per workgroup, several workgroups per tile; every slab written."""
    g = torch.Generator("cuda").manual_seed(M + N)
    x = torch.randn(3, M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * 0.1).bfloat16()
    pk = K.pack_dgemm_weight(w, bn=bn)
    nks, U = Kd // 64, N // bn * (Kd // 64)
    G = min(256, U)
    owner = [next(i for i in range(v * G // U, G) if i * U // G <= v < (i + 1) * U // G) for v in range(U)]
    slabs = max(owner[t * nks + nks - 1] - owner[t * nks] + 1 for t in range(N // bn))
    monkeypatch.setattr(K, "dgemm_slab_plan", lambda *a: (slabs, True))
    in_of = torch.randint(0, 3, (N // bn,), device="cuda", dtype=torch.int32, generator=g)
    for inputs in (None, in_of):
        out = torch.full((slabs, M, N), float("nan"), device="cuda")
        K.dgemm_slabs(x[0] if inputs is None else x, pk, out, inputs)
        rows = x[torch.zeros_like(in_of) if inputs is None else in_of].double()        # [tiles, M, K]
        tiles = w.view(N // bn, bn, Kd).double().transpose(1, 2).contiguous()
        want = torch.bmm(rows, tiles).permute(1, 0, 2).reshape(M, N)
        # sums of K products in fp32, in any order
        tol = Kd * 2.0 ** -24 * torch.bmm(rows.abs(), tiles.abs()).permute(1, 0, 2).reshape(M, N)
        assert ((out.double().sum(0) - want).abs() <= tol + 1e-30).all()


@pytest.mark.gpu
def test_what_does_not_fit_is_refused(monkeypatch):
    pk = K.pack_dgemm_weight(torch.zeros(256, 128, device="cuda", dtype=torch.bfloat16), bn=128)
    x = torch.zeros(5, 128, device="cuda", dtype=torch.bfloat16)
    monkeypatch.setattr(K, "dgemm_slab_plan", lambda *a: (1, True))
    with pytest.raises(ValueError):
        K.dgemm_slabs(x[:, ::2], pk)
    with pytest.raises(ValueError):
        K.dgemm_slabs(x.float(), pk)
    with pytest.raises(ValueError):
        K.dgemm_slabs(x, pk, torch.empty(2, 5, 256, device="cuda"))
    with pytest.raises(ValueError):
        K.dgemm_slabs(x[None], pk, None, torch.zeros(3, device="cuda", dtype=torch.int32))
    with pytest.raises(RuntimeError):
        K.dgemm_slabs(torch.zeros(65, 128, device="cuda", dtype=torch.bfloat16), pk)
