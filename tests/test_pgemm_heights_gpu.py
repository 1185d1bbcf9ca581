"""Tiles of 192 and 224 rows of the persistent prompt GEMM: the same bits as in tiles of 256, at the edges of rows, columns and
K, over many tiles a workgroup, and with every epilogue."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operands(M, N, Kd, swiglu=False, seed=0):
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(seed + M + N + Kd)
    x = torch.randn(M, Kd, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, Kd, device=DEV, generator=g) * Kd ** -0.5).bfloat16()
    return x, w, K.pack_dgemm_weight(w, bn=64)


def _probe(x, w, epi, mt):
    from copilot_for_consensus_amd.ops._native import check, kernels
    M, cols = x.shape[0], w.N // 2 if epi == 3 else w.N
    out = torch.full((M + 1, cols), float("nan"), device=DEV, dtype=torch.bfloat16)
    check(kernels().cfc_pgemm_ppp_probe(x.data_ptr(), w.data.data_ptr(), out.data_ptr(), M, w.N, w.K, epi | (mt << 5), cols, w.bn // 16, 8,
                                        torch.cuda.current_stream().cuda_stream), "probe")
    assert bool(out[M].isnan().all())             # nothing past the last row
    return out[:M]


@pytest.mark.parametrize("mt", [6, 7])
@pytest.mark.parametrize("epi", [0, 3])
@pytest.mark.parametrize("M", [1, 95, 97, 191, 192, 193, 223, 224, 225, 335, 449])
@pytest.mark.parametrize("N,K", [(64, 128), (320, 192), (512, 320)])
def test_edges(mt, epi, M, N, K):
    x, w, p = _operands(M, N, K)
    got = _probe(x, p, epi, mt)
    assert torch.equal(got, _probe(x, p, epi, 8))
    if epi == 0:
        want = x.double() @ w.double().T
        # fp32 sums, rounded to bf16 once
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.parametrize("mt", [6, 7])
@pytest.mark.parametrize("M,N,K", [(224 * 150 + 37, 576, 128), (192 * 150 - 5, 1024, 192), (224 * 260, 256, 256)])
def test_many_tiles_a_workgroup(mt, M, N, K):
    """An even and an odd number of K-tiles, stores of a whole tile in flight across its end, tiles past the edges between."""
    x, _, p = _operands(M, N, K)
    assert torch.equal(_probe(x, p, 0, mt), _probe(x, p, 0, 8))


@pytest.mark.parametrize("M,height", [(257, 6), (384, 6), (385, 7), (448, 7)])
@pytest.mark.parametrize("epi", ["bf16", "swiglu", "f32", "relu2", "glu"])
def test_epilogues(M, height, epi):
    """The height goes by the rows: a row's result is what it is among 512."""
    from copilot_for_consensus_amd.ops import kernels as K
    from copilot_for_consensus_amd.ops._native import kernels
    N, Kd = 28672, 1024
    x, _, p = _operands(512, N, Kd)
    assert kernels().cfc_ppp_height(M, N, Kd) == height and kernels().cfc_ppp_height(512, N, Kd) == 8

    def run(x):
        if epi == "glu":
            return K.pgemm_glu(x, p, torch.empty(x.shape[0], N // 2, device=DEV, dtype=torch.bfloat16), 7.0, 1.7, 1.0)
        return K.pgemm(x, p, epi, variant="ppp")
    assert torch.equal(run(x[:M]), run(x)[:M])
