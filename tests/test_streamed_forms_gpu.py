"""What comes by LDS-DMA, in forms beside the usual.  Against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dim,N", [(768, 5000), (768, 177), (1024, 333), (384, 393_300)])
@pytest.mark.parametrize("lo", [0, 1, 2, 3, 35])
@pytest.mark.parametrize("form", ["l2", "mask", "both"])
def test_search(dim, N, lo, form):
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N + lo)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, 3))
    xn, qn = (t.float().pow(2).sum(1) if form in ("l2", "both") else None for t in (X, Q))
    alive = torch.rand(N, device=DEV, generator=g) > 0.3 if form in ("mask", "both") else None
    v, i = K.knn_topk(X, Q, 40, xn, qn, alive=alive, row_lo=lo, N=N - 1)
    want = Q.double() @ X[lo:N - 1].double().T
    if xn is not None:
        want = 2 * want - qn.double()[:, None] - xn.double()[None, lo:N - 1]
    if alive is not None:
        want = want.masked_fill(~alive[None, lo:N - 1], float("-inf"))
        assert bool(alive[i].all())
    # fp32 sums of `dim` products and three terms of some dim at most
    tol = 2.0 ** -22 * dim * 4
    assert float((v.double() - want.gather(1, i - lo)).abs().max()) < tol
    assert float((v.double() - want.topk(40).values).abs().max()) < tol
