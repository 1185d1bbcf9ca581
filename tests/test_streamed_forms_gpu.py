"""What comes by LDS-DMA, in forms beside the usual; encoder scores at the end of the range.  Against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, want, scale):
    # bf16 weights and results (2^-9 each, of values that add up to `scale` at most); scores are fp32 sums
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -9 * scale).all()), float((got.double() - want).abs().max())


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


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("lens", [[40], [200, 31, 7]])
def test_encoder_scores_at_the_end_of_the_range(D, lens):
    """All of a row's scores -1.9 2^127, finite: weights of one each, and not of none."""
    from copilot_for_consensus_amd.ops import kernels as K
    H, T = 2, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(D)
    qkv = torch.zeros(T, 3, H, D, device=DEV)
    qkv[:, 0, :, 0] = 2.0 ** 63
    qkv[:, 1, :, 0] = -1.8984375 * 2.0 ** 64
    qkv[:, 2] = torch.randn(T, H, D, device=DEV, generator=g)
    qkv = qkv.bfloat16()
    cu = torch.tensor([0] + lens, dtype=torch.int32, device=DEV).cumsum(0).int()
    got = K.encoder_attention(qkv, cu, H, D, 0.6931471805599453, max(lens))
    at = 0
    for n in lens:
        v = qkv[at:at + n, 2].double()
        _close(got[at:at + n], v.mean(0).expand(n, H, D), float(v.abs().mean(0).max()))
        at += n
