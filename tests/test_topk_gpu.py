"""Exact top-k (knn.hip topk_select_kernel) where it can go wrong: block and chunk edges, ties, orders that defeat the
bound, masked rows; against torch's stable sort, whose values and indices it gives exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _scores(kind, nq, n):
    g = torch.Generator(device=DEV).manual_seed(n + nq)
    s = torch.randn(nq, n, device=DEV, generator=g)
    if kind == "ties":
        return (s * 3).round() + 0.0      # no negative zeros: they sort below zero here
    if kind == "equal":
        return torch.zeros_like(s) - 1.5
    if kind == "rising":
        return s.sort(1).values
    if kind == "runs":          # the best scores side by side in few blocks
        return s.sort(1, descending=True).values.roll(n // 3, 1)
    if kind == "masked":
        return s.masked_fill(torch.rand(nq, n, device=DEV, generator=g) < 0.97, float("-inf"))
    return s


@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "rising", "runs", "masked"])
@pytest.mark.parametrize("nq,n,k", [(1, 1, 1), (3, 15, 15), (2, 17, 5), (1, 4095, 150), (2, 4097, 2048), (1, 16 * 16384, 150),
                                    (2, 16 * 16384 + 1, 257), (1, 1_500_003, 2048), (20, 30_001, 10)])
def test_topk_is_the_stable_sort(kind, nq, n, k):
    from copilot_for_consensus_amd.ops import kernels as K
    s = _scores(kind, nq, n)
    v, i = K.topk(s, k)
    rv, ri = s.sort(dim=1, descending=True, stable=True)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])
    ids = torch.randint(0, 1 << 40, (nq, n), device=DEV)
    assert torch.equal(K.topk(s, k, ids)[1], ids.gather(1, ri[:, :k]))


@pytest.mark.parametrize("dim,nq,N,lo", [(128, 1, 1, 0), (384, 16, 33, 1), (768, 5, 5003, 2), (384, 3, 70_001, 40_000), (1024, 2, 4100, 3)])
def test_knn_topk_in_spans(monkeypatch, dim, nq, N, lo):
    """A search in one span and in many gives the same rows, in the order of the scores that knn_scores gives."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, nq))
    alive = torch.rand(N, device=DEV, generator=g) > 0.2
    k = min(100, N - lo)
    one = K.knn_topk(X, Q, k, alive=alive, row_lo=lo, N=N)
    want = K.knn_scores(X, Q)[:, lo:].masked_fill(~alive[lo:][None], float("-inf"))
    rv, ri = want.sort(dim=1, descending=True, stable=True)
    assert torch.equal(one[0], rv[:, :k]) and torch.equal(one[1], ri[:, :k] + lo)
    monkeypatch.setattr(K, "KNN_SCORES", nq * max(1, (N - lo) // 5))
    many = K.knn_topk(X, Q, k, alive=alive, row_lo=lo, N=N)
    assert torch.equal(one[0], many[0]) and torch.equal(one[1], many[1])


def test_a_last_span_of_more_blocks(monkeypatch):
    """Spans of 270000 rows, 8438 blocks of 32, and a last one of 262000, 16375 blocks of 16."""
    from copilot_for_consensus_amd.ops import kernels as K
    nq, dim, N, k = 3, 128, 532_000, 100
    g = torch.Generator(device=DEV).manual_seed(N)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, nq))
    rv, ri = K.knn_scores(X, Q).sort(dim=1, descending=True, stable=True)
    monkeypatch.setattr(K, "KNN_SCORES", nq * 270_000)
    v, i = K.knn_topk(X, Q, k)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])
