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
    """A search that may store all its scores and one that may store a fifth of them give the same rows, in the order of the
    scores that knn_scores gives."""
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


@pytest.mark.parametrize("metric", ["dot", "l2"])
@pytest.mark.parametrize("dim,nq,N,lo", [(128, 1, 1, 0), (384, 16, 33, 1), (768, 5, 5003, 2), (384, 3, 70_001, 40_000), (1024, 2, 4100, 3),
                                         (256, 1, 300, 17), (512, 7, 16 * 64, 0), (128, 3, 1_100_000, 8)])
def test_knn_topk_stored_and_by_blocks(monkeypatch, dim, nq, N, lo, metric):
    """A search that stores all scores and one that stores block maxima give the same rows, in the order of the scores that
    knn_scores gives; fewer blocks than winners, a last block of one row, maxima in two shares; rows that score alike."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, nq))
    X[N // 2:N // 2 + 9] = X[N // 3]
    alive = torch.rand(N, device=DEV, generator=g) > 0.2
    xn, qn = (t.float().pow(2).sum(1) if metric == "l2" else None for t in (X, Q))
    k = min(100, N - lo)
    want = K.knn_scores(X, Q, xn, qn)[:, lo:].masked_fill(~alive[lo:][None], float("-inf"))
    rv, ri = want.sort(dim=1, descending=True, stable=True)
    for most in (1 << 21, 0):
        monkeypatch.setattr(K, "KNN_SCORES", most)
        v, i = K.knn_topk(X, Q, k, xn, qn, alive=alive, row_lo=lo, N=N)
        assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k] + lo), most


@pytest.mark.parametrize("kind", ["equal", "few", "rising"])
def test_search_by_blocks_of_alike_rows(monkeypatch, kind):
    """Block maxima that are all equal, all but a few masked, and rising with the row."""
    from copilot_for_consensus_amd.ops import kernels as K
    N, k = 50_021, 150
    g = torch.Generator(device=DEV).manual_seed(1)
    X, Q = (torch.randn(n, 128, device=DEV, generator=g).bfloat16() for n in (N, 2))
    alive = None
    if kind == "equal":
        X[:] = X[:1]
    elif kind == "few":
        alive = torch.rand(N, device=DEV, generator=g) < 0.001
    else:
        X[:, 1:] = 0.0
        X[:, 0] = torch.arange(N, device=DEV) / 1000.0
        Q[:, 0] = 1.0
    want = K.knn_scores(X, Q)
    if alive is not None:
        want = want.masked_fill(~alive[None], float("-inf"))
    rv, ri = want.sort(dim=1, descending=True, stable=True)
    monkeypatch.setattr(K, "KNN_SCORES", 0)
    v, i = K.knn_topk(X, Q, k, alive=alive)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])


def test_one_row_and_results_of_other_strides():
    """A transposed column; results given flat, 4 bytes off 16, in wider rows."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(7)
    s = torch.randn(5003, 1, device=DEV, generator=g)
    v, i = K.topk(s.t(), 40)
    rv, ri = s.t().sort(dim=1, descending=True, stable=True)
    assert torch.equal(v, rv[:, :40]) and torch.equal(i, ri[:, :40])
    for nq, N in ((3, 1000), (1, 1001)):
        X, Q = (torch.randn(n, 128, device=DEV, generator=g).bfloat16() for n in (N, nq))
        want = K.knn_scores(X, Q)
        flat = torch.full((nq * N + 2,), 7.0, device=DEV)
        wide = torch.full((nq, N + 5), 7.0, device=DEV)
        K.knn_scores(X, Q, out=flat[1:-1])
        K.knn_scores(X, Q, out=wide[:, 3:N + 3])
        assert torch.equal(flat[1:-1].view(nq, N), want) and flat[0] == flat[-1] == 7.0
        assert torch.equal(wide[:, 3:N + 3], want) and (wide[:, :3] == 7.0).all() and (wide[:, N + 3:] == 7.0).all()
        if nq == 1:
            assert torch.equal(K.knn_scores(X, Q, out=torch.empty(N, 1, device=DEV).t()), want)


@pytest.mark.parametrize("n,k", [(16 * 16384 + 5, 100), (1_500_003, 300), (1_048_576, 2048)])
@pytest.mark.parametrize("kind", ["few", "plateau", "levels"])
def test_more_blocks_at_the_bound_than_winners(kind, n, k):
    """Of blocks whose best score is the bound, only the first can hold winners: all but a few rows masked; one value above
    a noisy floor, in every block and in late blocks more often; a few values everywhere."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(k)
    s = torch.randn(2, n, device=DEV, generator=g)
    r = torch.rand(2, n, device=DEV, generator=g)
    if kind == "few":
        s = s.masked_fill(r > 0.5 * k / n, float("-inf"))
    elif kind == "plateau":
        s = torch.where(r < 0.01 + torch.arange(n, device=DEV) / n, torch.full_like(s, 9.0), s)
        s[0, n - 7], s[1, 5] = 10.0, 11.0
    else:
        s = (r * 3).floor()
    v, i = K.topk(s, k)
    rv, ri = s.sort(dim=1, descending=True, stable=True)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])


def test_equal_scores_take_no_longer():
    """A million equal scores, as of an index whose rows are nearly all masked, within eight times the time of a million
    different ones (1.5 times where measured; 160 times where every block that reaches the bound is looked at)."""
    from copilot_for_consensus_amd.ops import kernels as K

    def us(s):
        ms = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                K.topk(s, 300)
            b.record()
            torch.cuda.synchronize()
            ms.append(a.elapsed_time(b))
        return sorted(ms)[3]
    s = torch.randn(1, 1_000_000, device=DEV)
    assert us(torch.full_like(s, float("-inf"))) < 8 * us(s)


@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "rising", "masked"])
@pytest.mark.parametrize("nq,n,k", [(2, 1 << 20, 5), (3, (1 << 20) + 1, 150), (1, (1 << 21) + 63, 2048), (2, 5_000_011, 257)])
def test_segments_of_scores(kind, nq, n, k):
    """One workgroup's most scores, and shares of two to five, the last one shorter; the winners' order among equals."""
    from copilot_for_consensus_amd.ops import kernels as K
    s = _scores(kind, nq, n)
    rv, ri = s.sort(dim=1, descending=True, stable=True)
    v, i = K.topk(s, k)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])
    ids = torch.randint(0, 1 << 40, (nq, n), device=DEV)
    assert torch.equal(K.topk(s, k, ids)[1], ids.gather(1, ri[:, :k]))


@pytest.mark.parametrize("n", [16 * 1023, 16 * 1024, 16 * 1025 + 1, 16 * 16384])
@pytest.mark.parametrize("k", [1, 150, 255, 256, 257])
@pytest.mark.parametrize("kind", ["normal", "stacked", "ties"])
def test_bound_from_the_threads_best(kind, k, n):
    """Selections that look at 1024 threads' best blocks first, and the next larger k and next fewer blocks, which do not.
    stacked: the best blocks belong to few threads (block b is thread b % 1024's), so that bound lets too many pass."""
    from copilot_for_consensus_amd.ops import kernels as K
    s = _scores("ties" if kind == "ties" else "normal", 2, n)
    if kind == "stacked":
        b = torch.arange(n, device=DEV) // 16 % 1024
        s = s + 100.0 * ((b < 40) | (b == 1023))
    rv, ri = s.sort(dim=1, descending=True, stable=True)
    v, i = K.topk(s, k)
    assert torch.equal(v, rv[:, :k]) and torch.equal(i, ri[:, :k])


@pytest.mark.parametrize("dim,nq,N", [(384, 3, 32_767), (384, 16, 32_769), (384, 2, 65_601), (512, 1, 163_840), (512, 1, 163_841),
                                      (128, 5, 655_347), (768, 2, 70_001)])
def test_scan_by_workgroups_of_one_round(dim, nq, N):
    """Sizes about 512 workgroups' first round and about the bytes up to which they take all blocks; rows wider than that."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, nq))
    want = K.knn_scores(X, Q, None, None)
    rv, ri = want.sort(dim=1, descending=True, stable=True)
    v, i = K.knn_topk(X, Q, 100, N=N)
    assert torch.equal(v, rv[:, :100]) and torch.equal(i, ri[:, :100])


@pytest.mark.parametrize("metric", ["cosine", "dot", "l2"])
@pytest.mark.parametrize("dim,nq", [(128, 1), (384, 16), (768, 2), (1024, 5)])
def test_float_queries_in_one_launch(metric, dim, nq):
    """Queries of floats beside the index, rounded and normalized by one launch, against those of other strides and alignments
    and of 16 bits, which are rounded before: the same bf16 values, so the same cosine and dot scores; of l2 the query's norm
    is summed in another order, dim products and sums of 2^-24 each."""
    from copilot_for_consensus_amd.ops import kernels as K
    from copilot_for_consensus_amd.vectorstore import HipFlatIndex
    g = torch.Generator().manual_seed(dim)
    index = HipFlatIndex(dim, distance=metric, device=DEV)
    index.add_embeddings([str(j) for j in range(700)], torch.randn(700, dim, generator=g))
    flat = torch.zeros(nq * dim + 1, device=DEV)
    q = torch.randn(nq, dim, generator=g) * torch.logspace(-20, 15, nq * dim).view(nq, dim)[:, torch.randperm(dim, generator=g)]
    q[0] = torch.randn(dim, generator=g)
    if nq > 2:
        q[1], q[2] = 0.0, torch.linspace(-1, 1, dim) * 2.0 ** -130
    q = q.to(DEV)
    flat[1:] = q.flatten()
    wide = torch.zeros(nq, dim + 8, device=DEV)
    wide[:, :dim] = q
    unit = K.l2_normalize(q.bfloat16()) if metric == "cosine" else q.bfloat16()
    got, n2 = K.knn_queries(q, metric == "cosine")
    assert torch.equal(got, unit)
    torch.testing.assert_close(n2, q.bfloat16().double().pow(2).sum(1).float(), rtol=dim * 2.0 ** -24, atol=2.0 ** -126)
    v, i = index.search(q, 20)
    for other in (flat[1:].view(nq, dim), wide[:, :dim], q.bfloat16()):
        ov, oi = index.search(other, 20)
        if metric == "l2":
            torch.testing.assert_close(v, ov, rtol=(dim + 4) * 2.0 ** -24, atol=0.0)
        else:
            assert torch.equal(v, ov) and torch.equal(i, oi)


@pytest.mark.parametrize("metric", ["dot", "l2"])
@pytest.mark.parametrize("dim,nq,N", [(768, 1, 1), (768, 3, 15), (1024, 16, 17), (768, 2, 63), (1024, 1, 65), (768, 5, 16 * 4 * 256 + 1), (1024, 2, 40_003),
                                      (384, 2, 393_300), (512, 1, 295_001), (256, 3, 600_007)])
def test_knn_scores_by_the_stream(dim, nq, N, metric):
    """Rows that come through LDS: fewer than a unit's sixteen, one more than whole blocks, rows of one and two units, more
    rows than the chip caches; infinite and masked rows spoil no other, and nothing is written past the last row."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N + dim)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, nq))
    bad = torch.arange(0, N, 1001, device=DEV)[1:]
    X[bad] = float("inf")
    alive = torch.rand(N, device=DEV, generator=g) > 0.1
    xn, qn = (t.float().pow(2).sum(1) if metric == "l2" else None for t in (X, Q))
    out = torch.full((nq, N + 3), 7.0, device=DEV)
    got = K.knn_scores(X, Q, xn, qn, out=out[:, :N])
    assert bool((out[:, N:] == 7.0).all())
    fine = torch.ones(N, dtype=torch.bool, device=DEV).index_fill_(0, bad, False)
    for at in range(0, N, 100_000):
        x = X[at:at + 100_000].double()
        want = Q.double() @ x.T
        if metric == "l2":
            want = 2 * want - qn.double()[:, None] - xn.double()[None, at:at + 100_000]
        ok = fine[at:at + 100_000]
        # fp32 sums of `dim` products (and three terms) of about 1 each, the largest sum some dim
        assert float((got[:, at:at + 100_000].double() - want)[:, ok].abs().max()) < 2.0 ** -22 * dim * 4
    assert not bool(got[:, bad].isfinite().any())
    v, i = K.knn_topk(X, Q, min(50, N), xn, qn, alive=alive & fine)
    rv, ri = got.masked_fill(~(alive & fine)[None], float("-inf")).sort(dim=1, descending=True, stable=True)
    assert torch.equal(v, rv[:, :min(50, N)]) and torch.equal(i, ri[:, :min(50, N)])


@pytest.mark.parametrize("lo,n", [(0, 1), (3, 15), (0, 16), (5, 17), (0, 262144), (1, 262145), (0, 1 << 20), (0, (1 << 20) + 1)])
@pytest.mark.parametrize("nq,k,unit,dead", [(1, 5, True, False), (3, 256, False, False), (16, 20, True, True), (7, 1, False, True)])
def test_a_search_by_one_call(lo, n, nq, k, unit, dead):
    """The same values and rows as from queries, scores and selection one after the other, bit for bit."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device="cuda").manual_seed(n + nq)
    X = torch.randn(lo + n + 2, 128, device="cuda", generator=g).bfloat16()
    q = torch.randn(nq, 128, device="cuda", generator=g)
    norms = None if unit else X.float().pow(2).sum(1)
    alive = torch.rand(len(X), device="cuda", generator=g) < 0.9 if dead else None
    Q, n2 = K.knn_queries(q, unit)
    want = K.knn_topk(X, Q, k, norms, n2, alive, lo, lo + n)
    got = K.knn_search(X, q, k, unit, norms, alive, lo, lo + n)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    for bad in (dict(k=0), dict(k=257), dict(row_lo=-1), dict(N=len(X) + 1)):
        with pytest.raises(ValueError):
            K.knn_search(X, q, **{"k": k, "unit": unit, "row_lo": lo, "N": lo + n, **bad})


@pytest.mark.parametrize("dim,n", [(128, 17), (256, 40_001), (256, 600_000), (384, 20_000), (384, 250_000), (384, 400_001), (512, 300_000), (768, 5_003),
                                   (1024, 1_000)])
@pytest.mark.parametrize("nq,unit,dead", [(1, True, False), (4, False, False), (5, True, True), (8, False, True), (9, True, False), (16, False, True)])
def test_float_queries_in_the_scan(dim, n, nq, unit, dead):
    """Queries that the scan's workgroups take to LDS themselves, by fragments and by rings, and those that are too many or whose
    workgroups are: the bits of a launch for the queries.  A query of zeros and one that is not finite among them."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device="cuda").manual_seed(n + nq)
    X = torch.randn(n, dim, device="cuda", generator=g).bfloat16()
    q = torch.randn(nq, dim, device="cuda", generator=g) * 3.0
    if nq > 4:
        q[1], q[4, dim - 1] = 0.0, float("inf")
    norms = None if unit else X.float().pow(2).sum(1)
    alive = torch.rand(n, device="cuda", generator=g) < 0.9 if dead else None
    Q, n2 = K.knn_queries(q, unit)
    k = min(150, n)
    want, got = K.knn_topk(X, Q, k, norms, n2, alive, 0, n), K.knn_search(X, q, k, unit, norms, alive, 0, n)
    assert torch.equal(got[0].view(torch.int32), want[0].view(torch.int32)) and torch.equal(got[1], want[1])
