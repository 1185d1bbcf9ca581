"""Kernels of one workgroup a row that ask for all they need at once: numbers of slabs about what is asked for ahead, row
widths about their vectors and workgroups, choices among equals."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("split", [1, 2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("F", [7, 512])
def test_slabs_are_added_in_order(split, F):
    from copilot_for_consensus_amd.ops import stream
    g = torch.Generator(device=DEV).manual_seed(split)
    x = torch.randn(split, 5, F, device=DEV, generator=g)
    y = torch.zeros(5, F, device=DEV)
    for s in x:
        y = y + s
    assert torch.equal(stream.relu_sq(x, torch.float32), y.clamp(min=0) * y.clamp(min=0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W", [1, 6, 7, 1020, 1024, 2052, 4096, 4100, 5001])
@pytest.mark.parametrize("place", [False, True])
def test_embedded_rows(W, dtype, place):
    from copilot_for_consensus_amd.ops import stream
    g = torch.Generator(device=DEV).manual_seed(W)
    table = torch.randn(11, W, device=DEV, generator=g).to(dtype)
    ids = torch.tensor([0, 10, 3, 99, -4], dtype=torch.int32, device=DEV)         # out of range: the nearest row
    pos = torch.tensor([0, 1, 77, 4095, 131071], dtype=torch.int32, device=DEV)
    turns = stream.sinusoid_turns(W, 10000.0, DEV)
    out = torch.empty(5, W, device=DEV)
    stream.embed_f32(table, ids, out, 1.5, *((pos, turns) if place else ()))
    want = 1.5 * table.double()[ids.long().clamp(0, 10)]
    if place:
        a = pos.double()[:, None] * turns * (2 * torch.pi)
        want = want + torch.stack([a.sin(), a.cos()], -1).flatten(1)[:, :W]
    # one rounding of the sum (2^-24), the angle's turn to fp32 (2 pi 2^-25 of a turn), a sine of 2 ulp
    assert bool(((out.double() - want).abs() <= 2.0 ** -24 * want.abs() + (6.3 * 2.0 ** -24 + 2.0 ** -23) * place).all())
    odd = torch.empty(11 * W + 1, dtype=dtype, device=DEV)[1:].view(11, W)          # no vector starts there
    again = torch.empty_like(out)
    stream.embed_f32(odd.copy_(table), ids, again, 1.5, *((pos, turns) if place else ()))
    assert torch.equal(again, out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,T,n,gap", [(5, 3, 1, 0), (4096, 300, 64, 0), (1020, 2, 1500, 3)])
def test_constant_columns_beside_embedded_rows(W, T, n, gap, dtype):
    from copilot_for_consensus_amd.ops import stream
    table = torch.randn(9, W, device=DEV).to(dtype)
    ids = torch.arange(T, dtype=torch.int32, device=DEV) % 9
    rows = torch.full((T, W + n + gap), 5.0, dtype=dtype, device=DEV)
    out = stream.embed_f32(table, ids, torch.empty(T, W, device=DEV), ones=rows[:, W:W + n])
    out = torch.empty(T, W, device=DEV) if out is None else out
    assert bool((rows[:, W] == 1).all()) and not rows[:, W + 1:W + n].any()
    assert bool((rows[:, :W] == 5).all()) and bool((rows[:, W + n:] == 5).all())
    with pytest.raises(ValueError):
        stream.embed_f32(table, ids, out, ones=rows[:-1, W:])


@pytest.mark.parametrize("dim,T", [(8, 1), (512, 7), (4096, 300), (4104, 5), (8200, 3), (24576, 2), (65536, 2)])
def test_norms_of_gathered_rows(dim, T):
    """The norm that begins a stream and that of its last rows: the bits of gathering, copying and norming one after the other."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(dim)
    table, x, res = (torch.randn(n, dim, device=DEV, generator=g).to(torch.bfloat16) for n in (13, T, T))
    w = torch.randn(dim, device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.randint(0, 13, (T,), device=DEV, generator=g, dtype=torch.int32)
    h, first = K.embed_rmsnorm(table, ids, w, 1e-5)
    assert torch.equal(first, table[ids.long()]) and torch.equal(h, K.rmsnorm(first, w, 1e-5))
    keep = x.clone(), res.clone()
    for rows in ([T - 1], list(range(T))[::-1], [0, T // 2, T // 2]):
        for dtype in (torch.int32, torch.int64):
            at = torch.tensor(rows, dtype=dtype, device=DEV)
            got = K.rmsnorm_rows(x, res, at, w, 1e-5)
            assert torch.equal(got, K.rmsnorm(x.index_select(0, at), w, 1e-5, residual=res.index_select(0, at)))
    assert torch.equal(x, keep[0]) and torch.equal(res, keep[1])
    with pytest.raises(RuntimeError):
        K.rmsnorm_rows(x, res, ids[:0], w, 1e-5)


@pytest.mark.parametrize("dim", [8, 4096, 8200])
def test_norms_of_rows_that_are_not_there(dim):
    """Nothing is read past the rows; a place beside the rows, or an index of no whole numbers, is refused."""
    from copilot_for_consensus_amd.ops import kernels as K
    x, res = (torch.randn(5, dim, device=DEV).to(torch.bfloat16) for _ in range(2))
    w = torch.ones(dim, device=DEV, dtype=torch.bfloat16)
    good = K.rmsnorm(x[4:].clone(), w, 1e-5, residual=res[4:].clone())
    for dtype, rows in ((torch.int32, [5, 4, -1, 2 ** 31 - 1, -2 ** 31]), (torch.int64, [5, 4, -1, 2 ** 32, -2 ** 40])):
        got = K.rmsnorm_rows(x, res, torch.tensor(rows, dtype=dtype, device=DEV), w, 1e-5)
        assert torch.equal(got[1:2], good) and bool(got[[0, 2, 3, 4]].isnan().all())
    for rows in (torch.tensor([0]), torch.tensor([0.0], device=DEV), torch.tensor([True], device=DEV), torch.tensor([[0]], device=DEV)):
        with pytest.raises(ValueError):
            K.rmsnorm_rows(x, res, rows, w, 1e-5)


@pytest.mark.parametrize("E,top", [(1, 1), (8, 8), (63, 2), (64, 6), (65, 8), (200, 5), (1024, 8)])
@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "few"])
def test_experts_chosen_among_equals(E, top, kind):
    """The largest scores, the lower expert first among equals; `few`: all but some are -inf, fewer than are chosen."""
    from copilot_for_consensus_amd.ops import moe
    from copilot_for_consensus_amd.ops.cols import Cols
    g = torch.Generator(device=DEV).manual_seed(E)
    x = torch.randn(1, 9, E, device=DEV, generator=g)
    c = torch.zeros(E, device=DEV)
    if kind == "ties":
        x = x.round() + 0.0
    if kind == "equal":
        x = torch.zeros_like(x)
    if kind == "few":
        c[top // 2 + 1:] = float("-inf")
    ids, w = moe.route(Cols(x), moe.Router(E, top, 1, 1, 1.0, c, renorm=False))
    s = torch.sigmoid(x[0].double())
    order = (x[0] + c).sort(dim=1, descending=True, stable=True).indices[:, :top]
    n = min(top, top // 2 + 1) if kind == "few" else top
    assert torch.equal(ids[:, :n].long(), order[:, :n])
    torch.testing.assert_close(w[:, :n].double(), s.gather(1, order)[:, :n], rtol=2.0 ** -21, atol=0)      # an exponential of 2 ulp
    if kind == "few":            # nothing is left to choose
        assert bool((ids[:, n:] == E - 1).all()) and bool((w[:, n:] == 0).all())


@pytest.mark.parametrize("split", [1, 3, 9])
@pytest.mark.parametrize("W", [1, 1020, 4096, 4100, 16384, 16400])
def test_rows_of_few_and_of_many_are_the_same(W, split):
    """256 rows ask for all they need at once, 257 do not, nor do rows wider than one vector a thread: the same sums."""
    from copilot_for_consensus_amd.ops import branch, gated, stream
    from copilot_for_consensus_amd.ops.cols import Cols
    g = torch.Generator(device=DEV).manual_seed(W + split)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    T, bf = 257, torch.bfloat16
    x, y, y2, gate, hist = rnd(T, W), rnd(split, T, W), rnd(split, T, W), rnd(split, T, W), rnd(5, T, W)
    gain, w1, w2, bias, dwa = rnd(W), rnd(W), rnd(W), rnd(W), torch.rand(6, device=DEV, generator=g)
    rows, own = rnd(4 * T, W).to(bf), rnd(T, W).to(bf)
    pos = torch.randint(0, 4 * T, (T, 5), device=DEV, generator=g).int()
    ids, wt = torch.randint(0, 5, (T, 5), device=DEV, generator=g).int(), torch.rand(T, 5, device=DEV, generator=g)

    def results(n):
        c = lambda t: t[..., :n, :].contiguous()  # noqa: E731
        out = []

        def norm(fn, *a, **kw):
            s, h = c(x).clone(), torch.empty(n, W, device=DEV, dtype=bf)
            fn(s, h, *a, **kw)
            out.extend([s, h])

        norm(lambda s, h: branch.branch_norm(s, branch.Branch(gain, 1e-6, y=c(y)), w1, 1e-6, h))
        norm(lambda s, h: branch.branch_norm(s, branch.Branch(gain, 1e-6, y=c(y), w=w1, y2=c(y2), w2=w2), w2, 1e-6, h))
        norm(lambda s, h: branch.branch_norm(s, branch.Branch(gain, 1e-6, y=c(y), routed=(rows, c(pos), c(wt), c(ids), 4, c(own))), w1, 1e-6, h))
        for z in (Cols(c(gate)), Cols(c(gate)[0].to(bf))):
            norm(lambda s, h: gated.gated_norm(s, gated.Branch(z, bias, w1, 1e-6, y=c(y), y2=c(y2)), bf, h))
            norm(lambda s, h: gated.gated_shift(s, gated.Branch(z, bias, w1, 1e-6, y=c(y)), bf, h))
        up = stream.Update(c(y), bias, dwa, 5)
        a, r = torch.empty(n, W, device=DEV), torch.empty(n, device=DEV)
        stream.depth_stats(c(x), c(hist).clone(), stream.Update(c(y), bias, dwa[:5], 4), 1e-6, a, r)
        out.extend([a, r[:, None], stream.depth_norm(c(x), torch.cat([c(hist), c(x)[None]]), up, w1, 1e-6, bf)])
        return out

    for few, many in zip(results(T - 1), results(T)):
        assert torch.equal(few, many[:T - 1])
