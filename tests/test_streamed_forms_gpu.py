"""What comes by LDS-DMA (index rows, decode attention's keys and values) in forms beside the usual: sources that are no whole
sixteens of bytes, masks at any byte, sixteen query heads a key head; and encoder scores at the end of the range.  Against float64."""
import pytest
import torch

import test_gqa_stream_gpu as stream

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _shifted(t):
    """The same values two bytes further on."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    assert out.data_ptr() % 16 == 2
    return out.copy_(t)


def _close(got, want, scale):
    # bf16 weights and results (2^-9 each, of values that add up to `scale` at most); scores are fp32 sums
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -9 * scale).all()), float((got.double() - want).abs().max())


@pytest.mark.parametrize("dim,N", [(768, 5000), (768, 177), (1024, 333), (384, 393_300)])
@pytest.mark.parametrize("lo", [0, 1, 2, 3, 35])
@pytest.mark.parametrize("form", ["l2", "mask", "both", "rows"])
def test_search(dim, N, lo, form):
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(N + lo)
    X, Q = (torch.randn(n, dim, device=DEV, generator=g).bfloat16() for n in (N, 3))
    if form == "rows":
        X = _shifted(X)
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


def _paged(heads, kv, ctx, blocks, g):
    n = -(-max(ctx) // 32)
    bt = torch.randperm(len(ctx) * n, device=DEV, generator=g).int().view(len(ctx), n).contiguous()
    kc = torch.randn(len(ctx) * n, kv, 32, 128, device=DEV, generator=g).bfloat16()
    vc = torch.randn(len(ctx) * n, kv, 128, 32, device=DEV, generator=g).bfloat16()
    q = torch.randn(len(ctx), heads, 128, device=DEV, generator=g).bfloat16()
    return bt, kc, vc, q, torch.tensor(ctx, dtype=torch.int32, device=DEV)


def _paged_want(q, kc, vc, bt, n):
    kv = kc.shape[1]
    slots = torch.tensor([4 * g + j if j < 4 else 16 + 4 * g + j - 4 for g in range(4) for j in range(8)], device=DEV)
    k = kc[bt.long()].transpose(0, 1).reshape(kv, -1, 128)[:, :n].double()
    v = torch.empty(len(bt), kv, 32, 128, dtype=torch.float64, device=DEV)
    v[:, :, slots] = vc[bt.long()].view(-1, kv, 4, 128, 8).permute(0, 1, 2, 4, 3).reshape(-1, kv, 32, 128).double()
    v = v.transpose(0, 1).reshape(kv, -1, 128)[:, :n]
    p = torch.softmax((q.double().view(kv, -1, 1, 128) * k[:, None]).sum(-1) * 128 ** -0.5, -1)
    return torch.matmul(p, v).view(-1, 128), torch.matmul(p, v.abs()).max()


# more than 512 workgroups of uneven contexts, in their order and longest first; few of them
@pytest.mark.parametrize("heads,kv,ctx", [(32, 2, [1500 - 23 * (i % 61) for i in range(128)] ), (16, 1, [900, 33, 1400, 256, 1]), (32, 2, [1300] * 40),
                                          (32, 8, [2100 - 170 * (i % 12) for i in range(90)])])
@pytest.mark.parametrize("P", [1, 3])
def test_many_heads_a_key_head(heads, kv, ctx, P):
    from copilot_for_consensus_amd.ops import kernels as K
    ctx = ctx[:128]
    g = torch.Generator(device=DEV).manual_seed(heads + len(ctx))
    bt, kc, vc, q, lens = _paged(heads, kv, ctx, 0, g)
    got = K.paged_decode_attention(q, kc, vc, bt, lens, 128 ** -0.5, part_blocks=-P)
    for s in {0, 1, len(ctx) // 2, len(ctx) - 1}:
        n = ctx[s]
        _close(got[s], *_paged_want(q[s], kc, vc, bt[s, :-(-n // 32)], n))


@pytest.mark.parametrize("P", [1, 2])
def test_paged_queries_at_any_element(P):
    from copilot_for_consensus_amd.ops import kernels as K
    ctx = [700, 1, 333, 640, 90, 512, 700]
    bt, kc, vc, q, lens = _paged(32, 8, ctx, 0, torch.Generator(device=DEV).manual_seed(P))
    want = K.paged_decode_attention(q, kc, vc, bt, lens, 128 ** -0.5, part_blocks=-P)
    got = K.paged_decode_attention(_shifted(q), kc, vc, bt, lens, 128 ** -0.5, part_blocks=-P)
    # the same weights to bf16 from maxima of other waves' blocks
    assert bool(((got.double() - want.double()).abs() <= 2.0 ** -8 * want.double().abs() + 2.0 ** -8).all())


# keys straight to registers and by the ring, one and several to a slice
@pytest.mark.parametrize("D", [32, 64, 96, 128, 160, 192, 256])
@pytest.mark.parametrize("B,P", [(3, 1), (3, 7), (40, 1), (40, 2), (70, 1)])
@pytest.mark.parametrize("shift", [False, True])
def test_grouped(D, B, P, shift):
    from copilot_for_consensus_amd.ops import gqa
    from copilot_for_consensus_amd.runtime.kv_cache import PagedHeads
    ctx = [700 - 37 * (i % 18) for i in range(B)]
    g = torch.Generator(device=DEV).manual_seed(D + B)
    n = -(-max(ctx) // 32)
    bt = torch.randperm(B * n, device=DEV, generator=g).int().view(B, n).contiguous()
    rows = PagedHeads(B * n, 8, D, 0, 0, DEV, torch.bfloat16)
    for t in (rows.k, rows.v):
        t.copy_(torch.randn(t.shape, device=DEV, generator=g))
    a = gqa.Heads(24, 8, D, D, D ** -0.5, gqa.Mask(0), 1e-6, None, None, False, None)
    q = (torch.randn(B, 24, D, device=DEV, generator=g) * a.q_scale).bfloat16()
    out = gqa.attention(a, _shifted(q) if shift else q, rows, bt, torch.tensor(ctx, dtype=torch.int32, device=DEV), P=P)
    for s in {0, 1, B // 2, B - 1}:
        k, v = (t[bt[s].long()].transpose(0, 1).reshape(8, -1, D)[:, :ctx[s]].double() for t in (rows.k, rows.v))
        p = torch.softmax((q[s].double().view(8, 3, 1, D) * k[:, None]).sum(-1) / gqa.LOG2E, -1)
        _close(out[s].view(8, 3, D), torch.matmul(p, v), torch.matmul(p, v.abs()).max())


# the same with windows, kept tokens, pooled means and biases: queries at any element send every form straight to registers
@pytest.mark.parametrize("case", stream.CASES)
def test_grouped_forms_straight(case, monkeypatch):
    attention = stream.A.attention
    monkeypatch.setattr(stream.A, "attention", lambda a, q, *rest, **kw: attention(a, _shifted(q), *rest, **kw))
    stream.test_decoded_tokens_by_the_stream(case)


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
