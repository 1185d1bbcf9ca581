"""Decode attention in slices of no, one and few key tiles: a slice's start asks for its first tiles at once and reads none
past its end.  Against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tables(B, longest, g):
    n = -(-longest // 32)
    return torch.randperm(B * n, device=DEV, generator=g).int().view(B, n).contiguous(), B * n


def _close(got, want, scale):
    # bf16 weights and results (2^-9 each, of values that add up to `scale` at most); scores are fp32 sums
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -9 * scale).all()), float((got.double() - want).abs().max())


@pytest.mark.parametrize("H,RS,RV", [(3, 64, None), (16, 512, None), (32, 512, None), (64, 256, None), (20, 96, None), (32, 576, 512), (40, 192, 128)])
@pytest.mark.parametrize("P", [1, 2, 3, 5, 16])
@pytest.mark.parametrize("window", [0, 100])
def test_latent_slices(H, RS, RV, P, window):
    from copilot_for_consensus_amd.ops import latent
    ctx = [1, 63, 64, 65, 127, 128, 129, 191, 193, 320, 385]
    g = torch.Generator(device=DEV).manual_seed(H * P + RS)
    bt, blocks = _tables(len(ctx), max(ctx), g)
    cache = torch.randn(blocks, 32, RS, device=DEV, generator=g).bfloat16()
    q = torch.randn(len(ctx), H, RS, device=DEV, generator=g).bfloat16()
    out = latent.latent_attention(q, cache, bt, None, torch.tensor(ctx, dtype=torch.int32, device=DEV), RS ** -0.5, P=P, window=window, RV=RV)
    for s, n in enumerate(ctx):
        c = cache[bt[s].long()].reshape(-1, RS)[max(0, n - window) if window else 0:n].double()
        p = torch.softmax(q[s].double() @ c.T * RS ** -0.5, -1)
        v = c[:, :RV]
        _close(out[s], p @ v, (p @ v.abs()).max())


@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (16, 1, 64), (40, 2, 128), (4, 4, 256)])
@pytest.mark.parametrize("P", [1, 2, 3, 7])
def test_grouped_slices(H, G, D, P):
    """Waves of no, one, two and three 32-key tiles."""
    from copilot_for_consensus_amd.ops import gqa
    from copilot_for_consensus_amd.runtime.kv_cache import PagedHeads
    ctx = [1, 31, 33, 64, 128, 129, 160, 257, 300, 390, 500]
    g = torch.Generator(device=DEV).manual_seed(H * P + D)
    bt, blocks = _tables(len(ctx), max(ctx), g)
    rows = PagedHeads(blocks, G, D, 0, 0, DEV, torch.bfloat16)
    for t in (rows.k, rows.v):
        t.copy_(torch.randn(t.shape, device=DEV, generator=g))
    a = gqa.Heads(H, G, D, D, D ** -0.5, gqa.Mask(0), 1e-6, None, None, False, None)
    q = (torch.randn(len(ctx), H, D, device=DEV, generator=g) * a.q_scale).bfloat16()
    out = gqa.attention(a, q, rows, bt, torch.tensor(ctx, dtype=torch.int32, device=DEV), P=P)
    for s, n in enumerate(ctx):
        kk, vv = (t[bt[s].long()].transpose(1, 2).reshape(-1, G, D)[:n].double().transpose(0, 1).contiguous() for t in (rows.k, rows.v))
        p = torch.softmax((q[s].double().view(G, H // G, 1, D) * kk[:, None]).sum(-1) / gqa.LOG2E, -1)
        _close(out[s].view(G, H // G, D), torch.matmul(p, vv), torch.matmul(p, vv.abs()).max())


@pytest.mark.parametrize("P", [2, 7, 15, 16, 17, 33, 63, 64, 65, 128, 131])
def test_merge_of_partitions(P):
    """Whole and broken runs of sixteen and sixty-four partitions, most of them empty for the short sequences; rows that are
    no whole workgroups of four, and a workspace and an output no more aligned than their elements."""
    from copilot_for_consensus_amd.ops import kernels as K
    ctx = [1, 32, 33, 500, 65 * 32, 131 * 32]
    heads, kv, D = 3, 3, 128
    g = torch.Generator(device=DEV).manual_seed(P)
    bt, blocks = _tables(len(ctx), max(ctx), g)
    kc = torch.randn(blocks, kv, 32, D, device=DEV, generator=g).bfloat16()
    vc = torch.randn(blocks, kv, D, 32, device=DEV, generator=g).bfloat16()
    q = torch.randn(len(ctx), heads, D, device=DEV, generator=g).bfloat16()
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    want = K.paged_decode_attention(q, kc, vc, bt, lens, D ** -0.5, part_blocks=-1)
    n = len(ctx) * heads * P * (D + 2)
    ws = torch.full((n + 1,), float("nan"), device=DEV)[1:]
    out = torch.full((q.numel() + 1,), float("nan"), device=DEV, dtype=torch.bfloat16)[1:].view_as(q)
    got = K.paged_decode_attention(q, kc, vc, bt, lens, D ** -0.5, part_blocks=-P, workspace=ws, out=out)
    # weights of a partition are rounded to bf16 from another maximum (2^-9 each, of values up to 4.5), results once more
    assert bool(((got.double() - want.double()).abs() <= 2.0 ** -8 * want.double().abs() + 2.0 ** -8).all())


@pytest.mark.parametrize("P", [1, 2, 3, 5, 8, 15, 16, 17, 33])
def test_merge_of_an_infinite_sum(P):
    """An infinite value, in the last partition or in all, is infinite in the result, and alone there."""
    from copilot_for_consensus_amd.ops import kernels as K
    g = torch.Generator(device=DEV).manual_seed(P)
    bt, blocks = _tables(2, 20 * 32, g)
    kc = torch.randn(blocks, 1, 32, 128, device=DEV, generator=g).bfloat16()
    vc = torch.randn(blocks, 1, 128, 32, device=DEV, generator=g).bfloat16()
    q = torch.randn(2, 1, 128, device=DEV, generator=g).bfloat16()
    lens = torch.tensor([640, 640], dtype=torch.int32, device=DEV)

    def run(P):
        return K.paged_decode_attention(q, kc, vc, bt, lens, 128 ** -0.5, part_blocks=-P).float()

    vc[bt[0, -1].long(), 0, 3, 31] = float("inf")
    vc[bt[1].long(), 0, 5] = float("-inf")
    one, many = run(1), run(P)
    assert one.isinf().sum() >= 2 and not bool(many.isnan().any())
    assert torch.equal(many[one.isinf()], one[one.isinf()]) and torch.equal(many.isinf(), one.isinf())


@pytest.mark.parametrize("B,kv,P,longest", [(65, 8, 1, 1030), (120, 8, 1, 1030), (66, 8, 2, 1030), (128, 6, 1, 2000), (129, 6, 1, 1030), (1, 9, 57, 2000),
                                            (128, 8, 1, 900)])
def test_longest_first(B, kv, P, longest):
    """More workgroups than are held at once start with the longest sequences: every sequence's result is what it is when the
    batch comes the other way round, whatever the order, with equal lengths among them."""
    from copilot_for_consensus_amd.ops import kernels as K
    heads, D = kv, 128
    g = torch.Generator(device=DEV).manual_seed(B)
    ctx = torch.randint(1, 8, (B,), generator=g, device=DEV) * 37 + torch.arange(B, device=DEV) % 2
    ctx[B // 2:B // 2 + 2] = longest - 6
    ctx[-1:] = longest
    lens = ctx.to(torch.int32)
    bt, blocks = _tables(B, longest + 20, g)
    kc = torch.randn(blocks, kv, 32, D, device=DEV, generator=g).bfloat16()
    vc = torch.randn(blocks, kv, D, 32, device=DEV, generator=g).bfloat16()
    q = torch.randn(B, heads, D, device=DEV, generator=g).bfloat16()
    run = lambda t, *a: K.paged_decode_attention(t, kc, vc, *a, D ** -0.5, part_blocks=-P)  # noqa: E731
    got = run(q, bt, lens)
    assert torch.equal(got.flip(0), run(q.flip(0).contiguous(), bt.flip(0).contiguous(), lens.flip(0).contiguous()))
    part = slice(0, B, max(1, B // 4))                  # another number of sequences, another share of waves
    some = run(q[part].contiguous(), bt[part].contiguous(), lens[part].contiguous())
    # weights rounded to bf16 from another maximum (2^-9 each, of values up to 4.5), results once more
    assert bool(((got[part].double() - some.double()).abs() <= 2.0 ** -8 * some.double().abs() + 2.0 ** -8).all())


def _keys_values(kc, vc, table, n):
    """Keys and values [kv, n, D] in float64 of a sequence, from the cache's layouts."""
    kv, D = kc.shape[1], kc.shape[3]
    slot = torch.tensor([4 * s + j if j < 4 else 16 + 4 * s + j - 4 for s in range(4) for j in range(8)], device=DEV)
    k = kc[table.long()].transpose(0, 1).reshape(kv, -1, D)[:, :n].double()
    t = vc[table.long()].view(-1, kv, 4, D, 8).permute(0, 1, 2, 4, 3).reshape(-1, kv, 32, D)
    v = torch.empty_like(t).index_copy_(2, slot, t).transpose(0, 1).reshape(kv, -1, D)[:, :n].double()
    return k, v


@pytest.mark.parametrize("G", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("B,kv,P", [(24, 8, 1), (40, 8, 1), (40, 8, 3), (70, 8, 1), (9, 1, 5)])
@pytest.mark.parametrize("width", [300, 1100])
def test_keys_and_values_by_the_stream(G, B, kv, P, width):
    """Workgroups of eight and of four waves; waves of no, one, two and three blocks, last blocks of one key; slices and whole
    sequences; a window; shared leading blocks.  Against float64."""
    from copilot_for_consensus_amd.ops import kernels as K
    D, heads = 128, kv * G
    edge = [1, 31, 32, 33, 64, 65, 96, 127, 129, 160, 193, 257, 288, 300]
    ctx = [edge[i % len(edge)] for i in range(B)]
    g = torch.Generator(device=DEV).manual_seed(G * B + P)
    bt, blocks = _tables(B, width, g)
    kc = torch.randn(blocks, kv, 32, D, device=DEV, generator=g).bfloat16()
    vc = torch.randn(blocks, kv, D, 32, device=DEV, generator=g).bfloat16()
    bt[1::2, :2] = bt[:1, :2]                           # what odd sequences share with the first
    q = torch.randn(B, heads, D, device=DEV, generator=g).bfloat16()
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    for window, shared in ((0, None), (70, None), (0, torch.tensor([2], dtype=torch.int32, device=DEV))):
        got = K.paged_decode_attention(q, kc, vc, bt, lens, D ** -0.5, part_blocks=-P, window=window, shared_blocks=shared)
        for s in range(0, B, 3):
            k, v = _keys_values(kc, vc, bt[s], ctx[s])
            lo = max(0, ctx[s] - window) if window else 0
            p = torch.softmax(q[s].double().view(kv, G, D) @ k[:, lo:].transpose(1, 2).contiguous() * D ** -0.5, -1)
            _close(got[s].view(kv, G, D), p @ v[:, lo:], (p @ v[:, lo:].abs()).max())


@pytest.mark.parametrize("G", [1, 4, 16])
@pytest.mark.parametrize("B,kv,first,others", [(40, 8, 64, 33), (70, 8, 33, 64), (2, 2, 16900, 70), (40, 8, 8500, 60)])
def test_stream_of_two_blocks_and_of_many(G, B, kv, first, others):
    """A wave for tables of two blocks; more blocks a wave than its lanes hold, of eight waves and of four.  Against float64."""
    from copilot_for_consensus_amd.ops import kernels as K
    D, ctx = 128, [first] + [others] * (B - 1)
    g = torch.Generator(device=DEV).manual_seed(G + first)
    width = -(-max(ctx) // 32)
    need = [-(-n // 32) for n in ctx]
    order = torch.randperm(sum(need) + 1, device=DEV, generator=g).int()
    bt = order[-1].repeat(B, width)                     # past a sequence: a block of no one's
    for s, m in enumerate(need):
        bt[s, :m] = order[sum(need[:s]):sum(need[:s]) + m]
    kc = torch.randn(len(order), kv, 32, D, device=DEV, generator=g).bfloat16()
    vc = torch.randn(len(order), kv, D, 32, device=DEV, generator=g).bfloat16()
    q = torch.randn(B, kv * G, D, device=DEV, generator=g).bfloat16()
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    for P, window in ((1, 0), (1, 50), (2, 0)):
        got = K.paged_decode_attention(q, kc, vc, bt, lens, D ** -0.5, part_blocks=-P, window=window)
        for s in (0, 1, B - 1):
            k, v = _keys_values(kc, vc, bt[s, :need[s]], ctx[s])
            lo = max(0, ctx[s] - window) if window else 0
            p = torch.softmax(q[s].double().view(kv, G, D) @ k[:, lo:].transpose(1, 2).contiguous() * D ** -0.5, -1)
            _close(got[s].view(kv, G, D), p @ v[:, lo:], (p @ v[:, lo:].abs()).max())
