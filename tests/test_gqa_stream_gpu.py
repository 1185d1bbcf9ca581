"""Grouped decode attention, its keys and values through rings in LDS: both sides of each rule that splits the work, and tiles
that come by rows (pooled pages, the far range's last), against the fp32 reference of some of the sequences."""
import numpy as np
import pytest
import torch

from copilot_for_consensus_amd.ops import gqa as A
from copilot_for_consensus_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

CASES = [  # sequences, H, G, dim, mask, keys of the first, of the others, slices, bias
    (2, 4, 2, 64, A.Mask(0), 16900, 40, 1, False),            # more tiles than a wave's lanes hold pages, eight waves
    (2, 4, 2, 64, A.Mask(16400), 16900, 16500, 2, False),     # the same behind a window
    (65, 8, 8, 32, A.Mask(0), 8300, 64, 1, False),            # four waves
    (65, 8, 8, 128, A.Mask(0), 64, 33, 1, False),             # two blocks: a wave each
    (65, 16, 8, 128, A.Mask(0), 65, 1, 1, True),              # three
    (2, 16, 8, 128, A.Mask(0), 128, 31, 1, False),            # four and five, few workgroups
    (2, 16, 8, 128, A.Mask(0), 129, 128, 1, False),
    (32, 8, 8, 128, A.Mask(0), 700, 200, 1, True),            # 256 workgroups, and more
    (33, 8, 8, 128, A.Mask(0), 700, 200, 1, False),
    (33, 8, 8, 64, A.Mask(0), 700, 200, 2, False),            # 528 of 64 columns
    (32, 8, 8, 160, A.Mask(0), 300, 100, 1, False),           # more than 128 columns
    (33, 8, 8, 160, A.Mask(0), 300, 100, 1, True),
    (33, 8, 8, 192, A.Mask(100, keep=40), 300, 100, 2, False),
    (65, 8, 8, 256, A.Mask(0), 100, 70, 1, False),
    (3, 40, 2, 96, A.Mask(0), 500, 100, 3, False),            # more rows of a key head than a tile's
    (3, 8, 2, 128, A.Mask(64, pool=1), 400, 90, 1, False),    # pages of 32, 16, 4 and one entries
    (3, 8, 2, 128, A.Mask(64, pool=2), 400, 90, 2, False),
    (3, 8, 2, 64, A.Mask(64, pool=8), 1200, 90, 1, False),
    (3, 8, 2, 160, A.Mask(64, pool=40), 1900, 90, 3, False),
    (3, 8, 2, 128, A.Mask(64, keep=64), 400, 90, 1, False),   # kept tokens: whole blocks, and a part
    (3, 8, 2, 128, A.Mask(64, keep=70), 400, 90, 2, True),
    (3, 8, 2, 128, A.Mask(64, chunked=True), 400, 129, 2, True)]


@pytest.mark.parametrize("case", CASES)
def test_decoded_tokens_by_the_stream(case):
    B, H, G, D, mask, n0, n1, P, biased = case
    gen = torch.Generator().manual_seed(sum(case[:4]) + n0)
    rnd = lambda *s: torch.randn(*s, generator=gen)
    lens = [n0] + [n1] * (B - 1)
    width, need = -(-max(lens) // 32), [-(-n // 32) for n in lens]
    order, blocks = torch.randperm(sum(need), generator=gen).tolist(), sum(need) + 1
    table = np.full((B, width), blocks - 1)                    # past a sequence: a block of no one's
    for s, m in enumerate(need):
        table[s, :m] = [order.pop() for _ in range(m)]
    table = torch.tensor(table, dtype=torch.int32)
    bias = rnd(H, 37) if biased else None
    a = A.Heads(H, G, D, D, D ** -0.5, mask, 1e-5, None, None, True, rnd(H), bias=bias)
    e = A.pool_entries(mask.pool) if mask.pool else 0
    k, v = (rnd(blocks, G, 32, D).bfloat16() for _ in range(2))
    pk, pv = (rnd(blocks, G, e, D).bfloat16() if e else None for _ in range(2))
    plain = [c.clone() if c is not None else None for c in (k, v, pk, pv)]     # the reference multiplies what it does not see by 0
    if mask.keep % 32:                                        # behind the kept tokens, ahead of every window: no one sees these
        for s in range(B):
            if lens[s] - mask.size >= 32 * (mask.keep // 32 + 1):
                for c in (k, v):
                    c[int(table[s, mask.keep // 32]), :, mask.keep % 32:] = float("nan")
    if e:                                                     # entries past the last that is seen
        for s in range(B):
            n = max(lens[s] - mask.size, 0) // mask.pool
            if n % e:
                for c in (pk, pv):
                    c[int(table[s, n // e]), :, n % e:] = float("nan")
    q = (rnd(B, H, D) * a.scale * A.LOG2E).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32)

    class Rows:
        pool, log2_entries = mask.pool, e.bit_length() - 1 if e else 0
    rows = Rows()
    rows.k, rows.v, rows.pk, rows.pv = (c.cuda() if c is not None else None for c in (k, v, pk, pv))
    dev = A.Heads(H, G, D, D, a.scale, mask, 1e-5, None, None, True, a.sink.cuda(), bias=bias.cuda() if biased else None)
    got = A.attention(dev, q.cuda(), rows, table.cuda(), ctx.cuda(), P=P).float().cpu()
    some = sorted({0, B // 2, B - 1})
    want = ref.grouped_attention(q[some], *plain[:2], plain[2:], table[some], range(len(some) + 1), [lens[s] for s in some], mask.size,
                                 mask.keep, mask.pool, a.sink, D, mask.chunked, 0.0, bias)
    # weights and results are rounded to bf16, half a unit of 2^-8 each: of no more than the largest value
    top = max(float(c.abs().max()) for c in plain[1::2] if c is not None)
    assert torch.isfinite(got).all()
    assert float((got[some] - want).abs().max()) <= 2.0 ** -8 * top
