"""Row kernels of prompts whose share of rows or work per workgroup follows the prompt's length."""
import pytest
import torch

from copilot_for_consensus_amd.ops import gqa as A
from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops import latent as L
from copilot_for_consensus_amd.ops.cols import Cols
from copilot_for_consensus_amd.runtime.kv_cache import PagedHeads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", (0, 4))
@pytest.mark.parametrize("per_head", (True, False))
def test_projections_of_a_row_do_not_depend_on_the_prompt(taps, per_head):
    """4, 8 and 16 rows per workgroup, ragged last ones: the same queries and cache rows bit for bit."""
    H, G, dim, dev = 8, 2, 64, "cuda"
    g = torch.Generator(dev).manual_seed(3)

    def rnd(*s):
        return torch.randn(*s, device=dev, generator=g)
    a = A.Heads(H=H, G=G, dim=dim, vdim=dim, scale=0.3, mask=A.Mask(20, keep=2), eps=1e-2, per_head=per_head, sink=None, freq=A.rope_freq(dim, 1e4, dev),
                q_norm=rnd(dim if per_head else H * dim), k_norm=rnd(dim if per_head else G * dim),
                conv=rnd(taps, (H + 2 * G) * dim) if taps else None)
    u = rnd(2100, a.columns).bfloat16()
    tail = rnd(2, 3, a.columns) if taps else None

    def run(T):
        n = -(-T // 32)
        rows = PagedHeads(n, G, a.D, 0, 0, dev, torch.bfloat16)
        at = torch.arange(T, dtype=torch.int32, device=dev)
        table = torch.arange(n, dtype=torch.int32, device=dev)[None]
        q = A.qkv_rows(a, Cols(u[:T]), rows, at, at, torch.ones_like(at), table, tail, at)
        return q, rows.k.transpose(1, 2).reshape(n * 32, G, -1)[:T], rows.v.transpose(1, 2).reshape(n * 32, G, -1)[:T]
    whole = run(2100)                                       # 132 workgroups of 16 rows and each of two parts
    for T in (1, 3, 4, 5, 17, 90, 511, 1021, 2049):         # 4 rows up to 1020, 8 up to 2040
        for x, y in zip(run(T), whole):
            assert torch.equal(x, y[:T])


@pytest.mark.parametrize("n_tiles", (1, 3, 63, 64, 65, 255, 600))
def test_gathered_latents_are_the_cache_rows(n_tiles):
    """Eight workgroups per 64-row tile down to one: rows, their slot order and the rest of the row, past the end zero."""
    RV, RS, dev = 512, 576, "cuda"
    g = torch.Generator(dev).manual_seed(n_tiles)
    tokens = 64 * n_tiles - 37
    blocks = -(-tokens // 32)
    cache = torch.randn(blocks, 32, RS, device=dev, generator=g).bfloat16()
    table = torch.randperm(blocks, device=dev, generator=g).to(torch.int32)[None]
    tiles = torch.tensor([[0, 64 * i] for i in range(n_tiles)], dtype=torch.int32, device=dev)
    rows = torch.full((2, n_tiles * 64, RV), 7.0, device=dev, dtype=torch.bfloat16)
    k2 = torch.full((n_tiles * 64, 64), 7.0, device=dev, dtype=torch.bfloat16)
    lib, ctx = L.kernels(), torch.tensor([tokens], dtype=torch.int32, device=dev)
    L.check(lib.cfc_latent_gather(cache.data_ptr(), table.data_ptr(), blocks, ctx.data_ptr(),
                                  tiles.data_ptr(), n_tiles, RS, RV, rows[0].data_ptr(), rows[1].data_ptr(), k2.data_ptr(),
                                  torch.cuda.current_stream().cuda_stream), "cfc_latent_gather")
    want = torch.zeros(n_tiles * 64, RS, device=dev, dtype=torch.bfloat16)
    want[:tokens] = cache[table[0].long()].reshape(-1, RS)[:tokens]
    assert torch.equal(rows[0], want[:, :RV]) and torch.equal(k2, want[:, RV:])
    # the slot-ordered copy: 16-byte pieces of each 32-row, 32-column part, permuted
    part = rows[1].view(n_tiles, RV // 32, 4, 64, 8)
    src = want[:, :RV].view(n_tiles, 64, RV // 32, 4, 8).permute(0, 2, 1, 3, 4)
    assert torch.equal(part.reshape(n_tiles, RV // 32, -1).sort(-1).values, src.reshape(n_tiles, RV // 32, -1).sort(-1).values)


@pytest.mark.parametrize("window", (0, 100))
@pytest.mark.parametrize("H, G", [(4, 4), (4, 2), (8, 2), (16, 8)])
@pytest.mark.parametrize("lens, past", [((1,), 0), ((33,), 0), ((63, 2), 5), ((300,), 0), ((65, 97, 128), 70), ((420,), 31)])
def test_attention_of_a_short_prompt_shares_its_tiles(lens, past, H, G, window):
    """One to eight workgroups per tile against one (the same sequences often enough to fill the chip): bit for bit."""
    dev, D = "cuda", 128
    g = torch.Generator(dev).manual_seed(sum(lens) + past)
    nb = [-(-(n + past) // 32) for n in lens]
    kc = torch.randn(sum(nb), G, 32, D, device=dev, generator=g).bfloat16()
    vc = torch.randn(sum(nb), G, 4, D, 8, device=dev, generator=g).bfloat16().view(sum(nb), G, 32, D)
    q1 = torch.randn(sum(lens), H, D, device=dev, generator=g).bfloat16()
    table = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    at = 0
    for i, n in enumerate(nb):
        table[i, :n] = torch.arange(at, at + n)
        at += n

    def run(copies):
        cu = [0]
        for n in lens * copies:
            cu.append(cu[-1] + n)
        return K.prefill_attention(q1.repeat(copies, 1, 1), kc, vc, table.repeat(copies, 1).to(dev),
                                   torch.tensor(cu, dtype=torch.int32, device=dev),
                                   torch.tensor([n + past for n in lens] * copies, dtype=torch.int32, device=dev), D ** -0.5, window=window)
    assert torch.equal(run(1), run(260)[:sum(lens)])
