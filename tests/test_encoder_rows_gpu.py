"""The encoder's kernels for few and for many rows (encoder.hip) at the edges of their tiles, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _model(cfg, seed):
    from copilot_for_consensus_amd.models.encoder import EncoderModel
    m = EncoderModel.random(cfg, DEV, seed=seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    for t in [m.p["emb_g"], m.p["emb_b"]] + [lw[k] for lw in m.layers for k in lw]:
        if t.dim() == 1:           # no norm's gain or bias is one or zero
            t.add_(0.1 * torch.randn(t.shape, device=DEV, generator=g).bfloat16())
    return m


def _states(m, ids, lens):
    """Token states in float64, sequence by sequence."""
    c, out = m.cfg, []
    ln = lambda x, g, b: torch.nn.functional.layer_norm(x, (c.hidden,), g.double(), b.double(), c.ln_eps)  # noqa: E731
    for part in ids.split(lens):
        x = ln(m.p["word"].double()[part] + m.p["pos"].double()[:len(part)] + m.p["type"].double()[0], m.p["emb_g"], m.p["emb_b"])
        for lw in m.layers:
            w = {k: v.double() for k, v in lw.items()}
            q, k, v = (t.view(len(part), c.heads, -1).transpose(0, 1) for t in (x @ w["qkv"].T + w["qkv_b"]).chunk(3, 1))
            a = (torch.softmax(q @ k.transpose(1, 2) * m.scale, -1) @ v).transpose(0, 1).reshape(len(part), -1)
            x = ln(x + a @ w["o"].T + w["o_b"], w["ln1_g"], w["ln1_b"])
            h = torch.nn.functional.gelu(x @ w["up"].T + w["up_b"])
            x = ln(x + h @ w["down"].T + w["down_b"], w["ln2_g"], w["ln2_b"])
        out.append(x)
    return torch.cat(out)


@pytest.mark.parametrize("lens", [[1], [15], [16, 1], [17, 46], [64], [65], [256, 256, 1], [200] * 12 + [160], [200] * 12 + [161],
                                  [256] * 52 + [1], [256] * 52 + [127, 1], [250] * 60 + [99]], ids=lambda v: str(sum(v)))
def test_rows_against_float64(lens):
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=3), seed=len(lens))
    T = sum(lens)
    g = torch.Generator(device=DEV).manual_seed(T)
    ids = torch.randint(0, m.cfg.vocab_size, (T,), device=DEV, dtype=torch.int32, generator=g)
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    tiles = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in K.prefill_tiles(cu.tolist(), K.ENCODER_TILE_ROWS))
    assert K.encoder_weights(T, m.p, m.layers, m.cfg.heads, max(lens)) is not None
    got = m.forward_packed(ids, pos, cu.to(DEV), max(lens), tiles=tiles).double()
    want = _states(m, ids.long(), lens)
    # bf16 states: 2^-9 of a value per rounding, some ten of them a layer that add up as a random walk, 3 layers
    rel = ((got - want).norm(dim=1) / want.norm(dim=1)).max()
    assert rel < 2.0 ** -9 * (3 * 10) ** 0.5, float(rel)


@pytest.mark.parametrize("T", [159, 160, 161, 319, 320, 321, 1279, 1280, 1281, 2687, 2688, 2689, 4095, 4096, 4097, 5440, 5441, 10752, 10753,
                               10880, 10881, 12161, 16383])
def test_rows_at_the_edges_of_the_tiles_rules(T):
    """Where the next larger tiles take over, with last tiles of one row, of all but one and of all."""
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=2), seed=T)
    lens = [250] * (T // 250) + [T % 250]
    g = torch.Generator(device=DEV).manual_seed(T)
    ids = torch.randint(0, m.cfg.vocab_size, (T,), device=DEV, dtype=torch.int32, generator=g)
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    tiles = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in K.prefill_tiles(cu.tolist(), K.ENCODER_TILE_ROWS))
    assert K.encoder_weights(T, m.p, m.layers, m.cfg.heads, 250) is not None
    got = m.forward_packed(ids, pos, cu.to(DEV), 250, tiles=tiles).double()
    want = _states(m, ids.long(), lens)
    rel = ((got - want).norm(dim=1) / want.norm(dim=1)).max()
    assert rel < 2.0 ** -9 * (2 * 10) ** 0.5, float(rel)        # roundings as above


def test_what_the_kernels_are_not_built_for():
    """Other shapes, types and alignments keep the general path."""
    from copilot_for_consensus_amd.models.encoder import EncoderModel
    from copilot_for_consensus_amd.ops import kernels as K
    m = EncoderModel.random("minilm-l6", DEV, seed=0)
    ok = lambda **kw: K.encoder_weights(kw.get("T", 12), m.p, kw.get("layers", m.layers), kw.get("heads", 12), kw.get("S", 12))  # noqa: E731
    assert ok() and ok(heads=6) and ok(T=4096) and ok(T=1 << 20)
    assert not (ok(T=0) or ok(S=513) or ok(heads=4) or ok(layers=[]))
    lw = dict(m.layers[0])
    odd = torch.empty(lw["o"].numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view_as(lw["o"])
    for bad in (lw["o"].float(), lw["o"].t(), odd, lw["o"][:, :352]):
        assert not ok(layers=[dict(lw, o=bad)])
    texts = [list(range(3, 20)), [7], list(range(100, 350))]
    want = m.encode_ids(texts)
    m.layers = [dict(lw, o=odd.copy_(lw["o"])) for lw in m.layers[:1]] + m.layers[1:]
    assert torch.allclose(m.encode_ids(texts), want, atol=4e-3)


@pytest.mark.parametrize("lens,layers", [([16], 1), ([17], 2), ([0, 3, 0, 1, 12, 0], 3), ([31, 1], 2), ([33], 2), ([1] * 63, 2), ([40, 0, 24], 3),
                                         ([1] * 64, 1), ([30, 34], 24), ([30, 34], 25)], ids=lambda v: str(v if isinstance(v, int) else sum(v)))
def test_a_few_short_texts(lens, layers):
    """One launch for all layers: edges of its row groups, texts without tokens, the most layers it takes and one more; a
    captured one again and again, its workspace filled anew each time."""
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=layers), seed=layers)
    T = sum(lens)
    assert (K.kernels().cfc_enc_tiny(T, layers, m.cfg.heads, None) > 0) == (layers <= 24)
    g = torch.Generator(device=DEV).manual_seed(T)
    ids = torch.randint(0, m.cfg.vocab_size, (T,), device=DEV, dtype=torch.int32, generator=g)
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    tiles = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in K.prefill_tiles(cu.tolist(), K.ENCODER_TILE_ROWS))
    cu = cu.to(DEV)
    got = m.forward_packed(ids, pos, cu, max(lens), tiles=tiles)
    want = _states(m, ids.long(), [n for n in lens if n])
    rel = ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max()
    assert rel < 2.0 ** -9 * (layers * 10) ** 0.5, float(rel)       # roundings as above
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        out = m.forward_packed(ids, pos, cu, max(lens), tiles=tiles)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)
        m.forward_packed(ids, pos, cu, max(lens), tiles=tiles)


@pytest.mark.parametrize("lens,layers", [([1], 1), ([12], 6), ([16], 24), ([9, 0, 8], 2), ([20, 12], 3), ([33], 2), ([1] * 40 + [24], 3)],
                         ids=lambda v: str(v if isinstance(v, int) else sum(v)))
def test_a_wait_that_is_given_up(lens, layers):
    """Workgroups of the one launch that give up on one another, at once or after a few loads, say so, and the launch behind
    it leaves the same bits; captured, again in each replay.  Where no wait is given up, it leaves what there is."""
    import ctypes
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=layers), seed=layers)
    T, lib, c = sum(lens), K.kernels(), m.cfg
    g = torch.Generator(device=DEV).manual_seed(T)
    ids = torch.randint(0, c.vocab_size, (T,), device=DEV, dtype=torch.int32, generator=g)
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    tiles = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in K.prefill_tiles(cu.tolist(), K.ENCODER_TILE_ROWS))
    cu, w = cu.to(DEV), K.encoder_weights(T, m.p, m.layers, c.heads, max(lens))
    want = m.forward_packed(ids, pos, cu, max(lens), tiles=tiles)
    call = lambda polls: K.encoder_forward(ids, pos, w, layers, cu, tiles, c.heads, max(lens), m.scale, c.ln_eps, polls)  # noqa: E731
    for polls in (0, 2, -1):
        assert torch.equal(call(polls), want)
    h = torch.empty(lib.cfc_enc_tiny(T, layers, c.heads, None), dtype=torch.bfloat16, device=DEV)
    ptrs, x = (ctypes.c_void_p * (12 * layers))(*w[5:]), torch.empty_like(want)
    for polls, late in ((0, 0), (-1, -1)):
        K.check(lib.cfc_enc_forward(ids.data_ptr(), pos.data_ptr(), *w[:5], cu.data_ptr(), tiles[0].data_ptr(), tiles[1].data_ptr(),
                                    tiles[0].numel(), K.ENCODER_TILE_ROWS, max(lens), layers, ptrs, c.heads, m.scale, c.ln_eps, T,
                                    x.data_ptr(), None, None, None, h.data_ptr(), polls, torch.cuda.current_stream().cuda_stream), "enc")
        assert int(h.view(torch.int32)[-4]) == late and torch.equal(x, want)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        out = call(0)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("lens", [[3, 4, 5], [1] * 16, [15, 2, 15], [16, 16], [31, 2, 31], [7, 30, 27], [1] * 64, [300, 40, 9], [200] * 60],
                         ids=lambda v: "-".join(map(str, v[:3])))
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_text_without_finite_states_spoils_no_other(lens, bad):
    """Where one text's embedding is infinite or not a number, its neighbours' rows are the same bits as without."""
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=2), seed=1)
    texts = [[100 * i + j for j in range(n)] for i, n in enumerate(lens)]
    hit = len(lens) // 2
    texts[hit][lens[hit] // 2] = 29_000
    want = m.encode_ids(texts)
    assert bool(want.isfinite().all())
    m.p["word"][29_000] = bad
    got = m.encode_ids(texts)
    others = [i for i in range(len(lens)) if i != hit]
    assert torch.equal(got[others], want[others]) and not bool(got[hit].isfinite().all())


def test_one_launch_needs_most_of_the_chip():
    """A stream of few CUs, where its workgroups would be long in coming, keeps a launch per product, and gives the same."""
    from copilot_for_consensus_amd.models.encoder import EncoderModel
    from copilot_for_consensus_amd.ops import kernels as K
    from copilot_for_consensus_amd.runtime.cu_partition import partition_streams
    half = partition_streams()[0]
    assert K.kernels().cfc_enc_tiny(12, 6, 12, half.cuda_stream) == 0 < K.kernels().cfc_enc_tiny(12, 6, 12, torch.cuda.Stream().cuda_stream)
    m = EncoderModel.random("minilm-l6", DEV, seed=0)
    texts = [list(range(3, 20)), [7]]
    want = m.encode_ids(texts)
    torch.cuda.synchronize()
    with torch.cuda.stream(half):
        got = m.encode_ids(texts)
    torch.cuda.synchronize()
    assert torch.allclose(got, want, atol=4e-3)


def test_texts_are_not_captured():
    """A graph would read the texts from host memory that is another call's by the time it runs."""
    from copilot_for_consensus_amd.models.encoder import EncoderModel
    m = EncoderModel.random("minilm-l6", DEV, seed=0)
    texts = [list(range(3, 20)), [7]]
    want = m.encode_ids(texts)
    torch.cuda.synchronize()
    x = torch.zeros(8, device=DEV)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with pytest.raises(RuntimeError, match="graph"):
            m.encode_ids(texts)
        x += 1
    g.replay()
    assert torch.equal(m.encode_ids(texts), want) and bool((x == 1).all())


@pytest.mark.parametrize("n", [0, 1, 255, 257, 895, 896])
def test_integers_that_go_with_the_launch(n):
    from copilot_for_consensus_amd.ops import kernels as K
    host = torch.arange(n, dtype=torch.int32) * 5 - 7
    want = host.clone()
    got = K.put_ints(host, DEV)
    host.fill_(-1)              # the launch has them already
    assert torch.equal(got.cpu(), want)
    with pytest.raises(ValueError):
        K.put_ints(torch.zeros(897, dtype=torch.int32), DEV)


@pytest.mark.parametrize("lens", [[1], [3, 4, 0, 5], [256, 64, 65], [256, 129, 20], [256, 130, 20], [7] * 40, [0, 0, 2], [200] * 9])
def test_texts_laid_out_for_the_encoder(lens):
    """What the host lays out for a batch that goes with a launch and one that is copied, against array operations."""
    import numpy as np
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model("minilm-l6", seed=0)
    cu = np.cumsum([0] + lens).astype(np.int64)
    ids = np.arange(cu[-1], dtype=np.int32) % 90
    per = [-(-n // K.ENCODER_TILE_ROWS) for n in lens]
    want = [ids, np.concatenate([np.arange(n) for n in lens]), cu, np.repeat(np.arange(len(lens)), per),
            np.concatenate([np.arange(n) * K.ENCODER_TILE_ROWS for n in per])]
    got, longest = m._texts(ids, cu)
    assert longest == max(lens) and all(np.array_equal(a.cpu().numpy(), b) for a, b in zip(got, want))
    for bad in ([0, 5, 3], [0, len(ids) + 1], [1, 2]):
        with pytest.raises(ValueError):
            m.encode_packed(ids, bad)


@pytest.mark.parametrize("rows", [32769, 32768 + 65, 33024 + 33, 65536])
def test_projections_of_more_rows_than_a_workgroup_a_cu(rows):
    """Workgroups of 256 rows: a last one of one row, of one wave, of a wave and one row, none.  The same sums as those of
    128 rows: the same texts in two batches of fewer rows, bit for bit."""
    import dataclasses
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    from copilot_for_consensus_amd.ops import kernels as K
    m = _model(dataclasses.replace(get_encoder_config("minilm-l6"), layers=2), seed=rows)
    g = torch.Generator(device=DEV).manual_seed(rows)
    lens = [256] * (rows // 256) + ([rows % 256] if rows % 256 else [])

    def states(lens, ids):
        pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)
        cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)
        tiles = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in K.prefill_tiles(cu.tolist(), K.ENCODER_TILE_ROWS))
        return m.forward_packed(ids, pos, cu.to(DEV), max(lens), tiles=tiles)

    ids = torch.randint(0, m.cfg.vocab_size, (rows,), device=DEV, dtype=torch.int32, generator=g)
    half = len(lens) // 2
    cut = sum(lens[:half])
    assert 10753 <= cut <= 32768 and 10753 <= rows - cut <= 32768
    assert torch.equal(states(lens, ids), torch.cat([states(lens[:half], ids[:cut]), states(lens[half:], ids[cut:])]))
