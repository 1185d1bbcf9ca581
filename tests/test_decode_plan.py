"""How decode attention shares its work out (host rules)."""
import math
import types

import pytest
import torch


def test_kv_partitions_fill_rounds_and_leave_short_contexts_whole():
    from copilot_for_consensus_amd.models.decoder import kv_partitions
    for B in (1, 2, 3, 5, 8, 24, 48, 64, 100, 128, 300):
        for blocks in (0, 1, 2, 3, 8, 24, 88, 176, 1024):
            P = kv_partitions(B, 32, 8, blocks)
            assert 1 <= P <= max(1, min(64, blocks // 2))
            if blocks <= 8 or B % 64 == 0:
                assert P == 1                                    # few keys, or whole rounds of 512 workgroups as they are
    for B in (3, 5, 24, 48):
        P = kv_partitions(B, 32, 8, 176)
        assert B * 8 * P % 512 == 0 or B * 8 * P % 512 > 128     # not a round for a few workgroups


def _model(heads, kv_heads, window=0):
    import functools
    from copilot_for_consensus_amd.models.decoder import DecoderModel
    w = types.SimpleNamespace(heads=heads, kv_heads=kv_heads)
    m = types.SimpleNamespace(w=w, window=window)
    m.decode_partitions = functools.partial(DecoderModel.decode_partitions, m)
    return m


@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (4, 1), (8, 2), (64, 8), (40, 10)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_engines_partitions_are_no_slower_for_short_contexts(heads, kv_heads, dtype, monkeypatch):
    """An engine's tables are as wide as its contexts may become: no more partitions than give 512 workgroups, whose launch
    short contexts would pay for, and those of the 8-bit cache as they were."""
    from copilot_for_consensus_amd.models.decoder import kv_partitions
    from copilot_for_consensus_amd.runtime.engine import LLMEngine
    monkeypatch.delenv("CFC_DECODE_WGS", raising=False)
    m = _model(heads, kv_heads)
    engine = types.SimpleNamespace(model=m, kv=types.SimpleNamespace(dtype=dtype))
    for B in (1, 2, 3, 5, 12, 24, 48, 91, 128):
        for blocks in (8, 24, 48, 128, 256, 344):
            fewest = min(max(1, math.ceil(512 / (B * kv_heads))), max(1, blocks // 2))
            P = -LLMEngine._part_blocks(engine, B, blocks)
            assert 1 <= P <= fewest and (P == fewest or dtype == torch.bfloat16)
            if dtype == torch.bfloat16:
                assert P == min(fewest, kv_partitions(B, heads, kv_heads, blocks))
                full = m.decode_partitions(B, blocks)
                assert full == (kv_partitions(B, heads, kv_heads, blocks) if (heads, kv_heads) == (32, 8) else P)
    monkeypatch.setenv("CFC_DECODE_WGS", "2048")
    assert -LLMEngine._part_blocks(engine, 128, 88) == m.decode_partitions(128, 88) == math.ceil(2048 / (128 * kv_heads))


def test_where_a_decode_step_turns_its_queries():
    """Inside its attention: few sequences always, more where the streaming kernels take them and win back the longer start."""
    from copilot_for_consensus_amd.ops import kernels as K
    inside = K.rope_inside
    assert all(inside(b, 8, n, p, t) for b in (1, 4) for n in (2, 500) for p in (-3, 16) for t in (True, False))
    assert inside(5, 8, 500, -6, True) and inside(32, 8, 90, -1, True) and inside(128, 8, 64, -1, True)
    assert not inside(33, 8, 65, -1, True) and not inside(128, 8, 88, -2, True)      # long contexts, two workgroups a CU
    assert not inside(5, 8, 40, -6, False) and not inside(5, 8, 40, 16, True) and not inside(129, 8, 4, -1, True)


def test_where_a_decode_step_turns_its_queries_without_the_ring():
    """Kernels that take keys and values to registers: inside for up to two workgroups a CU, and so whatever the engine plans; not in
    slices of a few blocks that are more, by their number or by a window."""
    from copilot_for_consensus_amd.models.decoder import kv_partitions
    from copilot_for_consensus_amd.ops import kernels as K
    inside = K.rope_inside
    for B in range(5, 129):
        for Hq, Hkv in ((32, 8), (16, 4), (8, 2), (4, 1), (64, 8)):
            for blocks in (1, 2, 3, 8, 9, 16, 22, 47, 64):
                P = kv_partitions(B, Hq, Hkv, blocks)
                assert inside(B, Hkv, blocks, -P, True) == (B * Hkv * P <= 512 or not K.paged_waves(B * Hkv * P, blocks, P)[2]), (B, Hkv, blocks, P)
    for B, blocks, P, window in ((64, 16, 4, 0), (128, 8, 2, 0), (128, 64, 2, 200), (33, 8, 2, 0)):
        assert K.paged_waves(B * 8 * P, min(blocks, (window + 30) // 32 + 1) if window else blocks, P)[2]
        assert not inside(B, 8, blocks, -P, True, window)
    assert inside(32, 8, 8, -2, True) and inside(128, 8, 64, -2, True) and inside(128, 8, 64, -2, True, 2048)
