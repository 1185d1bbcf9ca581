"""A flat search: what knn_topk and its parts allot, pass on and refuse, without a GPU."""
import types

import pytest
import torch

from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops._native import kernels, kernels_available

pytestmark = pytest.mark.skipif(not kernels_available(), reason="the built library is missing")


def _fake(*shape):
    """A tensor on the GPU as far as knn_topk looks at it: its launches are recorded, not made."""
    return types.SimpleNamespace(shape=shape, is_cuda=True, device="cpu", data_ptr=lambda: 0, element_size=lambda: 2)


def _record(monkeypatch):
    """(entry, its arguments) of every call."""
    seen = []
    lib = types.SimpleNamespace(cfc_topk_block=kernels().cfc_topk_block, cfc_topk_segment=kernels().cfc_topk_segment)
    for name in ("cfc_knn_scan", "cfc_topk_select", "cfc_knn_maxima", "cfc_knn_blocks"):
        setattr(lib, name, lambda *a, name=name: seen.append((name, a)) or 0)
    monkeypatch.setattr(K, "kernels", lambda: lib)
    monkeypatch.setattr(K, "_stream", lambda t: None)
    return seen


@pytest.mark.parametrize("nq", (1, 3, 7, 15, 16))
def test_block_maxima_have_room(monkeypatch, nq):
    """The blocks of n scores are not monotonic in n: 270000 are 8438 blocks of 32, 262144 are 16384 of 16."""
    seen = _record(monkeypatch)
    sizes = {1, 15, 16, 17, 5003, 5_500_000, 10_000_000, 35_000_000, 100_000_000} | {16384 * 2 ** a + d for a in range(4, 13) for d in (-1, 0, 1)}
    for rows in sorted(sizes):
        for k in (10, 256):
            K.knn_topk(_fake(rows + 7, 128), _fake(nq, 128), k, row_lo=7)
            for name, a in seen:
                if name == "cfc_knn_scan":
                    n, ld, room = a[2], a[9], a[11]
                    assert n == rows <= ld
                elif name == "cfc_topk_select":
                    n, ld, room = a[3], a[4], a[7]
                    assert n <= ld and a[5] <= n
                elif name == "cfc_knn_maxima":
                    assert a[2] == rows and a[9] >= -(-rows // 16)
                    continue
                else:
                    assert a[9] == min(k, -(-rows // 16))
                    continue
                assert room >= nq * -(-n // kernels().cfc_topk_block(n)), (name, rows, n)
            assert (seen[0][0] == "cfc_knn_scan") == (rows <= K.KNN_SCORES)
            seen.clear()


@pytest.mark.skipif(torch.cuda.is_available(), reason="looks at what is refused before any launch")
def test_entries_refuse_too_little_room():
    room = 15 * -(-270_000 // kernels().cfc_topk_block(270_000))
    assert kernels().cfc_knn_scan(None, None, 262_144, 15, 128, None, None, None, None, 262_144, 16, room, None) == -1
    assert kernels().cfc_topk_select(None, None, 15, 262_144, 262_144, 10, 16, room, 0, 0, None, None, None) == -1


@pytest.mark.parametrize("lo, hi", [(-1, 100), (-5, 0), (0, 101), (50, 50), (60, 50), (100, 101)])
def test_rows_outside_the_index_are_refused(monkeypatch, lo, hi):
    seen = _record(monkeypatch)
    with pytest.raises(ValueError):
        K.knn_topk(_fake(100, 128), _fake(1, 128), 10, row_lo=lo, N=hi)
    assert not seen


def test_rows_of_scores_keep_their_distance(monkeypatch):
    """A column transposed is one contiguous row of stride 1; a flat result is rows one after the other."""
    seen = _record(monkeypatch)
    X, Q, Q1 = (_fake(n, 128) for n in (40, 3, 1))
    for q, out, want in ((Q, None, 40), (Q, torch.empty(3, 52)[:, :40], 52), (Q, torch.empty(120), 40), (Q1, torch.empty(40, 1).t(), 40),
                         (Q1, torch.empty(2, 44)[1:, 4:], 44)):
        K.knn_scores(X, q, out=out)
        assert seen.pop()[1][9] == want
    for scores, want in ((torch.empty(40, 1).t(), 40), (torch.empty(3, 52)[:, :40].contiguous(), 40), (torch.empty(3, 52), 52)):
        K._select(scores, 40, 5, None, None)
        assert seen.pop()[1][4] == want


def test_segments_cover_the_scores_in_whole_blocks():
    """Every workgroup's share fits its registers' block maxima, and the last one holds as many as can be asked for."""
    lib = kernels()
    for n in [1, 15, 2048, 262_144, 262_145] + [(1 << 20) * a + d for a in (1, 2, 3, 7, 64, 2000) for d in (-1, 0, 1, 63, 64, 65, 500_000)]:
        seg, B = lib.cfc_topk_segment(n), lib.cfc_topk_block(n)
        parts = -(-n // seg)
        assert -(-seg // B) <= 16384 and B in (16, 32, 64)
        assert parts == 1 or seg % B == 0 and n - (parts - 1) * seg >= 2048
