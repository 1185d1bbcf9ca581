"""A flat search in spans of rows: what knn_topk allots and refuses, without a GPU."""
import types

import pytest
import torch

from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops._native import kernels, kernels_available

pytestmark = pytest.mark.skipif(not kernels_available(), reason="the built library is missing")


def _fake(*shape):
    """A tensor on the GPU as far as knn_topk looks at it: its launches are recorded, not made."""
    return types.SimpleNamespace(shape=shape, is_cuda=True, device="cpu")


def _search(monkeypatch, rows, nq, k=10, row_lo=0):
    spans = []

    def scan(X, Q, xnorm2, qnorm2, alive, lo, hi, out, bmax):
        spans.append((lo, hi, out, bmax))

    def select(scores, n, k, ids, bmax, row_lo=0):
        return torch.zeros(nq, k), torch.zeros(nq, k, dtype=torch.long)
    monkeypatch.setattr(K, "_knn_scan", scan)
    monkeypatch.setattr(K, "_select", select)
    K.knn_topk(_fake(row_lo + rows, 128), _fake(nq, 128), k, row_lo=row_lo)
    return spans


@pytest.mark.parametrize("small", (False, True))
@pytest.mark.parametrize("nq", range(1, 17))
def test_every_span_has_room_for_its_block_maxima(monkeypatch, nq, small):
    """A last span of fewer rows may have more blocks than a full one: 270000 rows are 8438 blocks of 32, 262144 rows 16384
    blocks of 16."""
    if small:
        monkeypatch.setattr(K, "KNN_SCORES", nq * 270_000)
    step = K.KNN_SCORES // nq
    rests = {1, 5003, step - 1, step} | {16384 * 2 ** a + d for a in range(4, 13) for d in (-1, 0, 1)}
    sizes = {1_000_000, 5_500_000, 10_000_000, 35_000_000, 100_000_000} | {step + r for r in rests} | {2 * step + r for r in rests}
    for rows in sorted(n for n in sizes if 0 < n <= min(100_000_000, 30 * step)):
        spans = _search(monkeypatch, rows, nq, row_lo=7)
        assert spans[0][0] == 7 and spans[-1][1] == 7 + rows and all(a[1] == b[0] for a, b in zip(spans, spans[1:]))
        for lo, hi, out, bmax in spans:
            n = hi - lo
            assert out.shape[0] == nq and n <= out.shape[1]
            assert bmax.numel() >= nq * -(-n // kernels().cfc_topk_block(n)), (rows, n)


@pytest.mark.skipif(torch.cuda.is_available(), reason="looks at what is refused before any launch")
def test_entries_refuse_too_little_room():
    room = 15 * -(-270_000 // kernels().cfc_topk_block(270_000))
    assert kernels().cfc_knn_scan(None, None, 262_144, 15, 128, None, None, None, None, 262_144, 16, room, None) == -1
    assert kernels().cfc_topk_select(None, None, 15, 262_144, 262_144, 10, 16, room, 0, 0, None, None, None) == -1


@pytest.mark.parametrize("lo, hi", [(-1, 100), (-5, 0), (0, 101), (50, 50), (60, 50), (100, 101)])
def test_rows_outside_the_index_are_refused(monkeypatch, lo, hi):
    monkeypatch.setattr(K, "_knn_scan", lambda *a: pytest.fail("launched"))
    with pytest.raises(ValueError):
        K.knn_topk(_fake(100, 128), _fake(1, 128), 10, row_lo=lo, N=hi)


def _strides(monkeypatch):
    """Row strides that the entries are called with."""
    seen = []
    lib = types.SimpleNamespace(cfc_topk_block=kernels().cfc_topk_block, cfc_topk_segment=kernels().cfc_topk_segment,
                                cfc_knn_scan=lambda *a: seen.append(a[9]) or 0, cfc_topk_select=lambda *a: seen.append(a[4]) or 0)
    monkeypatch.setattr(K, "kernels", lambda: lib)
    monkeypatch.setattr(K, "_stream", lambda t: None)
    return seen


def test_rows_of_scores_keep_their_distance(monkeypatch):
    """A column transposed is one contiguous row of stride 1; a flat result is rows one after the other."""
    seen = _strides(monkeypatch)
    X, Q, Q1 = (types.SimpleNamespace(shape=(n, 128), is_cuda=True, device="cpu", data_ptr=lambda: 0, element_size=lambda: 2)
                for n in (40, 3, 1))
    for q, out, want in ((Q, None, 40), (Q, torch.empty(3, 52)[:, :40], 52), (Q, torch.empty(120), 40), (Q1, torch.empty(40, 1).t(), 40),
                         (Q1, torch.empty(2, 44)[1:, 4:], 44)):
        K.knn_scores(X, q, out=out)
        assert seen.pop() == want
    for scores, want in ((torch.empty(40, 1).t(), 40), (torch.empty(3, 52)[:, :40].contiguous(), 40), (torch.empty(3, 52), 52)):
        K._select(scores, 40, 5, None, None)
        assert seen.pop() == want


def test_segments_cover_the_scores_in_whole_blocks():
    """Every workgroup's share fits its registers' block maxima, and the last one holds as many as can be asked for."""
    lib = kernels()
    for n in [1, 15, 2048, 262_144, 262_145] + [(1 << 20) * a + d for a in (1, 2, 3, 7, 64, 2000) for d in (-1, 0, 1, 63, 64, 65, 500_000)]:
        seg, B = lib.cfc_topk_segment(n), lib.cfc_topk_block(n)
        parts = -(-n // seg)
        assert -(-seg // B) <= 16384 and B in (16, 32, 64)
        assert parts == 1 or seg % B == 0 and n - (parts - 1) * seg >= 2048
