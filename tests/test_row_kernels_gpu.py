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
