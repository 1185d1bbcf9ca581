"""Several products of a prompt's rows in one launch (Projection's runs, mgemm_joint): against each product on its own and 64
bits."""
import pytest
import torch

from copilot_for_consensus_amd.models.projection import JointProjection
from copilot_for_consensus_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


def _close(got, x, w):
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # sums of K products in fp32, in any order; activations are rounded to bf16 once
    tol = x.shape[1] * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if got.dtype == torch.bfloat16 else 0)
    assert ((got.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("M", (1, 4, 5, 16, 128, 129, 257, 700))
@pytest.mark.parametrize("inputs, slabs", [((0, 0, 0, 0), ()), ((0, 1, 2, 3), (3,)), ((0, 1, 1, 1), (2,)), ((2, 2, 0, 1), (0, 3))])
@pytest.mark.parametrize("plan", (None, 128, 192, 256))
def test_parts_are_the_products(monkeypatch, M, inputs, slabs, plan):
    """Sizes that are no whole tiles, parts in fp32 between the others, every height of tile, and the chosen plan (None)."""
    g = torch.Generator("cuda").manual_seed(M)
    sizes, Kd = (1280, 2560, 1088, 64), 320
    ws = [(torch.randn(n, Kd, device="cuda", generator=g) * 0.1).bfloat16() for n in sizes]
    j = JointProjection(list(zip(ws, inputs)))
    if plan:
        monkeypatch.setattr(K, "joint_plan", lambda M, sizes, Kd, one: -1 if one else plan)
    acts = torch.randn(4, M, Kd, device="cuda", generator=g).bfloat16()
    for i, c in enumerate(j.prompt(acts, slabs)):
        assert c.n == sizes[i] and c.slabs == (i in slabs)
        got = c.t.sum(0) if c.slabs else c.t
        _close(got[:, c.c0:c.c0 + c.n], acts[inputs[i]], ws[i])


@pytest.mark.parametrize("bm", (128, 160, 192, 224, 256))
@pytest.mark.parametrize("M", (1, 127, 128, 161, 513))
def test_each_tile_multiplies_its_input(M, bm):
    g = torch.Generator("cuda").manual_seed(M + bm)
    N, Kd = 768, 192
    w = (torch.randn(N, Kd, device="cuda", generator=g) * 0.1).bfloat16()
    x = torch.randn(3, M, Kd, device="cuda", generator=g).bfloat16()
    in_of = torch.tensor([2, 0, 0, 1, 2, 1], dtype=torch.int32, device="cuda")
    out = K.mgemm_joint(x, K.pack_dgemm_weight(w, bn=128), in_of, bm)
    for t, i in enumerate(in_of.tolist()):
        _close(out[:, 128 * t:128 * (t + 1)], x[i], w[128 * t:128 * (t + 1)])
