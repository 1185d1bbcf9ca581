"""GELU in the prompt GEMM's epilogue (pgemm.h, pg_gelu) over its whole argument range."""
import pytest
import torch

from copilot_for_consensus_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ("pp", "pps", "ring4"))
def test_gelu_of_every_bf16(variant):
    """All 65536 arguments, infinities and NaN among them, as a bias over a product of zeros.  A rounding to bf16 apart (8 bits:
    2^-8 at most), and the 4e-7 that the fp32 value is within: 1.5e-7 |x| / 2 of the approximation up to |x| = 4, and its
    last places."""
    bias = torch.arange(65536, device="cuda").to(torch.int32).to(torch.int16).view(torch.bfloat16)
    x, w = (torch.zeros(n, 64, device="cuda", dtype=torch.bfloat16) for n in (3, 65536))
    got = K.pgemm(x, w, "bias_gelu", bias=bias, variant=variant)
    v = bias.double()
    want = torch.where(v < 0, v * 0.5 * torch.special.erfc(v.abs() * 0.5 ** 0.5), v * (1.0 - 0.5 * torch.special.erfc(v * 0.5 ** 0.5)))
    want = torch.where(v == float("inf"), v, want)
    assert want[bias == float("-inf")].isnan().all() and want[bias.isnan()].isnan().all()
    for row in got.double():
        assert torch.equal(row.isnan(), want.isnan()) and torch.equal(row == float("inf"), want == float("inf"))
        ok = want.isfinite()
        assert ((row - want).abs()[ok] <= 2.0 ** -8 * want.abs()[ok] + 4e-7).all()
