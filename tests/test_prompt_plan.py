"""Where the plan of a prompt product (mgemm.hip, cfc_prompt_plan) draws its lines."""
import pytest

from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops._native import kernels_available

pytestmark = pytest.mark.skipif(not kernels_available(), reason="the built library is missing")


@pytest.mark.parametrize("N, Kd, fewest, most", [(512, 4096, 15400, 16384), (1024, 4096, 7700, 8192), (512, 1024, 15700, 16384), (1024, 1024, 7850, 8192),
                                                 (768, 3072, 10300, 10700)])
def test_many_rows_of_few_columns_stay_on_the_large_tiles(N, Kd, fewest, most):
    """256-row tiles of a nearly full round, whose X goes to every L2: 8 to 25 % slower than pgemm's."""
    for M in range(fewest, most, 61):
        assert all(K.prompt_plan(M, N, Kd, kind) is None for kind in ("act", "whole"))


@pytest.mark.parametrize("N, Kd", [(256, 4096), (512, 4096), (1024, 4096), (1536, 4096), (2048, 4096), (512, 1024), (1024, 1024), (2048, 2048)])
def test_slices_of_an_activation_fill_their_ring(N, Kd):
    """No K slice of 8 stages or fewer where a product runs here as a whole."""
    for M in range(641, 5000, 53):
        plan = K.prompt_plan(M, N, Kd)
        if plan and plan[0] == 0:
            assert plan[2] == 1 or Kd // 64 // plan[2] > 8, (M, plan)
    assert K.prompt_plan(1507, 512, 1024)[2] == 1 and K.prompt_plan(339, 1536, 4096)[2] == 4


def test_products_with_few_large_tiles_are_planned_as_before():
    """Fewer tiles than pgemm is given: nothing else would take them but the decode GEMM."""
    assert K.prompt_plan(12029, 512, 1024, "whole") == (0, 224, 1) and K.prompt_plan(6000, 1024, 14336) is not None


def test_largest_products_are_planned():
    """More tiles than 32 bits count."""
    assert K.prompt_plan(2 ** 24, 2 ** 24, 64) is None and K.prompt_plan(2 ** 24, 2 ** 24, 64, "slabs") is None
