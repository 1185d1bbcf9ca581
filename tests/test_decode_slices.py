"""Key slices of a grouped decode step (ops.gqa.decode_slices): a rule of rows, heads and keys."""
import math

import pytest
import torch

from copilot_for_consensus_amd.ops import gqa as A


@pytest.mark.parametrize("visible", (255, 512, 1536, 1537, 2048, 6000, 100_000))
def test_long_rows_of_many_items_are_sliced(visible):
    """From 384 items on rows of more than 1536 keys get 1024 slices in all: a longest row is never one workgroup's work
    unless there are a thousand others."""
    for B in (48, 56, 64, 96, 127, 128, 200):
        items = 8 * B
        P = A.decode_slices(B, 32, 8, 128, visible, torch.bfloat16)
        assert P == (1 if visible <= 1536 else min(math.ceil(1024 / items), visible // 256))
    assert A.decode_slices(1, 32, 8, 128, visible, torch.bfloat16) == max(1, min(96, visible // 256, A.MAX_PARTITIONS))
    assert A.decode_slices(48, 32, 8, 128, visible, torch.float32) == max(1, min(math.ceil(1024 / (48 * math.ceil(32 / A.ANY_ROWS))), visible // 256))


@pytest.mark.parametrize("B,H,G,visible", [(2, 4, 1, 1_000_000), (2, 32, 8, 100_000), (3, 8, 1, 40_000), (47, 32, 8, 4000), (5, 32, 8, 1)])
def test_slices_are_no_more_than_the_merge_takes(B, H, G, visible):
    for D in (32, 128, 256):
        assert 1 <= A.decode_slices(B, H, G, D, visible, torch.bfloat16) <= min(A.MAX_PARTITIONS, max(1, math.ceil(visible / 256)))


@pytest.mark.parametrize("B,heads,RS,keys,plan", [(64, 128, 512, 4000, (32, 1)), (24, 128, 512, 4000, (32, 2)), (4, 32, 512, 200, (16, 4)), (8, 32, 512, 1000, (16, 8))])
def test_latent_plans_follow_the_measured_best(B, heads, RS, keys, plan):
    """us of these plans and of others: 133 and, in two slices of 64 rows, which spill at this rank, 202; 79 and 93 in five; 10.0 and in one
    slice 11.0; 14.6 and in sixteen 16.0."""
    from copilot_for_consensus_amd.ops import latent as L
    assert L.decode_plan(B, heads, RS, keys) == plan
