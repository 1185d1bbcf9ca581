"""Key slices of a grouped decode step (ops.gqa.decode_slices): a rule of rows, heads and keys."""
import math

import pytest
import torch

from copilot_for_consensus_amd.models.decoder import kv_partitions
from copilot_for_consensus_amd.ops import gqa as A
from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.ops._native import kernels, kernels_available


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


@pytest.mark.parametrize("B,heads,kv,keys,least", [(5, 32, 8, 400, 3), (8, 32, 8, 400, 3), (8, 64, 8, 700, 3), (5, 32, 2, 700, 5), (24, 32, 2, 700, 2), (5, 8, 1, 1500, 8)])
def test_few_items_are_sliced(B, heads, kv, keys, least):
    """us in one slice (as many as the merge was thought to allow) and in these: 5 x 400 10.4 and 8.1, 8 x 400 10.6 and 8.8, 8 x 700 of 64
    heads 14.9 and 12.0, two key heads 11.2 and 9.2, 15.8 and 12.4, one 10.2 and 8.3."""
    assert kv_partitions(B, heads, kv, math.ceil(keys / 32)) >= least


@pytest.mark.parametrize("B,keys", [(24, 700), (24, 1500), (24, 2617), (32, 2617), (128, 2617)])
def test_a_full_round_is_not(B, keys):
    assert kv_partitions(B, 32, 8, math.ceil(keys / 32)) == 1


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
def test_paged_plan_knows_the_launch():
    lib = kernels()
    for wgs in (1, 32, 33, 64, 65, 256, 257, 4000):
        for blocks in (1, 2, 3, 8, 9, 40, 41, 300):
            for P in (1, 2, 3, 10, 64):
                waves, _, straight = K.paged_waves(wgs, blocks, P)
                assert lib.cfc_paged_waves(wgs, blocks, P, blocks) == (-waves if straight else waves)


@pytest.mark.parametrize("H,G,D,B,keys,P", [(16, 1, 32, 24, 2048, 8), (32, 8, 32, 8, 2048, 8), (32, 8, 32, 5, 1024, 4)])
def test_few_items_of_narrow_heads_are_sliced(H, G, D, B, keys, P):
    """us in one slice and in these: heads of 32 with one key head 13.4 and 8.4, with eight 13.3 and 10.1, 8.6 and 7.8."""
    assert A.decode_slices(B, H, G, D, keys, torch.bfloat16) == P


@pytest.mark.skipif(not kernels_available(), reason="the built library is missing")
def test_grouped_plan_knows_the_launch():
    lib = kernels()
    for D in (32, 64, 96, 128, 160, 192, 256):
        for wgs in (1, 64, 65, 256, 257, 512, 513, 5000):
            for tiles in (1, 2, 3, 4, 5, 8, 9, 33, 200):
                for pooled in (False, True):
                    for blocks in (2, 3, 4, 5, 200):
                        waves, _, straight = A.decode_waves(D, pooled, wgs, tiles, blocks)
                        assert lib.cfc_gqa_decode_waves(D, int(pooled), wgs, tiles, blocks) == (-waves if straight else waves)
