"""How decode attention shares its work out (host rules)."""

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
