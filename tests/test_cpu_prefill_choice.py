"""Workgroup shape and key splits chosen for a prefill attention launch
(mc_kv_debug_prefill_choice, host only), where the rows, the splits asked for
and the prefix make another choice the faster one."""
import pytest

ROWS32, ROWS16, HALVES, SETS8, SETS4 = range(5)


@pytest.mark.parametrize("tokens,splits,want", [
    (1, 8, (SETS4, 8)), (64, 8, (SETS4, 8)), (65, 8, (SETS8, 8)), (160, 8, (SETS8, 6)), (128, 8, (SETS8, 8)),
    (200, 8, (SETS8, 5)), (201, 8, (ROWS16, 8)), (320, 8, (ROWS16, 8)), (384, 8, (ROWS16, 8)),
    (256, 4, (SETS8, 4)), (384, 2, (SETS8, 2)), (385, 2, (ROWS16, 2)), (777, 5, (ROWS16, 5))])
def test_splits_with_an_unknown_prefix(kvm, tokens, splits, want):
    """Key sets only where most of the splits asked for fit on the CUs: each of
    their workgroups reads the whole prefix, which may be long."""
    assert kvm.debug_prefill_choice(tokens, splits) == want


@pytest.mark.parametrize("tokens,keys,want", [
    (256, 4800, (SETS8, 4)), (256, 4801, (ROWS16, 8)), (300, 16300, (ROWS16, 8)),
    (320, 3600, (SETS8, 3)), (320, 3601, (ROWS16, 8)), (384, 2400, (SETS8, 2)),
    (384, 2401, (ROWS16, 8)), (384, 130000, (ROWS16, 8)), (100, 130000, (SETS8, 8))])
def test_splits_with_a_known_prefix(kvm, tokens, keys, want):
    """201 to 384 rows: key sets up to a prefix of 1200 keys per split."""
    assert kvm.debug_prefill_choice(tokens, 8, keys) == want


@pytest.mark.parametrize("tokens,want", [(512, SETS4), (513, SETS8), (1024, SETS8),
                                         (1025, HALVES), (4096, HALVES), (4097, ROWS16),
                                         (8192, ROWS32)])
def test_without_splits(kvm, tokens, want):
    assert kvm.debug_prefill_choice(tokens, 1) == (want, 1)
