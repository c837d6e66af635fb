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
    (320, 3600, (SETS8, 3)), (320, 3601, (ROWS16, 7)), (384, 2400, (SETS8, 2)),
    (384, 2401, (ROWS16, 4)), (384, 130000, (ROWS16, 8)), (100, 130000, (SETS8, 8))])
def test_splits_with_a_known_prefix(kvm, tokens, keys, want):
    """201 to 384 rows: key sets up to 1200 keys per split that fits; splits of
    at least 512 keys."""
    assert kvm.debug_prefill_choice(tokens, 8, keys) == want


@pytest.mark.parametrize("tokens,want", [(512, SETS4), (513, SETS8), (1024, SETS8),
                                         (1025, HALVES), (4096, HALVES), (4097, ROWS16),
                                         (8192, ROWS32)])
def test_without_splits(kvm, tokens, want):
    assert kvm.debug_prefill_choice(tokens, 1) == (want, 1)


@pytest.mark.parametrize("tokens,base,want", [
    (300, 300, (SETS4, 1)), (512, 1024, (SETS4, 1)), (777, 0, (SETS8, 1)),
    (777, 1554, (SETS8, 1)), (777, 3001, (ROWS16, 5)), (1024, 2048, (SETS8, 1)),
    (1024, 2051, (ROWS16, 4)), (40, 400, (SETS4, 1)),
    # two rounds of key-set workgroups: short prefixes only
    (1100, 1100, (SETS8, 1)), (1100, 1101, (ROWS16, 3)), (1100, 2200, (ROWS16, 3)),
    (1300, 2500, (ROWS16, 3)), (1500, 0, (SETS8, 1)), (1500, 1500, (HALVES, 1)),
    (1500, 2999, (HALVES, 1)), (1500, 3100, (ROWS16, 2)), (2048, 0, (SETS8, 1)),
    (2048, 2048, (HALVES, 1)), (2047, 8192, (ROWS16, 2)), (2048, 8192, (HALVES, 1)), (2049, 0, (HALVES, 1)),
    (8448, 0, (ROWS32, 1))])
def test_session_chunks(kvm, tokens, base, want):
    """A session asks for the reference's split count and knows the prefix: no
    splits only on a shape that is the faster one without, else all of them."""
    splits = kvm.prefill_flash_split_kv(tokens)
    assert kvm.debug_prefill_choice(tokens, splits, base + tokens) == want
