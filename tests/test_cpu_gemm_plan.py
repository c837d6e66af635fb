"""Plans of the tile GEMM (mc_model_debug_gemm_tiles_plan, host only) over all
row counts of the model's projections: a tile shape that takes the form, splits
that divide K, and a second launch only after whole tiles of the first."""
import ctypes as C

import pytest

from test_gpu_gemm_tiles import SHAPES

# name, N, K, form (0 plain, 1 swiglu, 2 rope), most splits
PROJECTIONS = [("qkv", 2560, 2048, 2, 1), ("o", 2048, 2048, 0, 8), ("down", 2048, 6144, 0, 8),
               ("down, full buffer", 2048, 6144, 0, 3), ("gate_up", 6144, 2048, 1, 1)]
ROPE = {0, 1, 2, 5, 6, 7, 8, 10, 11, 12, 13, 15, 16, 17}


@pytest.fixture(scope="module")
def plan(pkg):
    def get(M, N, K, form, low, high):
        p = (C.c_uint32 * 4)()
        r = pkg._native.lib().mc_model_debug_gemm_tiles_plan(M, N, K, form, low, high, p)
        return list(p) if r == 0 else r
    return get


@pytest.mark.parametrize("name,N,K,form,most", PROJECTIONS)
def test_every_row_count_has_a_sound_plan(plan, name, N, K, form, most):
    takes = [{i for i, s in enumerate(SHAPES) if s[2]}, {i for i, s in enumerate(SHAPES) if s[3]},
             ROPE][form]
    two = 0
    for M in [*range(1, 9000), *range(9001, 65536, 997), 65535]:
        rows0, shape0, shape1, splits = plan(M, N, K, form, 1, most)
        assert shape0 in takes and 1 <= splits <= most and K % (64 * splits) == 0, M
        assert 1 <= rows0 <= M, M
        if rows0 < M:
            two += 1
            assert splits == 1 and shape1 in takes and rows0 % SHAPES[shape0][0] == 0, M
    assert two > 0, name


def test_rejects_bad_arguments(plan):
    for a in ((0, 2048, 2048, 0, 1, 1), (8, 2080, 2048, 0, 1, 1), (8, 2048, 2048, 3, 1, 1),
              (8, 2048, 2048, 2, 1, 1), (8, 2048, 2048, 1, 1, 2), (8, 2048, 2048, 0, 3, 2),
              (8, 2048, 2048, 0, 1, 9), (8, 2048, 2048, 0, 3, 3), (65536, 2048, 2048, 0, 1, 1)):
        assert plan(*a) == 1, a
