"""Split counts of grids that do not fill the GPU (host only)."""


def test_small_grids_take_more_splits():
    from fused_turboquant import paged as P, v1 as V1
    assert P.default_splits(1, 8, 250, 32, 128) == 1      # the merge would cost more than it saves
    assert P.default_splits(1, 8, 1200, 32, 128) == 19    # one per 64 positions
    assert P.default_splits(1, 8, 5000, 32, 128) == 32    # one workgroup per CU
    assert P.default_splits(1, 2, 30000, 8, 128) == 64
    assert P.default_splits(4, 8, 1200, 32, 128) == 8
    assert P.default_splits(16, 8, 600, 32, 128) == 1 and P.default_splits(16, 8, 1200, 32, 128) == 2
    assert P.default_splits(0, 8, 100, 32, 128) == 1 and P.default_splits(1, 8, 0) == 1
    assert V1.default_splits(1, 8, 1000, 32, 128, 4, 4) == 1 and V1.default_splits(1, 8, 1200, 32, 128, 4, 4) == 19
    assert V1.default_splits(1, 8, 600, 32, 64, 4, 4) == 10  # the split-operand kernel, from 400 positions
    assert V1.default_splits(400, 8, 4000) == 1
