"""Split counts of grids that do not fill the GPU (host only)."""


def test_small_grids_take_more_splits():
    from fused_turboquant import paged as P, v1 as V1
    # below 2048 positions the one-launch form: a merge would add a launch to steps the host bounds
    assert P.default_splits(1, 8, 250, 32, 128) == 1 and P.default_splits(1, 8, 2047, 32, 128) == 1
    assert P.default_splits(1, 8, 2048, 32, 128) == 32    # one per 64 positions, one workgroup per CU
    assert P.default_splits(1, 2, 30000, 8, 128) == 64
    assert P.default_splits(4, 8, 3000, 32, 128) == 8
    assert P.default_splits(16, 8, 1200, 32, 128) == 1 and P.default_splits(16, 8, 2400, 32, 128) == 2
    assert P.default_splits(0, 8, 100, 32, 128) == 1 and P.default_splits(1, 8, 0) == 1
    assert V1.default_splits(1, 8, 2000, 32, 128, 4, 4) == 1 and V1.default_splits(1, 8, 2100, 32, 128, 4, 4) == 32
    assert V1.default_splits(1, 8, 2000, 32, 64, 4, 4) == 1 and V1.default_splits(1, 8, 2100, 32, 64, 4, 4) == 32
    assert V1.default_splits(400, 8, 4000) == 1
