"""The distance-match kernel's launches over many columns: a grid dimension of
2^32 work-items or more is refused, and the entry points take blocks and
databases of up to 2^30 columns."""
import ctypes

import numpy as np
import pytest

import cother_amd


@pytest.mark.parametrize("ncols", [1, 7, 8, 9, (1 << 23) - 1, 1 << 23, (1 << 23) + 1, 1 << 27, (1 << 27) + 1, 1 << 30])
def test_grids_stay_within_the_limit(ncols):
    out = (ctypes.c_uint64 * 2)()
    fn = cother_amd.lib().cth_selftest_ddms_launches
    fn.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_uint64)]
    fn.restype = None
    fn(ncols, out)
    assert out[0] < 1 << 32
    assert out[1] == ncols


@pytest.mark.gpu
def test_columns_of_a_second_launch(ctx):
    """more columns than one launch takes: the second launch's equal those of
    a block of its own, and the first's last ones too"""
    q = cother_amd.synth(1, 2, lmin=6, lmax=6, dist_mode=0, sort_desc=0, seed=2001)
    q.field("dd")[:, 0] = 8  # lists long enough for a term
    one = cother_amd.synth(1, 2, lmin=1000, lmax=1000, dist_mode=1, sort_desc=0, seed=2002)
    last = cother_amd.synth(4, 2, lmin=500, lmax=500, dist_mode=1, sort_desc=0, seed=2003)
    n = (1 << 23) // 1000
    db = cother_amd.concat([cother_amd.subset_list(one, [0] * n), last])
    assert db.npos > 1 << 23 and n * 1000 <= 1 << 23
    ctx.upload_queries(q)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof)
    a = n - 1
    sc1, md1 = ctx.score_block(0, a, db.nprof)
    for got, want in ((sc, sc1), (md, md1)):
        assert (got[:, a * 1000:].view(np.int32) == want.view(np.int32)).all()
    # (some of those cells have a term)
    plain = cother_amd.concat([last])
    plain.field("dd")[:, 0] = 0
    ctx.upload_db(plain)
    assert (ctx.score_block(0, 0, 4)[0] != sc[:, n * 1000:]).any()
