"""Phase 1's traceback bytes on their way back: the rows' padding is taken out
on the device, by a grid that stays within the limit of 2^32 work-items for any
block and takes further bytes in turns."""
import ctypes

import numpy as np
import pytest

import cother_amd


@pytest.mark.parametrize("n", [1, 4, 1024, 1 << 22, (1 << 34) - 1, 1 << 34, 50000 << 30])
def test_grid_stays_within_the_limit(n):
    fn = cother_amd.lib().cth_selftest_pack_grid
    fn.argtypes = [ctypes.c_uint64]
    fn.restype = ctypes.c_uint64
    assert 0 < fn(n) < 1 << 32


@pytest.mark.gpu
@pytest.mark.parametrize("lq,nt,lt", [(1, 1, 1), (3, 1, 65), (150, 301, 99), (129, 333, 127)])
def test_blocks_equal_their_parts(ctx, lq, nt, lt):
    """under and over one turn of the grid (4 MB), rows of odd lengths"""
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=2, sort_desc=0, seed=2101)
    db = cother_amd.synth(nt, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=2102)
    ctx.upload_queries(q)
    ctx.upload_db(db)
    res, bt = ctx.phase1_block(0, 0, nt, 1.0, want_btck=True)
    parts = [ctx.phase1_block(0, a, min(nt, a + 50), 1.0, want_btck=True)[1] for a in range(0, nt, 50)]
    assert (bt == np.concatenate(parts, axis=1)).all()
