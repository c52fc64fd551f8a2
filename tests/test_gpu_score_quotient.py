"""The plain score kernel's log-odds quotients where a query row has a
frequency outside the ranges that the quotient correction admits, so that its
tile has to divide: the bad row among those of a tile, the last block of
columns full, half full and with one column.  An infinite frequency and
frequencies whose products are near the smallest normal number, for both of
which the correction gives other numbers than the division; against the oracle,
bit for bit."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["infinite", "tiny"])
@pytest.mark.parametrize("cols", [(1,), (64,), (65,), (96,), (64, 64, 3)])
@pytest.mark.parametrize("row", [0, 5, 15, 21, 69])
def test_rows_outside_the_ranges_are_divided(ctx, oracle, kind, cols, row):
    q = cother_amd.synth(1, 2, lmin=70, lmax=70, dist_mode=2, sort_desc=0, seed=1901)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1902 + k)
                            for k, lt in enumerate(cols)])
    # (no zero frequencies: infinity times zero has no defined bits)
    t = db.field("trg")
    t[...] = np.maximum(t, np.float32(1e-3))
    f = q.field("trg")
    if kind == "infinite":
        f[3, row] = np.inf
    else:
        f[:, row] = np.float32(1e-38) * (1 + np.arange(20, dtype=np.float32) / 7)
    ctx.upload_queries(q)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof)
    osc, omd = oracle.score_matrix(q, 0, db, 0, db.nprof)
    assert (sc.view(np.int32) == osc.view(np.int32)).all(), np.argwhere(sc != osc)[:4].tolist()
    assert (md.view(np.int32) == omd.view(np.int32)).all()
