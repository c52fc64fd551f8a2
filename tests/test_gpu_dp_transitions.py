"""The phase-1 DP where transitions are large positive numbers, which no
log-probability is: from about 1000 up they would carry a path through the 32
columns before the profile to a positive match state, a cell outside the
matrix.  Such sets take the kernel form that tests for those columns; those
below its bound do not need the test.  Against the oracle, bit for bit."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [200.0, 256.0, 257.0, 1060.0, 1500.0, 5e4])
def test_maximum_lies_within_the_matrix(ctx, oracle, top):
    q = cother_amd.synth(1, 2, lmin=100, lmax=100, dist_mode=2, sort_desc=0, seed=1801)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1802 + lt)
                            for lt in (5, 33, 64, 120)])
    # match to delete, delete to delete and delete to match of the query's first rows
    q.field("trn")[[2, 5, 6], :40] = top
    ctx.upload_queries(q)
    ctx.upload_db(db)
    res, bt = ctx.phase1_block(0, 0, db.nprof, 0.0, want_btck=True)
    lens = db.lens()
    assert ((res["maxxy"] >> 16) < lens).all() and ((res["maxxy"] & 0xffff) < 100).all()
    sc, _ = oracle.score_matrix(q, 0, db, 0, db.nprof)
    ores, obt = oracle.phase1(q, 0, db, 0, db.nprof, sc, 0.0)
    assert (bt == obt).all()
    for f in ("maxsc", "maxxy", "passed", "psts", "beg", "score"):
        assert (res[f] == ores[f]).all(), f
    # the pass without traceback: a database of more profiles than compute units
    many = cother_amd.concat([db] + [cother_amd.synth(300, 0, lmin=5, lmax=40, dist_mode=2, seed=1850)])
    ctx.upload_db(many)
    hits, _, _ = ctx.search(eval=1e4, do_map=False)
    hits = hits[hits["profile"] < db.nprof]
    assert len(hits) > 0
    for h in hits:
        assert h["end"] == ores["maxxy"][h["profile"]] and h["score"] == ores["score"][h["profile"]]
