"""Phase 1 with different numbers of wavefronts per pair: the rule takes more of
them for few or long profiles and fewer for many short ones, and the records and
traceback bytes do not depend on it -- against the oracle on a sample, and
the same profiles alone and among many."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lq,nt", [(65, 700), (330, 900), (580, 600)])
def test_few_and_many(ctx, oracle, lq, nt):
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1700 + lq)
    few = cother_amd.synth(6, 0, lmin=20, lmax=400, dist_mode=2, sort_desc=1, seed=1701)
    db = cother_amd.concat([few, cother_amd.synth(nt, 0, lmin=20, lmax=60, dist_mode=2, sort_desc=1, seed=1702)])
    ctx.upload_queries(q)
    ctx.upload_db(db)
    n, m = few.npos, few.nprof
    res, bt = ctx.phase1_block(0, 0, db.nprof, 1.0, want_btck=True)
    one, bt1 = ctx.phase1_block(0, 0, m, 1.0, want_btck=True)
    for f in one.dtype.names:
        assert one[f].tobytes() == res[f][:m].tobytes(), f
    assert (bt1 == bt[:, :n]).all()
    sc, _ = oracle.score_matrix(q, 0, few, 0, m)
    ores, obt = oracle.phase1(q, 0, few, 0, m, sc, 1.0)
    assert (bt1 == obt).all()
    for f in ("maxsc", "maxxy", "passed", "psts", "beg"):
        assert (one[f] == ores[f]).all(), f
