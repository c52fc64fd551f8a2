"""The distance-match kernel at the edges of its tiles: 32, 16 or 8 query rows
by 8, 16 or 32 template columns, wavefronts of fewer rows in the last tile,
columns past the last template, and cells without lists beside cells with
them -- bit for bit against the oracle."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lq,lts", [(1, (1,)), (2, (33,)), (3, (31, 2)), (8, (32,)), (9, (15, 2)), (16, (16,)),
                                    (17, (7, 1)), (32, (8,)), (33, (40, 33)), (41, (65,)), (70, (9, 100))])
@pytest.mark.parametrize("mixed", [False, True])
def test_tiles(ctx, oracle, lq, lts, mixed):
    q = cother_amd.synth(1, 2, lmin=200, lmax=200, dist_mode=0, sort_desc=0, seed=1500)
    # rows of a longer profile, whose lists are full
    part = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1501 + lq)
    part.field("dd")[...] = q.field("dd")[60:60 + lq]
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=1, sort_desc=0, seed=1510 + lt)
                            for lt in lts])
    big = cother_amd.synth(1, 2, lmin=300, lmax=300, dist_mode=1, sort_desc=0, seed=1502)
    db.field("dd")[...] = big.field("dd")[80:80 + db.npos]
    if mixed:
        part.field("dd")[1::3, 0] = 5
        db.field("dd")[::4, 0] = np.resize([0, 5, 6, 50], len(db.field("dd")[::4]))
    ctx.upload_queries(part)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof)
    osc, omd = oracle.score_matrix(part, 0, db, 0, db.nprof)
    assert (sc.view(np.int32) == osc.view(np.int32)).all()
    assert (md.view(np.int32) == omd.view(np.int32)).all()
