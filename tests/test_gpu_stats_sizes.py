"""Statistics of passed profiles at the edges of the histogram's split over
workgroups, wavefronts and column blocks, with masked positions; against the
oracle (double precision)."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lq,lts", [(6, (6, 64, 257)), (17, (63, 65, 256, 600)), (130, (40, 255, 512, 513))])
def test_histogram_split(ctx, oracle, lq, lts):
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=2, sort_desc=0, seed=1200 + lq)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1210 + lt)
                            for lt in lts])
    q.field("aa")[lq // 2] = ord("X")
    db.field("aa")[::7] = ord("X")
    ctx.upload_queries(q)
    ctx.upload_db(db)
    res, plist, st = ctx.phase2_block(0, 0, db.nprof, -1.0, 1e9, 2)
    sc, _ = oracle.score_matrix(q, 0, db, 0, db.nprof)
    d = db.dists()
    qaa = q.field("aa")
    assert len(plist) > 0
    for j, k in enumerate(plist):
        lt = int(db.lens()[k])
        counts = np.zeros(641)
        taa = db.field("aa")[d[k]:d[k] + lt]
        sub = np.ascontiguousarray(sc[:, d[k]:d[k] + lt])
        oracle.L.orc_histogram(sub.ctypes.data, lt, 0, sub.shape[0], lt, qaa.ctypes.data, taa.ctypes.data,
                               counts.ctypes.data)
        par = oracle.stat_params(counts)
        sig = oracle.significance(2, lq, lt, float(q.field("eno")[0]), float(db.field("eno")[k]), 1e9,
                                  float(res["score"][k]), float(res["psts"][k]), par[4], par[5])
        np.testing.assert_allclose(st[j], np.concatenate([sig, par]), rtol=1e-9, atol=1e-12)
