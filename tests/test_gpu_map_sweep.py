"""The MAP stage's sweeps at the edges of their parts: stripes of 64 query
rows, phases of 32 columns, the wavefronts of one pair, boundary rows in LDS
and in global memory, with and without the modular scores, and sets whose
values could give a NaN (the reference's forms of the sums of exponentials);
against the oracle, bit for bit."""
import numpy as np
import pytest

import cother_amd
from tests.test_gpu_dp_sweep import _sets

pytestmark = pytest.mark.gpu

FIELDS = ("maxsc", "end", "beg", "idnts", "psts", "ngaps", "alnlen", "logz", "maxlog")


def _equals_oracle(ctx, oracle, q, db):
    ctx.upload_queries(q)
    ctx.upload_db(db)
    prof = np.arange(db.nprof, dtype=np.int32)
    sc, md = oracle.score_matrix(q, 0, db, 0, db.nprof)
    d = db.dists()
    # log pair E-values: modular scores in full, in part, not at all
    for shift in (0, 1, 2):
        epa = np.array([(-60.0, -23.5, 5.0)[(k + shift) % 3] for k in prof], np.float32)
        res = ctx.map_block(0, 0, db.nprof, prof, epa)
        for j in prof:
            want = oracle.map_profile(q, 0, db, int(j), sc, md, int(d[j] - d[0]), float(epa[j]))
            for f in FIELDS:
                assert np.asarray(res[j][f]).tobytes() == np.asarray(want[f]).tobytes(), (j, f, res[j][f], want[f])


@pytest.mark.parametrize("lq", [1, 31, 64, 65, 130, 577])
def test_edges_of_stripes_and_phases(ctx, oracle, lq):
    q, db = _sets(lq, (1, 2, 8, 31, 32, 33, 64, 95, 96, 97, 160, 301), 1100 + lq)
    _equals_oracle(ctx, oracle, q, db)


@pytest.mark.parametrize("lt", [6000, 6001])
def test_rows_in_lds_and_in_global_memory(ctx, oracle, lt):
    q, db = _sets(600, (lt, 70, 33), 1150)
    _equals_oracle(ctx, oracle, q, db)


def test_sets_outside_the_finite_ranges(ctx, oracle):
    q, db = _sets(100, (120, 64, 40), 1170)
    db.field("trg")[3, 50] = 2.0
    _equals_oracle(ctx, oracle, q, db)
