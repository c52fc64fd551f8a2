"""The phase-1 DP's sweep at the edges of its parts: stripes of 64 query
rows, phases of 32 columns, the wavefronts of one pair, boundary rows in LDS
and in global memory, and sets whose values could give a NaN (the reference's
select instead of the hardware's maximum); against the oracle, bit for bit."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


def _sets(lq, lts, seed):
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=2, sort_desc=0, seed=seed)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=seed + 1 + k)
                            for k, lt in enumerate(lts)])
    return q, db


def _equals_oracle(ctx, oracle, q, db, search=True):
    ctx.upload_queries(q)
    ctx.upload_db(db)
    res, bt = ctx.phase1_block(0, 0, db.nprof, 0.0, want_btck=True)
    sc, _ = oracle.score_matrix(q, 0, db, 0, db.nprof)
    ores, obt = oracle.phase1(q, 0, db, 0, db.nprof, sc, 0.0)
    assert (bt == obt).all(), np.argwhere(bt != obt)[:5].tolist()
    for f in ("maxsc", "maxxy", "passed", "psts", "beg", "score"):
        assert np.array_equal(res[f], ores[f], equal_nan=True), f
    if not search:
        return
    # the first pass of a search keeps no traceback
    hits, _, _ = ctx.search(eval=1e3)
    want = oracle.search_query(q, 0, db, eval_=1e3)
    assert len(hits) == len(want)
    for f in ("profile", "score", "beg", "end"):
        assert (hits[f] == want[f]).all(), f


@pytest.mark.parametrize("lq", [1, 31, 64, 65, 130, 520, 577])
def test_edges_of_stripes_and_phases(ctx, oracle, lq):
    q, db = _sets(lq, (1, 2, 8, 31, 32, 33, 64, 95, 96, 97, 160, 301), 900 + lq)
    _equals_oracle(ctx, oracle, q, db)


@pytest.mark.parametrize("lt", [4096, 4097])
def test_rows_in_lds_and_in_global_memory(ctx, oracle, lt):
    q, db = _sets(600, (lt, 70, 33), 950)
    _equals_oracle(ctx, oracle, q, db)


@pytest.mark.parametrize("kind", ["large", "nan"])
def test_sets_outside_the_finite_ranges(ctx, oracle, kind):
    q, db = _sets(100, (120, 64, 40), 970)
    if kind == "large":
        db.field("trg")[3, 50] = 2.0
    else:
        # no background and no frequency on either side: 0 / 0 in every cell of one position
        q.field("bkg")[:, 4] = 0.0
        db.field("bkg")[1, 4] = 0.0
        q.field("trg")[4, 60] = 0.0
        sc, _ = oracle.score_matrix(q, 0, db, 0, db.nprof)
        assert np.isnan(sc).any()
    # (the statistics stage has no defined histogram bin for a NaN score)
    _equals_oracle(ctx, oracle, q, db, search=kind == "large")


def test_few_pairs_and_long_profiles_in_a_batch(ctx):
    """fewer pairs than fill the chip (one wavefront per stripe), and a
    database whose rows are in global memory, as the per-query search"""
    q = cother_amd.synth(3, 0, lmin=150, lmax=300, dist_mode=2, sort_desc=0, seed=981)
    for longest in (300, 4500):
        db = cother_amd.concat([cother_amd.subset(q, 0, 2),
                                cother_amd.synth(1, 2, lmin=longest, lmax=longest, dist_mode=2, seed=982),
                                cother_amd.synth(30, 0, lmin=20, lmax=260, dist_mode=2, seed=983)])
        ctx.upload_queries(q)
        ctx.upload_db(db)
        a, na, _ = ctx.search(eval=1e3)
        b, nb, _ = ctx.search(eval=1e3, batch=True)
        assert len(a) > 2 and (na == nb).all()
        for f in ("query", "profile", "score", "beg", "end", "alnlen", "mapscore"):
            assert (a[f] == b[f]).all(), (longest, f)
