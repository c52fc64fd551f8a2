"""The distance-match scan where its steps are split: the cells that every
lane of a wavefront has are scanned without a test of the lane's end, the rest
with one, and lanes whose lists are too short take no part."""
import numpy as np
import pytest

import cother_amd
from tests import _ddms_lists as dl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qlens,tlens", [((6,), (6,)), ((99,), (99,)), ((98, 99), (6, 7)), ((6, 7), (5, 99)),
                                         ((9, 12), (0, 8, 13)), ((16, 17), (15, 16, 17, 99)), ((97, 5), (0,))])
def test_list_lengths_of_a_wavefront(ctx, oracle, qlens, tlens):
    q = cother_amd.synth(1, 0, lmin=21, lmax=21, dist_mode=0, sort_desc=0, seed=1401)
    db = cother_amd.synth(3, 0, lmin=30, lmax=70, dist_mode=1, sort_desc=0, seed=1402)
    rng = np.random.default_rng(1403 + sum(qlens) + 100 * sum(tlens))
    dl.fill(q, rng, lengths=list(qlens))
    dl.fill(db, rng, lengths=list(tlens))
    # the query's own lists among the templates: segments over whole diagonals
    for n in set(qlens) & set(tlens):
        own = q.field("dd")[q.field("dd")[:, 0] == n]
        db.field("dd")[np.flatnonzero(db.field("dd")[:, 0] == n)[:len(own)]] = own[:np.sum(db.field("dd")[:, 0] == n)]
    ctx.upload_queries(q)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof)
    osc, omd = oracle.score_matrix(q, 0, db, 0, db.nprof)
    assert (sc.view(np.int32) == osc.view(np.int32)).all()
    assert (md.view(np.int32) == omd.view(np.int32)).all()
