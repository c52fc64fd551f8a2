"""The MAP stage with the backward pass beside the forward one (few pairs)
against the passes one after the other (more than 64 pairs): the same records,
for templates around the edges of phases and queries of one to six stripes."""
import numpy as np
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lq", [1, 31, 64, 65, 200, 330])
def test_few_pairs_equal_many(ctx, lq):
    lts = [1, 2, 7, 8, 31, 32, 33, 63, 64, 65, 96, 130, 257] + [20 + k for k in range(57)]
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1600 + lq)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1610 + k)
                            for k, lt in enumerate(lts)])
    ctx.upload_queries(q)
    ctx.upload_db(db)
    n = db.nprof
    prof = np.arange(n, dtype=np.int32)
    # pair E-values on both sides of the one from which the modular scores count
    epa = np.where(prof % 2 == 0, -30.0, 5.0).astype(np.float32)
    many = ctx.map_block(0, 0, n, prof, epa)
    for sub in (prof[:1], prof[:13], prof[6:]):
        few = ctx.map_block(0, 0, n, sub, epa[sub])
        for f in few.dtype.names:
            a, b = few[f], many[f][sub]
            assert a.tobytes() == b.tobytes(), (f, np.flatnonzero(a != b)[:5])
