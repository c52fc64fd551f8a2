"""Alignment rows of a search whose chunk holds so many long profiles that
rows for all of them would be hundreds of megabytes: the hits' rows equal those
of the search in fixed memory, whose stages the host chooses."""
import pytest

import cother_amd

pytestmark = pytest.mark.gpu


def test_rows_of_a_large_chunk(ctx):
    q = cother_amd.synth(1, 2, lmin=1000, lmax=1000, dist_mode=2, sort_desc=0, seed=2301)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=2500, lmax=2500, dist_mode=2, seed=2302), q,
                            cother_amd.synth(23000, 1, 210.0, 0.35, 30, 900, dist_mode=2, sort_desc=1, seed=2303)])
    assert db.nprof * 5 * 3500 > 256 << 20
    ctx.upload_queries(q)
    ctx.upload_db(db)
    a, na, sa, ra = ctx.search(eval=10.0, alignments=True)
    assert sa.nchunks == 1 and len(a) > 0
    b, nb, _, rb = ctx.search(eval=10.0, alignments=True, noalloc=True)
    assert (na == nb).all() and ra == rb
    for f in a.dtype.names:
        if f not in ("reserved", "alnoff"):
            assert a[f].tobytes() == b[f].tobytes(), f
