"""Device memory of a search: the score, traceback and posterior buffers are
what mem_budget counts (13 bytes a cell with MAP); what comes beside them is in
proportion to the profiles' records and to the hits, not to what every profile
would need as a hit."""
import numpy as np
import pytest
import torch

import cother_amd

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _taken(q, db, **kw):
    """bytes that the first search of a new context takes, and its hits (a context
    before it has had the runtime reserve what it keeps: registers spilled to
    memory, code)"""
    for _ in range(2):
        c = cother_amd.Context(0)
        try:
            c.upload_queries(q)
            c.upload_db(db)
            torch.cuda.synchronize()
            free0 = torch.cuda.mem_get_info(0)[0]
            got = c.search(**kw)
            taken = free0 - torch.cuda.mem_get_info(0)[0]
        finally:
            c.close()
    return taken, got


def _sets(lq, nt, tmax, seed):
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=2, sort_desc=0, seed=seed)
    db = cother_amd.concat([q, cother_amd.synth(nt, 0, 220.0, 0.35, 30, tmax, dist_mode=2, sort_desc=1, seed=seed + 1),
                            cother_amd.synth(1, 2, lmin=tmax, lmax=tmax, dist_mode=2, seed=seed + 2)])
    return q, db


@pytest.mark.parametrize("rows", [False, True])
def test_within_a_small_budget(rows):
    q, db = _sets(250, 1500, 1500, 2201)
    budget = 128 * MB
    taken, got = _taken(q, db, mem_budget=budget, alignments=rows)
    assert len(got[0]) > 0
    # (an allocation keeps an eighth for growth)
    assert taken < budget * 9 // 8 + 24 * MB, taken / MB


@pytest.mark.parametrize("rows", [False, True])
def test_beside_large_buffers(rows):
    q, db = _sets(100, 6000, 1500, 2211)
    taken, got = _taken(q, db, alignments=rows)
    assert len(got[0]) > 0
    cells = 100 * ((db.npos + 63) // 64 * 64)
    assert taken < 13 * cells * 9 // 8 + 24 * MB, (taken / MB, 13 * cells / MB)


@pytest.mark.parametrize("nq,lq,nt,tmax", [(4, 60, 600, 5000), (2, 250, 20, 1500)])
def test_batch_beside_its_buffers(nq, lq, nt, tmax):
    """boundary rows in global memory (templates over 4096 positions), and the
    backward values of hits where the pairs are few"""
    q = cother_amd.synth(nq, 2, lmin=lq, lmax=lq, dist_mode=2, sort_desc=0, seed=2231)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=tmax, lmax=tmax, dist_mode=2, seed=2232),
                            cother_amd.subset(q, 0, 1),
                            cother_amd.synth(nt, 2, lmin=60, lmax=60, dist_mode=2, seed=2233)])
    taken, got = _taken(q, db, batch=True)
    assert len(got[0]) > 0
    cells = nq * lq * ((db.npos + 63) // 64 * 64)
    # the rows of one workgroup per compute unit: 28 bytes a position
    rows = 256 * 28 * tmax if tmax > 4096 else 0
    assert taken < (13 * cells + rows) * 9 // 8 + 24 * MB, (taken / MB, 13 * cells / MB)


@pytest.mark.parametrize("rows", [False, True])
def test_hits_few_many_and_none(ctx, rows):
    """the MAP stage sized before and after its hits are known, with as many
    as the list comes back with at once, more, and none: as the batched search"""
    q = cother_amd.synth(2, 0, lmin=60, lmax=90, dist_mode=2, sort_desc=0, seed=2221)
    for nt, ev in ((40, 1e3), (1500, 1e-30), (1500, 1e3), (1500, 1e6)):
        db = cother_amd.concat([cother_amd.subset(q, 0, 1),
                                cother_amd.synth(nt, 0, lmin=30, lmax=700, dist_mode=2, sort_desc=1, seed=2222 + nt)])
        ctx.upload_queries(q)
        ctx.upload_db(db)
        a = ctx.search(eval=ev, alignments=rows)
        b = ctx.search(eval=ev, alignments=rows, batch=True)
        t = ctx.search(eval=ev, alignments=rows, timing=True)
        assert (a[1] == b[1]).all() and (ev > 1 or len(a[0]) <= 1) and (ev < 1e6 or len(a[0]) > 1024)
        for other in (b, t):
            for f in a[0].dtype.names:
                if f not in ("reserved", "alnoff"):
                    assert a[0][f].tobytes() == other[0][f].tobytes(), (nt, ev, f)
            if rows:
                assert a[3] == other[3]
        assert a[2].npassed == t[2].npassed
        if len(a[0]):
            assert t[2].ms_k_map > 0 and t[2].ms_k_stats > 0
