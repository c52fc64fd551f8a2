"""The wall times that a search reports of its two phases, where the device
chooses the stages (with the hits known before the MAP stage and not) and where
the host does: both are there, and they add up to the search."""
import time

import pytest

import cother_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, {"noalloc": True}, {"alignments": True}, {"do_map": False}])
@pytest.mark.parametrize("nt", [60, 1500])
def test_both_phases_are_reported(ctx, nt, kw):
    q = cother_amd.synth(1, 2, lmin=150, lmax=150, dist_mode=2, sort_desc=0, seed=2401)
    db = cother_amd.concat([q, cother_amd.synth(nt, 0, lmin=30, lmax=700, dist_mode=2, sort_desc=1, seed=2402)])
    ctx.upload_queries(q)
    ctx.upload_db(db)
    ctx.search(eval=1e3, **kw)
    runs, timed = [], []
    for _ in range(5):
        t = time.perf_counter()
        st = ctx.search(eval=1e3, **kw)[2]
        wall = (time.perf_counter() - t) * 1e3
        assert 0 < st.ms_phase1 and 0 < st.ms_phase2 and st.ms_phase1 + st.ms_phase2 <= wall
        runs.append((st.ms_phase1, st.ms_phase2))
        st = ctx.search(eval=1e3, timing=True, **kw)[2]
        timed.append((st.ms_k_score + st.ms_k_dp, st.ms_k_stats + st.ms_k_map))
    # a phase's kernels take part of its time (the least of the runs, and by
    # half: clocks differ), and those of phase 2 most of it
    for k in range(2):
        assert min(r[k] for r in runs) > 0.5 * min(t[k] for t in timed)
    assert min(r[1] for r in runs) < 2 * min(t[1] for t in timed) + 1.0


def test_no_hits(ctx):
    q = cother_amd.synth(1, 2, lmin=60, lmax=60, dist_mode=2, sort_desc=0, seed=2411)
    db = cother_amd.synth(1500, 0, lmin=30, lmax=700, dist_mode=2, sort_desc=1, seed=2412)
    ctx.upload_queries(q)
    ctx.upload_db(db)
    hits, _, st = ctx.search(eval=1e-30)
    assert len(hits) == 0 and st.ms_phase1 > 0 and st.ms_phase2 > 0
