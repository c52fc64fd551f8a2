"""The wavefront's walk over the traceback bytes: runs of each move longer than
a chunk of the path (32 and 64 steps) and a tile (64 rows, 61 columns), at all
alignments of a template's first column, against the oracle, bit for bit."""
import numpy as np
import pytest

import cother_amd
from tests.test_gpu_dp_sweep import _equals_oracle as phase1_equals_oracle
from tests.test_gpu_map_sweep import _equals_oracle as map_equals_oracle

pytestmark = pytest.mark.gpu


def _like(q, parts, seed):
    """A template of the query's windows (a, b) and, for a number, of so many other positions."""
    n = sum(p if isinstance(p, int) else p[1] - p[0] for p in parts)
    t = cother_amd.synth(1, 0, lmin=n, lmax=n, dist_mode=2, sort_desc=0, seed=seed)
    o = 0
    for p in parts:
        if isinstance(p, int):
            o += p
            continue
        w, to = slice(*p), slice(o, o + p[1] - p[0])
        for f in ("trg", "ss", "cv"):
            t.field(f)[:, to] = q.field(f)[:, w]
        for f in ("cvprior", "cvnorm2", "sss", "aa"):
            t.field(f)[to] = q.field(f)[w]
        o = to.stop
    return t


@pytest.mark.parametrize("lead", [1, 2, 3, 4])
def test_long_runs_of_each_move(ctx, oracle, lead):
    q = cother_amd.synth(1, 0, lmin=230, lmax=230, dist_mode=2, sort_desc=0, seed=1501)
    # the strongest residues at every position, so that the copied windows align, and cheap gaps
    q.field("trg")[...] = 0.002
    q.field("trg")[np.random.default_rng(1502).integers(0, 20, 230), np.arange(230)] = 0.962
    db = cother_amd.concat([cother_amd.synth(1, 0, lmin=lead, lmax=lead, dist_mode=2, sort_desc=0, seed=1503),
                            _like(q, [(0, 230)], 1504),
                            _like(q, [(0, 110), 90, (110, 230)], 1505),
                            _like(q, [(0, 75), (165, 230)], 1506),
                            _like(q, [(0, 61), 1, (61, 125), (130, 190), 66, (192, 230)], 1507)])
    for s in (q, db):
        trn = s.field("trn")
        trn[...] = np.log(np.array([0.96, 0.02, 0.02, 0.02, 0.98, 0.02, 0.98], np.float32))[:, None]
    phase1_equals_oracle(ctx, oracle, q, db)
    map_equals_oracle(ctx, oracle, q, db)
    # the cases are what they are meant to be: runs across chunks and tiles
    prof = np.arange(1, 4, dtype=np.int32)
    res = ctx.map_block(0, 0, db.nprof, prof, np.full(3, 5.0, np.float32))
    assert res["alnlen"][0] >= 200 and (res["ngaps"][1:] > 64).all(), (res["alnlen"], res["ngaps"])
