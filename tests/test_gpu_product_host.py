"""The reduced-precision product within the plain score kernel at the edges of
its tiles (32 of a wavefront's rows, 64 columns, up to 256 rows a workgroup),
against a product formed on the host: the operands rounded to BF16 or FP16 to
nearest even, multiplied and summed in 64 bits."""
import ctypes

import numpy as np
import pytest

import cother_amd
from tests._cv import set_informative_cv

pytestmark = pytest.mark.gpu

# Products of the operands are exact in FP32.  What is left against 64 bits:
# 32 additions of non-negative numbers, each within 2^-23 of the sum whatever
# its rounding (3.9e-6 in the logarithm); the logarithm's ulp and the
# subtraction of the shift (|log| < 16: 2 x 9.6e-7); the sum with the other
# terms (|S| < 16: 9.6e-7); their value taken back from the modular scores
# (2 x 1.2e-7).
TOL = 3.9e-6 + 3 * 9.6e-7 + 2 * 1.2e-7
CVSWGT = 0.15  # the modular scores are the other terms less half of it


def _operand(x, prec):
    if prec == 2:
        return x.astype(np.float16).astype(np.float64)
    u = x.view(np.uint32).astype(np.uint64)
    u = ((u + 0x7fff + ((u >> np.uint64(16)) & np.uint64(1))) >> np.uint64(16)) << np.uint64(16)
    return u.astype(np.uint32).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("lq,nt,lt,tile", [(1, 1, 1, 16), (5, 1, 65, 16), (33, 1, 64, 16), (129, 2, 70, 16),
                                           (130, 160, 200, 28), (300, 250, 240, 128), (300, 520, 230, 256)])
def test_scores_against_a_host_product(ctx, prec, lq, nt, lt, tile):
    rule = cother_amd.lib().cth_score_tile_rows
    rule.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64]
    # the smallest tile that the sizes have to reach
    assert rule(0, lq, nt * lt) >= tile
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1950 + lq)
    db = cother_amd.synth(nt, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1960 + nt)
    set_informative_cv(q, 5)
    q.field("trg")[:, lq // 2] = 0.0  # a row whose sums are zero
    ctx.upload_queries(q)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof, prec)
    pro = np.repeat(np.arange(db.nprof), db.lens())
    den = np.float32(0.5) * (q.field("bkg")[0][:, None] + db.field("bkg")[pro].T)
    A = _operand(np.ascontiguousarray(q.field("trg").T, np.float32), prec)
    B = _operand(np.ascontiguousarray(db.field("trg") / den, np.float32), prec)
    for r in range(0, lq, 50):
        with np.errstate(divide="ignore"):
            want = np.log(A[r:r + 50] @ B) - 0.002
        got = sc[r:r + 50].astype(np.float64) - (md[r:r + 50].astype(np.float64) + 0.5 * CVSWGT)
        zero = np.isneginf(want)
        assert (np.isneginf(got) == zero).all()
        err = np.abs(np.where(zero, 0.0, got) - np.where(zero, 0.0, want))
        assert err.max() < TOL, (r + int(err.max(1).argmax()), int(err.max(0).argmax()), err.max())
