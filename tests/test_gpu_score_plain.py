"""The plain score kernel (every term but the distance one): the logarithm it
uses, ragged tiles, rows and columns outside the quotient correction's ranges,
and the reduced-precision contraction over databases with and without distance
lists, which take the same kernel (test_gpu_product_host.py holds the product
against one formed on the host, test_gpu_score_quotient.py rows that have to be
divided in ragged blocks)."""
import ctypes

import numpy as np
import pytest

import cother_amd
from tests._cv import set_informative_cv

pytestmark = pytest.mark.gpu


def test_device_logarithm_over_all_significands():
    bad = ctypes.c_int(-1)
    assert cother_amd.lib().cth_selftest_logf(ctypes.byref(bad)) == 0
    assert bad.value == 0


@pytest.mark.parametrize("lq,lts", [(1, (1, 2)), (63, (64, 63)), (64, (65, 70)), (65, (30, 34, 64)), (130, (300, 7))])
@pytest.mark.parametrize("divide", [False, True])
def test_matrices_equal_the_oracle(ctx, oracle, lq, lts, divide):
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1300 + lq)
    db = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1310 + lt)
                            for lt in lts])
    set_informative_cv(q, 1, frac=0.8)
    set_informative_cv(db, 2, frac=0.8)
    if divide:
        q.field("trg")[3, lq // 2] = 1e-12
        db.field("trg")[5, 0] = 3.0
    ctx.upload_queries(q)
    ctx.upload_db(db)
    sc, md = ctx.score_block(0, 0, db.nprof)
    osc, omd = oracle.score_matrix(q, 0, db, 0, db.nprof)
    assert (sc.view(np.int32) == osc.view(np.int32)).all()
    assert (md.view(np.int32) == omd.view(np.int32)).all()


@pytest.mark.parametrize("contraction", [1, 2])
def test_contraction_route_equals_the_general_kernel(ctx, contraction):
    q = cother_amd.synth(1, 2, lmin=97, lmax=97, dist_mode=0, sort_desc=0, seed=1321)
    plain = cother_amd.synth(3, 0, lmin=40, lmax=150, dist_mode=2, sort_desc=0, seed=1322)
    mixed = cother_amd.concat([plain, cother_amd.synth(1, 2, lmin=50, lmax=50, dist_mode=1, seed=1323)])
    set_informative_cv(q, 3)
    ctx.upload_queries(q)
    got = {}
    for name, db in (("plain", plain), ("mixed", mixed)):
        ctx.upload_db(db)
        got[name] = ctx.score_block(0, 0, db.nprof, contraction)
    n = plain.npos
    for a, b in zip(got["plain"], got["mixed"]):
        assert (a.view(np.int32) == b[:, :n].view(np.int32)).all()


@pytest.mark.parametrize("contraction", [1, 2])
@pytest.mark.parametrize("lq,lts", [(1, (1,)), (5, (63, 2)), (33, (64,)), (128, (65,)), (129, (31, 33)), (300, (7, 90))])
def test_product_tiles_equal_the_general_kernel(ctx, contraction, lq, lts):
    """The product within the plain kernel at the edges of its tiles (32 of a
    wavefront's rows by 64 columns, 256 rows a workgroup) against the product
    before the general kernel: bit for bit, as both form the same sums."""
    q = cother_amd.synth(1, 2, lmin=lq, lmax=lq, dist_mode=0, sort_desc=0, seed=1330 + lq)
    plain = cother_amd.concat([cother_amd.synth(1, 2, lmin=lt, lmax=lt, dist_mode=2, sort_desc=0, seed=1340 + lt)
                               for lt in lts])
    mixed = cother_amd.concat([plain, cother_amd.synth(1, 2, lmin=50, lmax=50, dist_mode=1, seed=1341)])
    set_informative_cv(q, 4)
    q.field("trg")[:, lq // 2] = 0.0  # a row whose sums are zero
    ctx.upload_queries(q)
    ctx.upload_db(plain)
    got = ctx.score_block(0, 0, plain.nprof, contraction)
    ctx.upload_db(mixed)
    want = ctx.score_block(0, 0, mixed.nprof, contraction)
    for a, b in zip(got, want):
        assert (a.view(np.int32) == b[:, :plain.npos].view(np.int32)).all()
