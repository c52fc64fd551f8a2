"""Timed cases of the search path, through the entry points a program calls.

A case is a dict of plain values:
  call     what a pass runs: "search" (Context.search, one query at a time),
           "batch" (Context.search with batch=True), "serve" (a burst of
           requests to a Server), or one layer of the search for one query:
           "score" (Context.score_block), "phase1", "phase2" and "map"
           (Context.phase1_block, phase2_block, map_block)
  nq       queries, of qmin..qmax positions each
  nt       templates, of tmin..tmax positions (lognormal around tmed, or
           uniform where tmed is 0)
  lists    whether the templates carry distance lists (queries always do)
  rel      templates that are relatives of a query (perturbed windows of its
           profile), so that a pass has hits to report and to realign
  eval     E-value threshold
  contraction, rows
           log-odds product (0 FP32, 1 BF16, 2 FP16); alignment rows wanted

Profiles are the seeded synthetic ones of cother_amd.synth (the reference's
value conventions, the benchmark's length distributions); relatives are cut
from the queries here.  Contexts, with the queries uploaded and the database
resident, are what a program has in hand before it searches.
"""
import ctypes
import math
import os

import numpy as np
import torch

import cother_amd

DEFAULTS = {"nq": 1, "tmed": 220, "lists": True, "rel": 0, "eval": 10.0, "contraction": 0, "rows": False}


def _case(name, **kw):
    return {"name": name, **DEFAULTS, **kw}


def listed():
    return [
        # a short domain against a small private collection, rows wanted for
        # the results file: the smallest call, where latency counts
        _case("small_search", call="search", qmin=61, qmax=61, nt=96, tmin=30, tmax=120, tmed=0, rel=3, rows=True),
        # the everyday search: a median query against a resident database
        _case("typical_search", call="search", qmin=250, qmax=250, nt=4000, tmin=30, tmax=1500, rel=8, rows=True),
        # the same with templates that have no distance information
        _case("nolists_search", call="search", qmin=165, qmax=165, nt=6000, tmin=30, tmax=1500, lists=False, rel=8),
        # a multi-domain query against long templates
        _case("long_search", call="search", qmin=2000, qmax=2000, nt=130, tmin=1000, tmax=3000, tmed=0, rel=2),
        # a permissive threshold: many profiles pass to statistics and MAP
        _case("many_hits_search", call="search", qmin=130, qmax=130, nt=3000, tmin=30, tmax=400, rel=16, eval=1e4),
        # the reduced-precision option, templates without lists
        _case("bf16_search", call="search", qmin=203, qmax=203, nt=3000, tmin=30, tmax=1500, lists=False, rel=4,
              contraction=1),
        # many short queries at once, with and without distance lists
        _case("batch_lists", call="batch", nq=16, qmin=40, qmax=150, nt=1000, tmin=30, tmax=400, rel=16),
        _case("batch_nolists", call="batch", nq=32, qmin=40, qmax=150, nt=4000, tmin=30, tmax=400, lists=False, rel=32),
        # the serving loop: a burst of requests gathered into ticks
        _case("serve_burst", call="serve", nq=12, qmin=40, qmax=150, nt=1500, tmin=30, tmax=400, lists=False, rel=12),
        # single layers of the search
        _case("score_layer", call="score", qmin=89, qmax=89, nt=60, tmin=30, tmax=400, lists=False, rel=1),
        _case("phase2_layer", call="phase2", qmin=372, qmax=372, nt=1500, tmin=30, tmax=700, lists=False, rel=64),
        _case("map_layer", call="map", qmin=372, qmax=372, nt=300, tmin=30, tmax=700, lists=False, rel=48),
    ]


def _loguni(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["search"] * 5 + ["batch", "batch", "serve", "score", "phase1", "phase2", "map"])
    lists = rng.random() < 0.6
    nq, contraction, ev, rows, tmed = 1, 0, 10.0, False, 220
    if call == "search":
        lq, nt, tmin, tmax = _loguni(rng, 40, 1000), _loguni(rng, 50, 6000), 30, rng.choice([400, 1500])
        if rng.random() < 0.15:
            lq, nt, tmin, tmax, tmed = _loguni(rng, 800, 2000), rng.randint(20, 100), 1000, 3000, 0
        contraction = rng.choice([0, 0, 0, 0, 1, 2])
        ev = rng.choice([0.1, 10.0, 10.0, 1e4])
        rows = ev < 100 and rng.random() < 0.5
        qmin = qmax = lq
        cap = 2.2e8 if lists else 4e8
    elif call in ("batch", "serve"):
        nq, nt, tmin, tmax = rng.randint(4, 32), _loguni(rng, 100, 4000), 30, 400
        qmin, qmax = 40, rng.randint(90, 200)
        cap = 2.5e8 if lists else 2.5e9
    else:
        nt = _loguni(rng, 20, 60) if call == "score" else _loguni(rng, 40, 1500)
        qmin = qmax = _loguni(rng, 40, 130) if call == "score" else _loguni(rng, 40, 600)
        tmin, tmax = 30, rng.choice([400, 700])
        contraction = rng.choice([0, 0, 1, 2]) if call == "score" else 0
        cap = 1e8
    mean = (tmin + tmax) / 2 if not tmed else 230
    nt = max(8, min(nt, int(cap / (nq * (qmin + qmax) / 2 * mean))))
    return {"call": call, "nq": nq, "qmin": qmin, "qmax": qmax, "nt": nt, "tmin": tmin, "tmax": tmax, "tmed": tmed,
            "lists": lists, "rel": max(1, min(nt // 2, rng.randint(1, 24))), "eval": ev, "contraction": contraction,
            "rows": rows}


def _relatives(q, n, rng):
    """n templates cut from the queries: windows of at least half a query, frequencies mixed with
    others, distance lists with some values moved by an Angstrom."""
    lens, dist = q.lens(), q.dists()
    own, wins = [], []
    part = np.random.default_rng(n).uniform(0.5, 1.0, n)
    for k in range(n):
        p = k % q.nprof
        ln = max(6, int(round(part[k] * int(lens[p]))))
        own.append(p)
        wins.append((int(rng.integers(0, int(lens[p]) - ln + 1)), ln))
    ls = np.array([w[1] for w in wins], np.int32)
    out = cother_amd.Pset(cother_amd.lib().cth_pset_alloc(n, ls.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))))
    o = 0
    for k, (p, (a, ln)) in enumerate(zip(own, wins)):
        b = int(dist[p]) + a
        w = slice(b, b + ln)
        mix = 0.7 * q.field("trg")[:, w] + 0.3 * rng.dirichlet(np.full(20, 0.5), ln).T
        mix = np.rint(mix * 10000) / 10000
        out.field("trg")[:, o:o + ln] = mix
        out.field("aa")[o:o + ln] = np.frombuffer(b"ARNDCQEGHILKMFPSTWYV", np.uint8)[mix.argmax(0)]
        for f in ("ss", "cv"):
            out.field(f)[:, o:o + ln] = q.field(f)[:, w]
        for f in ("cvprior", "cvnorm2", "sss"):
            out.field(f)[o:o + ln] = q.field(f)[w]
        dd = q.field("dd")[w].copy()
        body = dd[:, 1:]
        body[...] = np.where((body > 2) & (body < 20) & (rng.random(body.shape) < 0.3),
                             body + rng.integers(-1, 2, body.shape).astype(np.int8).view(np.uint8), body)
        out.field("dd")[o:o + ln] = dd
        out.field("trn")[:, o + k:o + k + ln + 1] = q.field("trn")[:, b + p:b + p + ln + 1]
        out.field("bkg")[k] = q.field("bkg")[p]
        out.field("eno")[k] = q.field("eno")[p]
        o += ln
    return out


def _no_lists(ps):
    dd = ps.field("dd")
    dd[...] = 255
    dd[:, 0] = 0


def _informative(ps, rng):
    """Context vectors, norms and priors as profiles of real sequences carry them."""
    n = ps.npos
    v = np.rint(rng.normal(0, 1, (19, n)) * rng.uniform(0.05, 0.3, n) * 10000).astype(np.float32) / np.float32(10000)
    ps.field("cv")[...] = v
    ps.field("cvnorm2")[...] = np.rint((v.astype(np.float64) ** 2).sum(0) * 10000) / 10000
    ps.field("cvprior")[...] = np.rint(rng.uniform(-30, -10, n) * 10000) / 10000


def _sets(case, seed):
    rng = np.random.default_rng(seed)
    threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or len(os.sched_getaffinity(0))
    s1, s2 = (int(v) for v in rng.integers(1, 1 << 40, 2))
    q = cother_amd.synth(case["nq"], 0, lmin=case["qmin"], lmax=case["qmax"], dist_mode=0, sort_desc=0, seed=s1,
                         threads=threads)
    nrel = min(case["rel"], case["nt"] - 1)
    mode = 1 if case["lists"] else 2
    if case["call"] in ("score", "phase1"):
        # matrices come back: their shape, and so the template lengths, are the case's own
        ls = np.random.default_rng(case["nt"]).uniform(case["tmin"], case["tmax"] + 1, case["nt"] - nrel).astype(int)
        db = cother_amd.concat([cother_amd.synth(1, 2, lmin=int(n), dist_mode=mode, seed=s2 + k, threads=1)
                                for k, n in enumerate(np.sort(ls)[::-1])])
    else:
        db = cother_amd.synth(case["nt"] - nrel, 1 if case["tmed"] else 0, float(case["tmed"]), 0.35, case["tmin"],
                              case["tmax"], dist_mode=mode, sort_desc=1, seed=s2, threads=threads)
    if nrel:
        rel = _relatives(q, nrel, rng)
        if not case["lists"]:
            _no_lists(rel)
        db = cother_amd.concat([rel, db])
    if case["call"] == "score":
        _informative(q, rng)
        _informative(db, rng)
    return q, db, rng


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = dict(case)
    s.q, s.db, rng = _sets(case, seed)
    s.ctx = cother_amd.Context(0)
    s.ctx.upload_queries(s.q)
    s.ctx.upload_db(s.db)
    if case["call"] == "serve":
        s.srv = cother_amd.Server(s.ctx, nslots=2, chunk_cols=0, eval=case["eval"], batch=case["nq"],
                                  batch_wait_us=2000)
    if case["call"] == "phase2":
        # the score that the strongest quarter of the profiles reaches passes to statistics
        s.thld = 6.0
        s.space = float(cother_amd.search_space(int(s.q.lens()[0]), s.db.npos, s.db.nprof)[0])
    if case["call"] == "map":
        n = min(case["rel"], case["nt"] - 1)
        s.prof = np.arange(n, dtype=np.int32)
        s.epa = np.rint(rng.uniform(-60, -5, n) * 100).astype(np.float32) / np.float32(100)
    return s


def _hits(c, hits, nh, rows=None):
    """The hit records field by field, at the front of arrays with room for more."""
    room = max(len(hits), c["nq"] * c["nt"] if c["eval"] > 100 else c["rel"] + 32 * c["nq"] + 64)
    out = {"count": np.asarray(nh)}
    for f in hits.dtype.names:
        if f not in ("reserved", "alnoff"):
            out[f] = np.zeros(room, np.int64 if hits[f].dtype.kind == "u" else hits[f].dtype)
            out[f][:len(hits)] = hits[f]
    if rows is not None:
        text = "".join("".join(r) for r in rows).encode()
        out["rows"] = np.zeros(max(len(text), 10 * c["qmax"] * (c["rel"] + 32)), np.uint8)
        out["rows"][:len(text)] = np.frombuffer(text, np.uint8)
    return out


def run(s):
    c = s.case
    call = c["call"]
    if call == "search":
        r = s.ctx.search(eval=c["eval"], contraction=c["contraction"], alignments=c["rows"])
        return _hits(c, r[0], r[1], r[3] if c["rows"] else None)
    if call == "batch":
        r = s.ctx.search(eval=c["eval"], batch=True)
        return _hits(c, r[0], r[1])
    if call == "serve":
        tickets = [s.srv.submit(k) for k in range(c["nq"])]
        got = [s.srv.wait(t)[0] for t in tickets]
        return _hits(c, np.concatenate(got), [len(g) for g in got])
    n = s.db.nprof
    if call == "score":
        sc, md = s.ctx.score_block(0, 0, n, c["contraction"])
        return {"scores": sc, "modscores": md}
    if call == "phase1":
        res, bt = s.ctx.phase1_block(0, 0, n, 6.0, want_btck=True)
        return {**_records(res), "btck": bt}
    if call == "phase2":
        res, passed, stats = s.ctx.phase2_block(0, 0, n, s.thld, s.space)
        # each profile's statistics at its own place
        full = np.zeros((n, 10))
        full[passed] = stats
        return {**_records(res), "stats": full}
    return _records(s.ctx.map_block(0, 0, n, s.prof, s.epa))


def _records(res):
    return {f: res[f] if res[f].dtype.kind != "u" else res[f].astype(np.int64) for f in res.dtype.names}


def _mean_len(case):
    return (case["tmin"] + case["tmax"]) / 2 if not case["tmed"] else min(1.06 * case["tmed"], case["tmax"])


def _updates(n1, n2):
    """Segment-cell updates of one distance-list comparison of lists of n1 and n2 values."""
    if min(n1, n2) < 6:
        return 0
    return 4 * (sum((min(n1, n2 - j) + 3) // 4 for j in range(n2 >> 2, -1, -2)) +
                sum((min(n2, n1 - i) + 3) // 4 for i in range(n1 >> 2, 0, -2)))


def work(case):
    # per position: 44 floats of frequencies, SS, context vector, norm and
    # prior, 7 transitions, two letters, and up to 100 bytes of list; per cell
    # 216 operations of the log-odds, SS and context terms, four for each
    # update of the distance-list comparison, and 45 of the phase-1 DP
    lq = case["nq"] * (case["qmin"] + case["qmax"]) / 2
    mean = _mean_len(case)
    cols = case["nt"] * mean
    cells = lq * cols
    call = case["call"]
    per = 216
    if case["lists"]:
        per += 4 * _updates(int(min(99, lq / case["nq"])), int(min(99, mean)))
    if call != "score":
        per += 45
    out = 104.0 * case["rel"]
    if call == "score":
        out = 8.0 * cells
    elif call == "phase1":
        out = 24.0 * case["nt"] + cells
    elif call == "phase2":
        out = 104.0 * case["nt"]
    flops = per * cells
    if call in ("map", "search", "batch", "serve"):  # forward, backward and the alignment of the relatives
        flops += 300 * case["rel"] * lq / case["nq"] * 0.75 * lq / case["nq"]
    return {"bytes": (lq + cols) * (176 + 28 + 2 + (100 if case["lists"] else 0)) + out, "flops": float(flops)}


# ---- the score matrix in 64 bits -------------------------------------------------


def _table(name):
    return [ln.split() for ln in open(os.path.join(cother_amd.ENVDIR, name)) if ln.strip() and ln.lstrip()[0] != "#"]


def _ss_table():
    rows = _table("ssss")[3:33]
    t = np.zeros((30, 30))
    for r, row in enumerate(rows):
        t[r, :r + 1] = t[:r + 1, r] = [float(v) for v in row[:r + 1]]
    return t


def _cv_map():
    """Keys of the context map and its scores, each the running mean of five; the entries given
    as "+" and the ends take the nearest mean."""
    rows = [r for r in _table("cvs2s") if len(r) > 20]
    keys = np.array([float(v) for v in rows[0]])
    given = [float(v) for v in rows[1] if not v.startswith("+")]
    mean = [sum(given[k:k + 5]) / 5 for k in range(len(given) - 4)]
    vals = [mean[0]] * 2 + mean
    return keys, np.array(vals + [mean[-1]] * (len(keys) - len(vals)))


def exact(case, seed):
    """The score matrices in 64 bits where templates carry no distance lists.  With lists a cell
    adds the three best of segments that often tie exactly, and rounding says which of them count,
    so those outputs, and the later stages' that follow from them (with their piecewise
    exponentials), have no such value."""
    if case["call"] != "score" or case["lists"]:
        return None
    q, db, _ = _sets(case, seed)

    def f64(ps, name):
        return torch.from_numpy(ps.field(name).astype(np.float64))

    pro = torch.from_numpy(np.repeat(np.arange(db.nprof), db.lens()))
    den = 0.5 * (f64(q, "bkg")[0][:, None] + f64(db, "bkg")[pro].T)
    init = torch.log(f64(q, "trg").T @ (f64(db, "trg") / den)) - 0.002
    sq, st = f64(q, "ss"), f64(db, "ss")
    table = torch.from_numpy(_ss_table())
    ss = torch.zeros_like(init)
    for a in range(3):
        r = 10 * a + (sq[a] * 9.999).long()
        for b in range(3):
            c = 10 * b + (st[b] * 9.999).long()
            ss += sq[a][:, None] * st[b] * table[r][:, c]
    ss = 0.12 * (ss + (sq[2][:, None] + 0.1) * (st[2] + 0.1) / 9 - 0.05)
    kap, nu, dim = 10.0, -0.5 * 21, 19
    cterm = (0.5 * dim + nu) * (math.log(0.1) - math.log(2.1))
    cterm += sum(math.log(dim + 1.0 - k) - math.log(2.0) for k in range(1, dim + 1))
    dot = f64(q, "cv").T @ f64(db, "cv") + kap
    lo = (f64(q, "cvnorm2") + 1 + kap)[:, None] * (f64(db, "cvnorm2") + 1 + kap) - dot * dot
    lo = nu * torch.log(lo) + cterm - f64(q, "cvprior")[:, None] - f64(db, "cvprior")
    keys, vals = _cv_map()
    at = (torch.round(2 * lo) - 2 * keys[0]).clamp(0, len(keys) - 1).long()
    sc = ss + 0.15 * torch.from_numpy(vals)[at]
    return {"scores": init + sc, "modscores": sc - 0.5 * 0.15}
