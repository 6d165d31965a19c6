"""Performance cases: the work a user of this framework has it do.

Five forms of the clause-vs-assignment path, each through the entry points a
program calls, and the residency network's training pass:

  sweep   Engine.sweep: every clause against every assignment of the table,
          the records (both masks) then taken on the device with
          gss_hits_gather;
  step    a batched step (gss_step_submit / gss_step_wait): table updates,
          check, roll forward, records on the host;
  gpurun  the drop-in GpuClauseSharer: solvers set values and send an
          assignment, gpuRun twice, reported clauses popped;
  serve   the serving loop (GpuServer): a burst of requests, each one's
          records read when it completes;
  grad    Residency.grad: one forward and backward pass of the scorer's MLP.

Records come in no set order, so a pass files them by clause, as a program
that delivers them to its solvers does: `sweep` into both masks per (clause,
word), `step` into the words with a report per clause, the others sorted.

Two distributions, as in gpusharesat_amd/workloads.py: "random" (uniform
signs and values, a fraction of the variables assigned: short clauses report
in most words) and "planted" (assignments and clauses near one solution, the
slots of a word copies of a base with a few variables redrawn: few reports,
as solvers send them).  Clause lengths are 2 + Geometric(p) or Pareto(1.5)
from 2, capped.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from gpusharesat_amd import _lib, serving
from gpusharesat_amd.engine import Engine, VAR_UPDATE_DTYPE, round_words
from gpusharesat_amd.residency import FEATURES, HIDDEN, PARAMS, Residency
from gpusharesat_amd.sharer import GpuClauseSharer, default_options

DEV = "cuda"
P_ASSIGNED, AGREE, LIT_TRUE = 0.95, 0.99, 0.9  # planted distribution
REPORT_ROOM = 256  # clauses reported to a solver in a pass, at most


def listed():
    return [
        # one solver thread of the reference's perfTest shape, a GPU thread
        # that turns over as fast as it can: launches and latency
        {"name": "gpurun-1", "kind": "gpurun", "solvers": 1, "vars": 500, "moved": 500,
         "clauses": 200_000, "min_len": 10},
        # a small portfolio of solver threads over one clause DB, each sending
        # two assignments that differ in the tail of its trail
        {"name": "gpurun-4", "kind": "gpurun", "solvers": 4, "vars": 20_000, "moved": 300,
         "clauses": 300_000, "min_len": 12},
        # the plain-64 instance: 64 assignments of one solver, a small DB
        {"name": "sweep-64", "kind": "sweep", "vars": 10_000, "clauses": 100_000, "slots": 64,
         "dist": "random", "assigned": 0.6, "lengths": "geometric", "p": 0.15, "cap": 100},
        # an odd number of assignments over a table narrower than a line
        {"name": "sweep-333", "kind": "sweep", "vars": 99_991, "clauses": 1_000_003, "slots": 333,
         "dist": "planted", "assigned": P_ASSIGNED, "lengths": "geometric", "p": 0.1, "cap": 200},
        # the headline instance: 1M variables, 4M clauses, 1024 assignments
        {"name": "sweep-1024", "kind": "sweep", "vars": 1_000_000, "clauses": 4_000_000,
         "slots": 1024, "dist": "random", "assigned": 0.4, "lengths": "geometric", "p": 0.1,
         "cap": 200},
        # 16 solvers' windows near a solution
        {"name": "sweep-1024-planted", "kind": "sweep", "vars": 500_000, "clauses": 2_000_000,
         "slots": 1024, "dist": "planted", "assigned": P_ASSIGNED, "lengths": "geometric",
         "p": 0.1, "cap": 200},
        # the widest table, heavy-tailed lengths
        {"name": "sweep-4096", "kind": "sweep", "vars": 200_000, "clauses": 400_000,
         "slots": 4096, "dist": "planted", "assigned": P_ASSIGNED, "lengths": "pareto", "p": 1.5,
         "cap": 500},
        # a step of few updates over a young DB: latency of the graph
        {"name": "step-small", "kind": "step", "vars": 50_000, "clauses": 100_000, "slots": 512,
         "flips": 2, "screen": False, "records": serving.RECORDS_IDS, "lengths": "geometric",
         "p": 0.1, "cap": 200},
        # batched-16: 64 words, screened steps, one record per clause
        {"name": "step-batched", "kind": "step", "vars": 1_000_000, "clauses": 3_000_000,
         "slots": 2176, "flips": 64, "screen": True, "records": serving.RECORDS_CLAUSES,
         "lengths": "pareto", "p": 1.5, "cap": 500},
        # the same table without screening, records per (clause, word)
        {"name": "step-exact", "kind": "step", "vars": 300_000, "clauses": 1_000_000,
         "slots": 1024, "flips": 16, "screen": False, "records": serving.RECORDS_IDS,
         "lengths": "geometric", "p": 0.1, "cap": 200},
        # requests of several solvers that arrive together
        {"name": "serve-burst", "kind": "serve", "vars": 1_000_000, "clauses": 400_000,
         "solvers": 8, "requests": 6, "slots": 200, "flips": 32},
        # one snapshot of the residency scorer, forward and backward
        {"name": "grad-8192", "kind": "grad", "samples": 8192},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gpurun", "sweep", "sweep", "sweep", "step", "step", "serve", "grad"])
    if kind == "gpurun":
        vars_ = _log_uniform(rng, 300, 30_000)
        return {"kind": kind, "solvers": rng.randint(1, 8), "vars": vars_,
                "moved": _log_uniform(rng, 50, min(vars_, 1000)),
                "clauses": _log_uniform(rng, 20_000, 300_000), "min_len": rng.randint(10, 13)}
    if kind == "serve":
        return {"kind": kind, "vars": _log_uniform(rng, 50_000, 1_000_000),
                "clauses": _log_uniform(rng, 50_000, 600_000), "solvers": rng.randint(2, 16),
                "requests": rng.randint(1, 8), "slots": rng.randint(17, 400),
                "flips": rng.randint(8, 40)}
    if kind == "grad":
        return {"kind": kind, "samples": _log_uniform(rng, 400, 40_000)}
    if rng.random() < 0.7:
        lengths, p, cap = "geometric", round(rng.uniform(0.08, 0.2), 3), 200
    else:
        lengths, p, cap = "pareto", 1.5, 500
    slots = _log_uniform(rng, 40, 4096)
    if kind == "step":
        clauses = _log_uniform(rng, 20_000, min(3_000_000, 4_000_000_000 // slots))
        return {"kind": kind, "vars": _log_uniform(rng, 20_000, min(1_000_000, 600_000_000 // slots)),
                "clauses": clauses, "slots": slots, "flips": _log_uniform(rng, 2, 64),
                "screen": rng.random() < 0.5,
                "records": rng.choice([serving.RECORDS_IDS, serving.RECORDS_CLAUSES]),
                "lengths": lengths, "p": p, "cap": cap}
    clauses = _log_uniform(rng, 20_000, min(4_000_000, 4_000_000_000 // slots))
    dist = rng.choice(["random", "planted", "planted"])
    return {"kind": kind, "vars": _log_uniform(rng, 5_000, min(1_000_000, 600_000_000 // slots)),
            "clauses": clauses, "slots": slots, "dist": dist,
            "assigned": round(rng.uniform(0.3, 0.7), 2) if dist == "random" else P_ASSIGNED,
            "lengths": lengths, "p": p, "cap": cap}


# ---- inputs ------------------------------------------------------------------

def _lengths(g, case):
    u = torch.rand(case["clauses"], generator=g, device=DEV, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    if case["lengths"] == "geometric":  # failures before the first success
        n = 2 + torch.floor(torch.log(u) / math.log(1.0 - case["p"]))
    else:
        n = torch.floor(2.0 * u ** (-1.0 / case["p"]))
    return n.clamp_(max=case["cap"]).to(torch.int64)


def _clauses(g, case, sigma):
    """Literals and lengths on the host; with sigma each literal is true under
    it with probability LIT_TRUE, else signs are uniform."""
    lens = _lengths(g, case)
    total = int(lens.sum())
    v = torch.randint(0, case["vars"], (total,), generator=g, device=DEV)
    if sigma is None:
        sign = torch.randint(0, 2, (total,), generator=g, device=DEV)
    else:  # literal 2v + 1 is the negation: true where sigma is false
        true = torch.rand(total, generator=g, device=DEV) < LIT_TRUE
        sign = (true != sigma[v]).to(torch.int64)
    lits = (2 * v + sign).to(torch.int32)
    return lits.cpu().numpy().view(np.uint32), lens.to(torch.int32).cpu().numpy()


def _random_bits(g, shape, p):
    """int64 words whose bits are each set with probability p (to 1/256)."""
    x = torch.zeros(shape, dtype=torch.int64, device=DEV)
    k = round(p * 256)
    for b in range(8):
        r = torch.randint(-(1 << 63), (1 << 63) - 1, shape, generator=g, device=DEV)
        x = (r | x) if k >> b & 1 else (r & x)
    return x


def _base(g, vars_, words, sigma):
    """Planted words: every slot of a word holds the same assignment."""
    d = torch.rand((vars_, words), generator=g, device=DEV) < P_ASSIGNED
    t = d & ((torch.rand((vars_, words), generator=g, device=DEV) < AGREE) == sigma[:, None])
    return -d.to(torch.int64), -t.to(torch.int64)


def _valid(slots, words):
    v = np.zeros(words, np.uint64)
    v[: slots // 64] = np.uint64(0xFFFFFFFFFFFFFFFF)
    if slots % 64:
        v[slots // 64] = np.uint64((1 << slots % 64) - 1)
    return v


def _redraws(g, case, words, sigma):
    """`flips` variables redrawn per slot: (var, word), the slots redrawn and
    their values, one row per (var, word)."""
    slot = torch.arange(case["slots"], device=DEV).repeat_interleave(case["flips"])
    v = torch.randint(0, case["vars"], slot.shape, generator=g, device=DEV)
    key = torch.unique((v * words + slot // 64) * 64 + slot % 64)
    cell, bit = key // 64, torch.bitwise_left_shift(torch.ones_like(key), key % 64)
    d = torch.rand(key.shape, generator=g, device=DEV) < P_ASSIGNED
    t = d & ((torch.rand(key.shape, generator=g, device=DEV) < AGREE) == sigma[cell // words])
    cells, inv = torch.unique(cell, return_inverse=True)
    sums = [torch.zeros_like(cells).scatter_add_(0, inv, bit * on)  # distinct bits: a sum is an or
            for on in (torch.ones_like(bit), d.to(torch.int64), t.to(torch.int64))]
    return cells, *sums


def _engine(case, lits, lens, is_def, is_true):
    e = Engine(0)
    words = round_words((case["slots"] + 63) // 64)
    e.append(lits, lens)
    e.reset_assignments(case["vars"], words)
    e.upload(is_def.cpu().numpy().view(np.uint64), is_true.cpu().numpy().view(np.uint64))
    # first place of each length's clauses in the results
    count = np.bincount(lens, minlength=int(lens.max()) + 2)
    start = torch.from_numpy(np.concatenate([[0], np.cumsum(count)])[:-1]).to(DEV)
    return {"e": e, "words": words, "start": start, "n": lens.size,
            "valid": _valid(case["slots"], words)}


def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    if kind == "grad":
        return _prepare_grad(case, seed)
    if kind == "gpurun":
        return _prepare_gpurun(case, seed)
    sigma = torch.rand(case["vars"], generator=g, device=DEV) < 0.5
    if kind == "serve":
        return _prepare_serve(case, g, sigma, seed)
    words = (case["slots"] + 63) // 64
    if kind == "sweep" and case["dist"] == "random":
        lits, lens = _clauses(g, case, None)
        d = _random_bits(g, (case["vars"], words), case["assigned"])
        t = d & _random_bits(g, (case["vars"], words), 0.5)
        return {"kind": kind, **_engine(case, lits, lens, d, t)}
    lits, lens = _clauses(g, case, sigma)
    d, t = _base(g, case["vars"], words, sigma)
    redrawn = dict(case, flips=case.get("flips", 32))
    cells, mask, rd, rt = _redraws(g, redrawn, words, sigma)
    fd, ft = d.view(-1), t.view(-1)
    nd, nt = (fd[cells] & ~mask) | rd, (ft[cells] & ~mask) | rt
    if kind == "sweep":
        fd[cells], ft[cells] = nd, nt
        return {"kind": kind, **_engine(case, lits, lens, d, t)}
    st = {"kind": kind, **_engine(case, lits, lens, d, t)}
    ups = np.empty(cells.numel(), VAR_UPDATE_DTYPE)
    ups["var"] = (cells // words).cpu().numpy()
    ups["word"] = (cells % words).cpu().numpy()
    ups["is_def"] = nd.cpu().numpy().view(np.uint64)
    ups["is_true"] = nt.cpu().numpy().view(np.uint64)
    last = np.full(st["words"], -1, np.int8)
    last[:words] = 63
    if case["slots"] % 64:
        last[words - 1] = case["slots"] % 64 - 1
    st.update(ups=ups, last=last, records=case["records"],
              flags=serving.STEP_SCREEN if case["screen"] else 0)
    return st


def _prepare_gpurun(case, seed):
    rng = np.random.default_rng(seed)
    n, lo = case["clauses"], case["min_len"]
    lens = rng.integers(lo, lo + 9, size=n)
    lits = rng.integers(0, 2 * case["vars"], size=int(lens.sum())).astype(np.int32)
    s = GpuClauseSharer(default_options(min_gpu_latency_micros=0, verbosity=0))
    s.setVarCount(case["vars"])
    s.setCpuSolverCount(case["solvers"])
    add, cid = _lib.load().gss_sharer_add_clause, ctypes.c_int64()
    at, ref = lits.ctypes.data, ctypes.byref(cid)
    for k in lens.tolist():
        add(s._h, -1, at, k, ref)
        at += 4 * k
    # a solver's variables are true, false or unset with equal chances; the
    # first `moved` ones take two sets of values in turn
    tails = []
    for k in range(case["solvers"]):
        def values(lo, hi):
            p = rng.integers(0, 3, size=hi - lo)
            vs = np.flatnonzero(p < 2)
            return (2 * (vs + lo) + (p[vs] == 1)).astype(np.int32)
        s.trySetSolverValues(k, values(case["moved"], case["vars"]))
        tails.append((values(0, case["moved"]), values(0, case["moved"])))
    s.execute()  # the clauses reach the GPU
    return {"kind": "gpurun", "s": s, "tails": tails, "width": lo + 10}


def _prepare_serve(case, g, sigma, seed):
    rng = np.random.default_rng(seed)
    c = dict(case, lengths="geometric", p=0.1, cap=200)
    lits, lens = _clauses(g, c, sigma)
    srv = serving.GpuServer(case["vars"], case["solvers"], records=serving.RECORDS_IDS)
    for s in range(case["solvers"]):
        d = torch.rand(case["vars"], generator=g, device=DEV) < float(rng.uniform(0.7, P_ASSIGNED))
        t = d & ((torch.rand(case["vars"], generator=g, device=DEV) < AGREE) == sigma)
        d, t = d.cpu().numpy(), t.cpu().numpy()
        vs = np.flatnonzero(d)
        u = np.zeros(vs.size, serving.BASE_UP_DTYPE)
        u["var"], u["base"], u["is_def"], u["is_true"] = vs, s, 1, t[vs]
        srv.update_base(u)
    if srv.add_clauses(lits, lens) != 0:
        raise RuntimeError("clauses refused")
    host_sigma = sigma.cpu().numpy()
    reqs = []
    for r in range(case["requests"]):
        k = int(rng.integers(max(1, case["slots"] // 2), case["slots"] + 1))
        reqs.append((r % case["solvers"], k,
                     serving.slot_patches(rng, case["vars"], k, case["flips"], P_ASSIGNED,
                                          host_sigma, AGREE)))
    st = {"kind": "serve", "srv": srv, "reqs": reqs, "room": case["clauses"] // 4}
    rid = srv.submit(0, 1, np.zeros(0, serving.PATCH_DTYPE))  # clauses and bases reach the GPU
    while rid not in srv.poll(16, 1_000_000):
        pass
    srv.release(rid)
    return st


def _grad_inputs(case, seed):
    """Feature rows in the scorer's ranges, labels, class weights, weights."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    x = rng.random((n, FEATURES), dtype=np.float32)
    x[:, 1] = x[:, 1] < 0.1
    x[:, 3] = x[:, 3] < 0.2
    x[:, 11] = 2 * x[:, 11] - 1
    y = (rng.random(n) < 0.2).astype(np.float32)
    wt = np.where(y > 0.5, np.float32(2.5), np.float32(0.625)).astype(np.float32)
    p = np.zeros(PARAMS, np.float32)
    o = HIDDEN * FEATURES
    p[:o] = (rng.random(o) * 2 - 1) * math.sqrt(6 / FEATURES)
    p[o:o + HIDDEN] = (rng.random(HIDDEN) - 0.5) * 0.2
    o += HIDDEN
    p[o:o + HIDDEN * HIDDEN] = (rng.random(HIDDEN * HIDDEN) * 2 - 1) * math.sqrt(6 / HIDDEN)
    o += HIDDEN * HIDDEN
    p[o:o + HIDDEN] = (rng.random(HIDDEN) - 0.5) * 0.2
    o += HIDDEN
    p[o:o + HIDDEN] = (rng.random(HIDDEN) * 2 - 1) * 0.1
    return x, y, wt, p


def _prepare_grad(case, seed):
    x, y, wt, p = _grad_inputs(case, seed)
    e = Engine(0)
    e.enable_tags()
    r = Residency(e, 1024)
    r.params = p
    return {"kind": "grad", "e": e, "r": r, "x": x, "y": y, "wt": wt}


# ---- one pass ----------------------------------------------------------------

def run(st):
    return {"sweep": _run_sweep, "step": _run_step, "gpurun": _run_gpurun, "serve": _run_serve,
            "grad": _run_grad}[st["kind"]](st)


def _run_sweep(st):
    """Both masks of every (clause, word), zero without a report."""
    e, words = st["e"], st["words"]
    n = e.sweep(st["valid"])
    rec = torch.empty((n, 3), dtype=torch.int64, device=DEV)
    if n:
        torch.cuda.current_stream().synchronize()  # the engine writes rec on its own stream
        got = ctypes.c_int64()
        _lib.call("gss_hits_gather", e.handle, rec.data_ptr(), n, ctypes.byref(got))
    out = torch.zeros((st["n"] * words, 2), dtype=torch.int64, device=DEV)
    if n:
        first = rec[:, 0].contiguous()  # row, length, word
        half = first.view(torch.int16).view(n, 4)
        clause = st["start"].index_select(0, half[:, 2].int()) + first.view(torch.int32)[::2]
        out.index_copy_(0, torch.add(half[:, 3], clause, alpha=words), rec[:, 1:])
    return out


def _run_step(st):
    """The words with a report of every clause."""
    e = st["e"]
    serving.submit(e, st["valid"], ups=st["ups"], last_pos=st["last"], records=st["records"],
                   flags=st["flags"])
    n, _ = e.step_wait()
    out = torch.zeros(st["n"], dtype=torch.int64, device=DEV)
    if n:
        by_clause = st["records"] == serving.RECORDS_CLAUSES
        view = e.step_clauses_view() if by_clause else e.step_ids_view()
        rec = torch.from_numpy(view.view(np.int64)).to(DEV).view(n, -1)
        half = rec.view(torch.int16)
        clause = st["start"].index_select(0, half[:, 2].int()) + rec.view(torch.int32)[:, 0]
        if by_clause:
            out.index_copy_(0, clause, rec[:, 1])
        else:
            out.scatter_add_(0, clause, torch.bitwise_left_shift(torch.ones_like(clause),
                                                                 half[:, 3].long()))
    return out


def _run_gpurun(st):
    """Id, length and literals of the clauses reported to each solver, one a
    row, by id; rows past them are zero."""
    s, tails = st["s"], st["tails"]
    for k, (first, second) in enumerate(tails):
        for old, new in ((second, first), (first, second)):
            s.unsetSolverValues(k, old)
            if not s.trySetSolverValues(k, new) or s.trySendAssignment(k) < 0:
                raise RuntimeError("no assignment slot")
    s.execute()
    out = []
    for k in range(len(tails)):
        rows = np.zeros((REPORT_ROOM, st["width"]), np.int64)
        for i, (cid, lits) in enumerate(sorted((cid, lits) for lits, cid in s.popAll(k))):
            rows[i, 0], rows[i, 1] = cid, len(lits)
            rows[i, 2:2 + len(lits)] = lits
        out.append(rows)
    return out


def _run_serve(st):
    """clause * 64 + word of every request's records, ascending; zeros past
    them."""
    srv = st["srv"]
    ids = [srv.submit(*r) for r in st["reqs"]]
    left = set(ids)
    while left:
        left.difference_update(srv.poll(64, 1_000_000))
    out = []
    for rid in ids:
        rec = srv.result(rid)[1]
        srv.release(rid)
        keys = np.zeros(st["room"], np.int64)
        keys[:rec.size] = np.sort(rec["clause"] * 64 + rec["word"])
        out.append(keys)
    return out


def _run_grad(st):
    loss, grad = st["r"].grad(st["x"], st["y"], st["wt"])
    return {"loss": np.float32(loss), "grad": grad}


def exact(case, seed):
    """Loss and gradient in 64 bits; the other kinds return whole numbers."""
    if case["kind"] != "grad":
        return None
    x, y, wt, p = (a.astype(np.float64) for a in _grad_inputs(case, seed))
    o = np.cumsum([0, HIDDEN * FEATURES, HIDDEN, HIDDEN * HIDDEN, HIDDEN, HIDDEN])
    w1, b1 = p[o[0]:o[1]].reshape(HIDDEN, FEATURES), p[o[1]:o[2]]
    w2, b2 = p[o[2]:o[3]].reshape(HIDDEN, HIDDEN), p[o[3]:o[4]]
    w3, b3 = p[o[4]:o[5]], p[o[5]]
    n = y.size
    z1 = x @ w1.T + b1
    a1 = np.maximum(z1, 0)
    z2 = a1 @ w2.T + b2
    a2 = np.maximum(z2, 0)
    z3 = a2 @ w3 + b3
    loss = np.sum(wt * (np.maximum(z3, 0) - z3 * y + np.log1p(np.exp(-np.abs(z3))))) / n
    d3 = wt * (1 / (1 + np.exp(-z3)) - y)
    d2 = np.where(z2 > 0, d3[:, None] * w3, 0)
    d1 = np.where(z1 > 0, d2 @ w2, 0)
    grad = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ a1).ravel(), d2.sum(0),
                           a2.T @ d3, [d3.sum()]]) / n
    return {"loss": np.float64(loss), "grad": grad}


def work(case):
    kind = case["kind"]
    if kind == "grad":
        n = case["samples"]
        return {"bytes": 4 * (n * (FEATURES + 2) + 2 * PARAMS), "flops": 6 * n * (PARAMS - 2 * HIDDEN)}
    if kind == "gpurun":
        lits = case["clauses"] * (case["min_len"] + 4)
        return {"bytes": 4 * lits + 16 * case["solvers"] * case["vars"], "flops": 0}
    if kind == "serve":
        words = case["requests"] * ((case["slots"] * 3 // 4 + 63) // 64)
        return {"bytes": 4 * case["clauses"] * 11 + 16 * words * case["vars"], "flops": 0}
    mean = 1 / case["p"] + 1 if case["lengths"] == "geometric" else 5.0
    words = (case["slots"] + 63) // 64
    out = 16 * words if kind == "sweep" else 8
    return {"bytes": int(case["clauses"] * (4 * mean + out)) + 16 * words * case["vars"], "flops": 0}
