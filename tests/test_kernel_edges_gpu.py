"""Sweep kernels and steps at the sizes where they change course, against the
oracle: clause lengths around the literals held per lane group (4, 8, 16) and
the rows kept for the negated-row reads (4, 8), clause counts around the
clauses of a wave pass (64 / W, 64 when screened), and step records around the
size up to which the step itself writes them to pinned memory.
"""
import numpy as np
import pytest

import _oracle as orc
from gpusharesat_amd import serving as sv
from gpusharesat_amd.engine import (HIT_CLAUSE_DTYPE, HIT_DTYPE, HIT_ID_DTYPE, TUNE_SCHEDULE,
                                    TUNE_TASK_CLAUSES, TUNE_WAVES_PER_CU)

pytestmark = pytest.mark.gpu

ALL = np.uint64(0xFFFFFFFFFFFFFFFF)
DIRECT_WORDS = 64 * 1024  # 8-byte words of records a step writes to pinned memory itself


def edge_case(W):
    """Clauses of 1 to 36, 64, 65 and 129 literals, mostly false with about one
    other literal anywhere in the clause, so that many end with exactly one
    non-false literal past the kept rows; words that are copies of one value
    but for a few slots."""
    rng = np.random.default_rng(4000 + W)
    V, cpw = 700, 64 // W
    counts = [1, max(1, cpw - 1), cpw, cpw + 1, 3 * cpw + 2, 65]
    lens = np.concatenate([np.full(counts[i % len(counts)], n, np.int32)
                           for i, n in enumerate([*range(1, 37), 64, 65, 129])])
    lens = rng.permutation(lens)
    base_def = rng.random((V, W)) < 0.9
    sigma = rng.random(V) < 0.5
    is_def = np.where(base_def, ALL, np.uint64(0))
    is_true = np.where(base_def & sigma[:, None], ALL, np.uint64(0))
    for _ in range(4):  # a few slots differ
        bit = np.uint64(1) << rng.integers(0, 64, size=(V, W), dtype=np.uint64)
        is_def ^= np.where(rng.random((V, W)) < 0.2, bit, np.uint64(0))
        is_true ^= np.where(rng.random((V, W)) < 0.2, bit, np.uint64(0))
    is_true &= is_def
    v = rng.integers(0, V, size=int(lens.sum()))
    false = rng.random(v.size) > 1.0 / np.repeat(lens, lens)
    # literal 2v is false where v is, 2v + 1 where v is true
    lits = (2 * v + (false == sigma[v])).astype(np.uint32)
    valid = np.full(W, ALL)
    valid[-1] = np.uint64(0x7FFFFFFFFFFFFF0F)
    if W > 2:
        valid[1] = 0
    off = np.zeros(lens.size + 1, np.int64)
    off[1:] = np.cumsum(lens)
    return V, lits, lens, is_def, is_true, valid, orc.sweep(off, lits, is_def, is_true, valid)


@pytest.mark.parametrize("W", [1, 2, 4, 8, 16, 32, 64])
def test_edges_of_lengths_and_passes(engine_factory, W):
    V, lits, lens, is_def, is_true, valid, exp = edge_case(W)
    assert (exp["unit_mask"] != 0).sum() > 100 and (exp["false_mask"] != 0).sum() > 100
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    key = rows[exp["clause"]] | (lens[exp["clause"]].astype(np.uint64) << np.uint64(32))
    ids = key | (exp["word"].astype(np.uint64) << np.uint64(48))
    full = np.zeros(exp.size, HIT_DTYPE)
    full.view(np.uint64).reshape(-1, 3)[:, 0] = ids
    full["false_mask"], full["unit_mask"] = exp["false_mask"], exp["unit_mask"]
    clauses, inv = np.unique(key, return_inverse=True)
    by_clause = np.zeros(clauses.size, HIT_CLAUSE_DTYPE)
    by_clause.view(np.uint64).reshape(-1, 2)[:, 0] = clauses
    np.bitwise_or.at(by_clause["words"], inv, np.uint64(1) << exp["word"].astype(np.uint64))

    def same(got, want):
        a = got.view(np.uint64).reshape(got.size, -1)
        b = want.view(np.uint64).reshape(want.size, -1)
        assert np.array_equal(a[np.argsort(a[:, 0])], b[np.argsort(b[:, 0])])

    print(f"{W} words: {lens.size} clauses, {exp.size} records", flush=True)
    e.sweep(valid)
    same(e.hits(), full)
    for flags in (0, sv.STEP_SCREEN):
        for form, view, want in ((sv.RECORDS_FULL, e.step_hits_view, full),
                                 (sv.RECORDS_IDS, e.step_ids_view, ids.view(HIT_ID_DTYPE)),
                                 (sv.RECORDS_CLAUSES, e.step_clauses_view, by_clause)):
            print(f"step: form {form}, flags {flags}", flush=True)
            sv.submit(e, valid, records=form, flags=flags)
            assert e.step_wait()[0] == want.size
            same(view(), want)


@pytest.mark.parametrize("form, words", [(sv.RECORDS_FULL, 3), (sv.RECORDS_IDS, 1),
                                         (sv.RECORDS_CLAUSES, 2)])
def test_records_around_the_direct_size(engine_factory, form, words):
    """One-literal clauses over an undefined table, one record each: steps whose
    records take just up to the size and just past it, appended by steps of few
    literals and of many, two steps in flight; a step's records keep their
    place until its slot is waited for again."""
    e = engine_factory()
    e.reset_assignments(64, 1)
    at = DIRECT_WORDS // words
    totals = [1, 16384, 16385, at - 1, at, at + 1, at + 2, at + 2]
    view = {sv.RECORDS_FULL: e.step_hits_view, sv.RECORDS_IDS: e.step_ids_view,
            sv.RECORDS_CLAUSES: e.step_clauses_view}[form]
    have, held = 0, []
    for k, n in enumerate(totals):
        sv.submit(e, np.full(1, ALL), lits=np.full(n - have, 2 * (k % 64), np.uint32),
                  lens=np.ones(n - have, np.int32), records=form)
        have = n
        if k > 0:  # two in flight
            assert e.step_wait()[0] == totals[k - 1]
            held.append((view(), totals[k - 1]))
        # step k has taken the slot of step k - 2, whose records are still to be read
        for got, m in held[-2:]:
            rows = np.sort(got["row"])
            assert got.size == m and np.array_equal(rows, np.arange(m)), (k, m)
    assert e.step_wait()[0] == totals[-1]
    assert np.array_equal(np.sort(view()["row"]), np.arange(totals[-1]))


def test_first_sweeps_of_engines_in_turn():
    """Engines that run one sweep each and go: a new engine's first wait must not
    take what the one before left in the pinned counts it is handed again."""
    from gpusharesat_amd.engine import Engine
    for n in (100, 7000, 3, 50000, 1, 900):
        e = Engine(0)
        e.reset_assignments(64, 1)
        e.append(np.full(n, 2, np.uint32), np.ones(n, np.int32))
        assert e.sweep(np.full(1, ALL)) == n
        assert np.array_equal(np.sort(e.hits()["row"]), np.arange(n))
        e.close()


@pytest.mark.parametrize("passes", [1, 2, 3, "W", "W+1", 1000])
@pytest.mark.parametrize("W", [1, 2, 4, 8, 16, 32, 64])
def test_passes_a_wave_takes_at_a_time(engine_factory, W, passes):
    """Runs of one pass, an odd number, W (the passes a clause record is held
    for) and more, few waves with many tasks, short clauses first: all records
    as without these settings."""
    V, lits, lens, is_def, is_true, valid, exp = edge_case(W)
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    n = {"W": W, "W+1": W + 1}.get(passes, passes)
    e.set_tuning(TUNE_TASK_CLAUSES, n * (64 // W))
    if n != 2:
        e.set_tuning(TUNE_WAVES_PER_CU, 4)
    if n % 2:
        e.set_tuning(TUNE_SCHEDULE, 2)
    key = rows[exp["clause"]] | (lens[exp["clause"]].astype(np.uint64) << np.uint64(32))
    ids = np.sort(key | (exp["word"].astype(np.uint64) << np.uint64(48)))
    clauses, inv = np.unique(key, return_inverse=True)
    words = np.zeros(clauses.size, np.uint64)
    np.bitwise_or.at(words, inv, np.uint64(1) << exp["word"].astype(np.uint64))
    assert e.sweep(valid) == exp.size
    assert np.array_equal(np.sort(e.hits().view(np.uint64).reshape(-1, 3)[:, 0]), ids)
    for flags in (0, sv.STEP_SCREEN):
        sv.submit(e, valid, records=sv.RECORDS_CLAUSES, flags=flags)
        assert e.step_wait()[0] == clauses.size
        got = e.step_clauses_view().view(np.uint64).reshape(-1, 2)
        got = got[np.argsort(got[:, 0])]
        assert np.array_equal(got[:, 0], clauses) and np.array_equal(got[:, 1], words)


@pytest.mark.parametrize("W", [1, 2, 4])
def test_long_clauses_of_narrow_tables(engine_factory, W):
    """Lengths around the rows read per step past the held literals, most clauses
    with one or two literals that may be non-false anywhere, the last included."""
    rng = np.random.default_rng(4600 + W)
    V = 3000
    lens = rng.permutation(np.repeat([*range(37, 54), 199, 200, 203, 204, 205, 400], 67))
    lens = lens.astype(np.int32)
    off = np.zeros(lens.size + 1, np.int64)
    off[1:] = np.cumsum(lens)
    sigma = rng.random(V) < 0.5
    v = rng.integers(0, V, size=int(off[-1]))
    false = np.ones(v.size, bool)
    false[off[:-1] + rng.integers(0, lens)] = rng.random(lens.size) < 0.3
    false[off[1:] - 1] &= rng.random(lens.size) < 0.8
    lits = (2 * v + (false == sigma[v])).astype(np.uint32)
    one = np.where(sigma, ALL, np.uint64(0))
    is_def, is_true = np.full((V, W), ALL), np.repeat(one[:, None], W, axis=1)
    bit = np.uint64(1) << rng.integers(0, 64, size=(V, W), dtype=np.uint64)
    is_def ^= np.where(rng.random((V, W)) < 0.05, bit, np.uint64(0))
    undef = rng.random(V) < 0.3  # half of them: undefined in the upper slots
    is_def[undef] &= np.uint64(0xFFFFFFFF)
    is_true &= is_def
    valid = np.full(W, ALL)
    exp = orc.sweep(off, lits, is_def, is_true, valid)
    assert (exp["unit_mask"] != 0).sum() > 100 and (exp["false_mask"] != 0).sum() > 100
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    c = exp["clause"]
    want = np.empty((exp.size, 3), np.uint64)
    want[:, 0] = (rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                  | (exp["word"].astype(np.uint64) << np.uint64(48)))
    want[:, 1], want[:, 2] = exp["false_mask"], exp["unit_mask"]
    want = want[np.argsort(want[:, 0])]
    print(f"{W} words: {lens.size} clauses, {exp.size} records", flush=True)
    assert e.sweep(valid) == exp.size
    got = e.hits().view(np.uint64).reshape(-1, 3)
    assert np.array_equal(got[np.argsort(got[:, 0])], want)
    for flags in (0, sv.STEP_SCREEN):
        sv.submit(e, valid, flags=flags)
        assert e.step_wait()[0] == exp.size
        got = e.step_hits_view().view(np.uint64).reshape(-1, 3)
        assert np.array_equal(got[np.argsort(got[:, 0])], want)
