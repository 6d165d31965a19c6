"""Screened steps (GSS_STEP_SCREEN) whose words mostly hold one value in all
slots, against the oracle: literals known from the screening entries alone,
true, false or undefined in all slots of a word group, beside literals whose
rows have to be read, at clause lengths around the positions the check keeps
apart (31), over steps that change the table and roll it forward.  And plain
sweeps of so many clauses that they may be screened too, over tables whose slots
agree, differ, or agree for a share of the variables.
"""
import numpy as np
import pytest

import _oracle as orc
from gpusharesat_amd import serving as sv
from gpusharesat_amd.engine import VAR_UPDATE_DTYPE

pytestmark = pytest.mark.gpu

ALL = np.uint64(0xFFFFFFFFFFFFFFFF)
V = 400


def planes(rng, words, sigma):
    """Most variables one value in a word (true under sigma, false, undefined),
    the same in its neighbours more often than not; a few differ in a slot."""
    d = np.repeat(rng.random((V, (words + 3) // 4)) < 0.95, 4, axis=1)[:, :words]
    t = np.where(rng.random((V, words)) < 0.99, sigma[:, None], ~sigma[:, None])
    is_def = np.where(d, ALL, np.uint64(0))
    is_true = np.where(d & t, ALL, np.uint64(0))
    bit = np.uint64(1) << rng.integers(0, 64, size=(V, words), dtype=np.uint64)
    is_def ^= np.where(rng.random((V, words)) < 0.02, bit, np.uint64(0))
    is_true ^= np.where(rng.random((V, words)) < 0.02, bit, np.uint64(0))
    return is_def, is_true & is_def


@pytest.mark.parametrize("W, used", [(1, [1] * 4), (2, [2] * 4), (4, [4] * 4), (8, [8] * 4),
                                     (16, [16] * 4), (32, [32] * 4), (64, [64] * 4),
                                     (16, [4, 4, 16, 9, 9]), (32, [17, 17, 8, 32, 32]),
                                     (64, [3, 3, 34, 34, 20, 64, 64])])
def test_words_of_one_value(engine_factory, W, used):
    """`used` = words with valid slots at each step; updates go to any word."""
    rng = np.random.default_rng(500 + W)
    sigma = rng.random(V) < 0.5
    lens = np.concatenate([np.full(70, n, np.int32)
                           for n in [*range(1, 9), 16, 30, 31, 32, 33, 34, 64, 130]])
    v = rng.integers(0, V, size=int(lens.sum()))
    false = rng.random(v.size) > 0.5 / np.repeat(lens, lens)
    lits = (2 * v + (false == sigma[v])).astype(np.uint32)
    off = np.zeros(lens.size + 1, np.int64)
    off[1:] = np.cumsum(lens)
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    is_def, is_true = planes(rng, W, sigma)
    e.upload(is_def, is_true)
    units = 0
    for step, n_used in enumerate(used):
        ups = np.zeros(0, VAR_UPDATE_DTYPE)
        if step:  # changed words, rolled forward by the step before
            cells = np.unique(rng.integers(0, V * W, size=V * W // 8))
            nd, nt = planes(rng, W, sigma)
            ups = np.zeros(cells.size, VAR_UPDATE_DTYPE)
            ups["var"], ups["word"] = cells // W, cells % W
            ups["is_def"], ups["is_true"] = nd.ravel()[cells], nt.ravel()[cells]
            is_def.ravel()[cells], is_true.ravel()[cells] = ups["is_def"], ups["is_true"]
        valid = np.full(W, ALL)
        valid[-1] = np.uint64(0x7FFFFFFFFFFFFF0F)
        valid[n_used:] = 0
        if n_used > 2:
            valid[step % n_used] = 0
        last = np.full(W, 63, np.int8)
        last[-1] = 62
        exp = orc.sweep(off, lits, is_def, is_true, valid)
        units += int((exp["unit_mask"] != 0).sum())
        print(f"{W} words, step {step}: {ups.size} updates, {exp.size} records", flush=True)
        sv.submit(e, valid, ups=ups, last_pos=last, flags=sv.STEP_SCREEN)
        assert e.step_wait()[0] == exp.size
        got = e.step_hits_view().view(np.uint64).reshape(-1, 3)
        want = np.empty((exp.size, 3), np.uint64)
        c = exp["clause"]
        want[:, 0] = (rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                      | (exp["word"].astype(np.uint64) << np.uint64(48)))
        want[:, 1], want[:, 2] = exp["false_mask"], exp["unit_mask"]
        assert np.array_equal(got[np.argsort(got[:, 0])], want[np.argsort(want[:, 0])])
        for k in range(ups.size):  # the roll forward: the word takes its last slot's value
            x, w = int(ups["var"][k]), int(ups["word"][k])
            b = np.uint64(int(last[w]))
            one = np.uint64(1)
            is_true[x, w] = ALL if (is_true[x, w] >> b) & one else np.uint64(0)
            is_def[x, w] = ALL if (is_def[x, w] >> b) & one else np.uint64(0)
    assert units > 50


@pytest.mark.parametrize("agree", [1.0, 0.42, 0.38, 0.0])
@pytest.mark.parametrize("W, n", [(8, 450_000), (16, 450_000), (32, 160_000), (64, 80_000)])
def test_plain_sweeps_that_may_be_screened(engine_factory, W, n, agree):
    rng = np.random.default_rng(W + int(100 * agree))
    sigma = rng.random(V) < 0.5
    lens = rng.integers(1, 6, size=n).astype(np.int32)
    v = rng.integers(0, V, size=int(lens.sum()))
    # mostly true literals: few records
    lits = (2 * v + ((rng.random(v.size) < 0.15) == sigma[v])).astype(np.uint32)
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(lens)
    is_def = np.full((V, W), ALL)
    is_true = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
    mixed = rng.random(V) >= agree
    is_def[mixed] &= rng.integers(0, 1 << 63, size=(int(mixed.sum()), W), dtype=np.uint64)
    is_true &= is_def
    valid = np.full(W, ALL)
    valid[1] = 0
    valid[-1] = np.uint64(0x7FFFFFFFFFFFFF0F)
    exp = orc.sweep(off, lits, is_def, is_true, valid)
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    print(f"{W} words, {agree} agree: {exp.size} records", flush=True)
    want = np.empty((exp.size, 3), np.uint64)
    c = exp["clause"]
    want[:, 0] = (rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                  | (exp["word"].astype(np.uint64) << np.uint64(48)))
    want[:, 1], want[:, 2] = exp["false_mask"], exp["unit_mask"]
    want = want[np.argsort(want[:, 0])]
    for _ in range(2):
        assert e.sweep(valid) == exp.size
        got = e.hits().view(np.uint64).reshape(-1, 3)
        assert np.array_equal(got[np.argsort(got[:, 0])], want)
    # unscreened steps' sweeps may be too
    sv.submit(e, valid)
    assert e.step_wait()[0] == exp.size
    got = e.step_hits_view().view(np.uint64).reshape(-1, 3)
    assert np.array_equal(got[np.argsort(got[:, 0])], want)
    sv.submit(e, valid, records=sv.RECORDS_IDS)
    assert e.step_wait()[0] == exp.size
    assert np.array_equal(np.sort(e.step_ids_view().view(np.uint64).ravel()), want[:, 0])
    sv.submit(e, valid, records=sv.RECORDS_CLAUSES)
    assert e.step_wait()[0] == np.unique(c).size
    got = e.step_clauses_view().view(np.uint64).reshape(-1, 2)
    words = np.bitwise_count(got[:, 1]).sum()
    assert words == exp.size and np.unique(got[:, 0]).size == got.shape[0]


@pytest.mark.parametrize("variables", [1, 3, 403])
@pytest.mark.parametrize("W, n", [(8, 450_000), (16, 450_000), (32, 160_000), (64, 80_000)])
def test_screening_tables_of_odd_sizes(engine_factory, W, n, variables):
    """Fewer variables than a wave's turn over the table, and a last turn in part:
    plain sweeps that may be screened, and screened steps."""
    rng = np.random.default_rng(W + variables)
    lens = rng.integers(1, 4, size=n).astype(np.int32)
    lits = rng.integers(0, 2 * variables, size=int(lens.sum())).astype(np.uint32)
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(lens)
    is_def = np.full((variables, W), ALL)
    is_true = np.repeat(np.where(rng.random(variables) < 0.5, ALL, np.uint64(0))[:, None], W, axis=1)
    is_def[-1, W // 2:] = 0  # the last variable: undefined from half of the words on
    is_true &= is_def
    valid = np.zeros(W, np.uint64)
    valid[[0, W // 2, W - 1]] = [3, 1 << 63, 1]
    exp = orc.sweep(off, lits, is_def, is_true, valid)
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(variables, W)
    e.upload(is_def, is_true)
    c = exp["clause"]
    want = np.sort(rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                   | (exp["word"].astype(np.uint64) << np.uint64(48)))
    print(f"{W} words, {variables} variables: {exp.size} records", flush=True)
    assert e.sweep(valid) == exp.size
    assert np.array_equal(np.sort(e.hits().view(np.uint64).reshape(-1, 3)[:, 0]), want)
    for flags in (0, sv.STEP_SCREEN):
        sv.submit(e, valid, records=sv.RECORDS_IDS, flags=flags)
        assert e.step_wait()[0] == exp.size
        assert np.array_equal(np.sort(e.step_ids_view().view(np.uint64).ravel()), want)


@pytest.mark.parametrize("agree", [True, False])
@pytest.mark.parametrize("W, used", [(8, 1), (16, 2), (16, 3), (32, 4), (64, 8), (64, 17)])
def test_choice_looks_at_the_words_in_use(engine_factory, W, used, agree):
    """Few words with a valid slot, whose slots agree beside words that hold
    nothing, or differ beside words that hold one value: what the other words hold
    does not count."""
    rng = np.random.default_rng(70 + W + used)
    n = 900_000
    sigma = rng.random(V) < 0.5
    lens = rng.integers(3, 6, size=n).astype(np.int32)
    v = rng.integers(0, V, size=int(lens.sum()))
    lits = (2 * v + ((rng.random(v.size) < 0.15) == sigma[v])).astype(np.uint32)
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(lens)
    one = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
    is_def, is_true = np.full((V, W), ALL), one.copy()
    if agree:
        is_def[:, used:] = 0
    else:
        is_true[:, :used] = rng.integers(0, 1 << 63, size=(V, used), dtype=np.uint64)
    is_true &= is_def
    valid = np.zeros(W, np.uint64)
    valid[:used] = ALL
    valid[used - 1] = np.uint64(0x7FFFFFFFFFFFFF0F)
    exp = orc.sweep(off, lits, is_def, is_true, valid)
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    c = exp["clause"]
    want = np.sort(rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                   | (exp["word"].astype(np.uint64) << np.uint64(48)))
    print(f"{W} words, {used} in use: {exp.size} records", flush=True)
    assert e.sweep(valid) == exp.size
    assert np.array_equal(np.sort(e.hits().view(np.uint64).reshape(-1, 3)[:, 0]), want)
    assert e.screened() == int(agree)
    sv.submit(e, valid, records=sv.RECORDS_IDS)
    assert e.step_wait()[0] == exp.size
    assert e.screened() == int(agree)
    assert np.array_equal(np.sort(e.step_ids_view().view(np.uint64).ravel()), want)


@pytest.mark.parametrize("W, n", [(8, 450_000), (16, 450_000), (32, 160_000), (64, 80_000)])
@pytest.mark.parametrize("variables", [60, 128, 3001])
def test_choice_follows_the_share_of_known_variables(engine_factory, W, n, variables):
    """Tables of which 20 or 60 % of the variables hold one value in all slots, the
    threshold lying at 40: 128 variables in turn are looked at, and of 16 such
    samples none is 20 points off (less than one in 10^4, at 60 variables the whole
    table)."""
    rng = np.random.default_rng(W + variables)
    lens = rng.integers(5, 8, size=n).astype(np.int32)
    sigma = rng.random(variables) < 0.5
    v = rng.integers(0, variables, size=int(lens.sum()))
    e = engine_factory()
    e.append((2 * v + ~sigma[v]).astype(np.uint32), lens)  # true where known
    e.reset_assignments(variables, W)
    is_def = np.full((variables, W), ALL)
    for k in range(16):
        share = (0.2, 0.6)[k % 2]
        mixed = rng.permutation(variables) >= share * variables
        is_true = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
        is_true[mixed] = rng.integers(0, 1 << 63, size=(int(mixed.sum()), W), dtype=np.uint64)
        e.upload(is_def, is_true)
        e.sweep(np.full(W, ALL))
        assert e.screened() == k % 2, (k, share)


@pytest.mark.parametrize("W, n, known", [(1, 470_000, 0.3), (2, 470_000, 0.9), (4, 3000, 0.3),
                                         (4, 470_000, 0.6), (8, 20_000, 0.9), (16, 120_000, 0.0),
                                         (16, 470_000, 0.5), (32, 40_000, 0.7), (64, 30_000, 0.0),
                                         (64, 100_000, 0.8)])
def test_screened_steps_of_mostly_false_clauses(engine_factory, W, n, known):
    """Clauses of 1 to 60 literals, most of them false, that the entries leave open
    in some groups, most or all, passes of 64 clauses whole and split among the
    waves: the records of a step that is not screened."""
    rng = np.random.default_rng(900 + W + n)
    variables = 5000
    lens = np.where(rng.random(n) < 0.9, rng.integers(1, 20, size=n),
                    rng.integers(20, 61, size=n)).astype(np.int32)
    sigma = rng.random(variables) < 0.5
    v = rng.integers(0, variables, size=int(lens.sum()))
    false = rng.random(v.size) < np.repeat(1.0 - 1.0 / (1.0 + lens), lens)
    lits = (2 * v + (false == sigma[v])).astype(np.uint32)
    e = engine_factory()
    e.append(lits, lens)
    e.reset_assignments(variables, W)
    is_true = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
    is_def = np.full((variables, W), ALL)
    bit = np.uint64(1) << rng.integers(0, 64, size=(variables, W), dtype=np.uint64)
    differ = rng.random((variables, W)) >= known
    is_true ^= np.where(differ, bit, np.uint64(0))
    is_def ^= np.where(differ & (rng.random((variables, W)) < 0.5), bit, np.uint64(0))
    e.upload(is_def, is_true & is_def)
    valid = np.full(W, ALL)
    valid[-1] = np.uint64(0x7FFFFFFFFFFFFF0F)
    if W > 2:
        valid[1] = 0
    for form, view, words in ((sv.RECORDS_FULL, e.step_hits_view, 3),
                              (sv.RECORDS_CLAUSES, e.step_clauses_view, 2)):
        got = []
        for flags in (0, sv.STEP_SCREEN):
            sv.submit(e, valid, records=form, flags=flags)
            e.step_wait()
            r = view().view(np.uint64).reshape(-1, words).copy()
            got.append(r[np.argsort(r[:, 0])])
        print(f"{W} words, {n} clauses: {got[0].shape[0]} records", flush=True)
        assert got[0].shape[0] > 100 and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("false, chosen", [(0.1, 1), (0.95, 0)])
@pytest.mark.parametrize("W, n", [(8, 450_000), (16, 450_000), (32, 160_000), (64, 80_000)])
def test_choice_looks_at_the_clauses(engine_factory, W, n, false, chosen):
    """Tables of which 60 % of the variables are known: enough where most literals
    are true, so that hardly a clause stays open; not where one in twenty is (seven
    in ten clauses of 8 to 14 literals then do, at 0.4 rows and a third per literal
    three times the threshold)."""
    rng = np.random.default_rng(W)
    variables = 3001
    lens = rng.integers(8, 15, size=n).astype(np.int32)
    sigma = rng.random(variables) < 0.5
    v = rng.integers(0, variables, size=int(lens.sum()))
    lits = (2 * v + ((rng.random(v.size) < false) == sigma[v])).astype(np.uint32)
    e = engine_factory()
    e.append(lits, lens)
    e.reset_assignments(variables, W)
    is_true = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
    mixed = rng.permutation(variables) >= 0.6 * variables
    is_true[mixed] = rng.integers(0, 1 << 63, size=(int(mixed.sum()), W), dtype=np.uint64)
    e.upload(np.full((variables, W), ALL), is_true)
    valid = np.full(W, ALL)
    hits = e.sweep(valid)
    assert e.screened() == chosen
    sv.submit(e, valid, records=sv.RECORDS_IDS)
    assert e.step_wait()[0] == hits and e.screened() == chosen
