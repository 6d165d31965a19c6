"""Sweeps and steps whose records overflow their hit buffer, where they are
screened: steps of at most 8 words, whose own kernels keep the screening entries
current, over a halt, the re-run and the replay of the step behind; and sweeps
that the device chose to screen, plain ones and steps', re-run with the same
choice.
"""
import numpy as np
import pytest

import _oracle as orc
from gpusharesat_amd import serving as sv
from gpusharesat_amd.engine import TUNE_MAX_HIT_CHUNKS, VAR_UPDATE_DTYPE
from test_step_gpu import run_steps

pytestmark = pytest.mark.gpu

ALL = np.uint64(0xFFFFFFFFFFFFFFFF)


@pytest.mark.parametrize("read_in_flight", [False, True])
@pytest.mark.parametrize("W", [1, 2, 4, 8])
def test_overflowing_screened_steps_of_few_words(engine_factory, W, read_in_flight):
    """Every fifth step is not screened: the next one rebuilds the entries."""
    run_steps(engine_factory, seed=2100 + W, V=2000, W=W, nsteps=9, n_new=900, maxlen=12,
              n_ups=300 * W, pipelined=True, screen=lambda k: k % 5 != 3, uniform=True,
              uniform_init=True, tuning=((TUNE_MAX_HIT_CHUNKS, 1),),
              read_in_flight=read_in_flight)


@pytest.mark.parametrize("W, n", [(8, 450_000), (16, 450_000), (32, 160_000), (64, 80_000)])
def test_sweeps_chosen_to_be_screened_overflow(engine_factory, W, n):
    rng = np.random.default_rng(2200 + W)
    V = 400
    sigma = rng.random(V) < 0.5
    lens = rng.integers(1, 6, size=n).astype(np.int32)
    v = rng.integers(0, V, size=int(lens.sum()))
    lits = (2 * v + ((rng.random(v.size) < 0.15) == sigma[v])).astype(np.uint32)  # mostly true
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(lens)
    is_def = np.full((V, W), ALL)
    is_true = np.repeat(np.where(sigma, ALL, np.uint64(0))[:, None], W, axis=1)
    mixed = rng.random(V) < 0.1
    is_true[mixed] = rng.integers(0, 1 << 63, size=(int(mixed.sum()), W), dtype=np.uint64)
    valid = np.full(W, ALL)
    valid[-1] = np.uint64(0x7FFFFFFFFFFFFF0F)
    last = np.full(W, 63, np.int8)
    last[-1] = 62
    e = engine_factory()
    rows = e.append(lits, lens).astype(np.uint64)
    e.reset_assignments(V, W)
    e.upload(is_def, is_true)
    e.set_tuning(TUNE_MAX_HIT_CHUNKS, 1)

    def expected():
        exp = orc.sweep(off, lits, is_def, is_true, valid)
        c = exp["clause"]
        return np.sort(rows[c] | (lens[c].astype(np.uint64) << np.uint64(32))
                       | (exp["word"].astype(np.uint64) << np.uint64(48)))

    want = expected()
    print(f"{W} words: {want.size} records", flush=True)
    assert want.size > 20_000  # many chunks
    assert e.sweep(valid) == want.size and e.screened() == 1
    assert np.array_equal(np.sort(e.hits().view(np.uint64).reshape(-1, 3)[:, 0]), want)
    # steps, two in flight, each changing 200 cells and rolling them forward
    wants = []
    for k in range(5):
        cells = np.unique(rng.integers(0, V * W, size=200))
        ups = np.zeros(cells.size, VAR_UPDATE_DTYPE)
        ups["var"], ups["word"] = cells // W, cells % W
        ups["is_def"] = ALL
        ups["is_true"] = rng.integers(0, 1 << 63, size=cells.size, dtype=np.uint64)
        print(f"step {k}", flush=True)
        sv.submit(e, valid, ups=ups, last_pos=last, records=sv.RECORDS_IDS)
        is_def.ravel()[cells], is_true.ravel()[cells] = ups["is_def"], ups["is_true"]
        wants.append(expected())
        bit = (ups["is_true"] >> last[ups["word"]].astype(np.uint64)) & np.uint64(1)
        is_true.ravel()[cells] = np.where(bit != 0, ALL, np.uint64(0))
        if k > 0:
            assert e.step_wait()[0] == wants[k - 1].size
            assert np.array_equal(np.sort(e.step_ids_view().view(np.uint64).ravel()), wants[k - 1])
    assert e.step_wait()[0] == wants[-1].size and e.screened() == 1
    assert np.array_equal(np.sort(e.step_ids_view().view(np.uint64).ravel()), wants[-1])
    assert e.step_stats()["reruns"] >= 5
    d, t = e.download()
    assert np.array_equal(d, is_def) and np.array_equal(t, is_true)
