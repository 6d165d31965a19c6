"""HIP runtime calls that are refused (no memory, a failed event) leave the engine
as it was: the next call gives what it gives without the refusal.  Each case runs
in a process of its own, in which tests/cpp/hip_fail.cpp stands in front of the
runtime and refuses the call; nothing reaches the GPU for it.
"""
import pathlib
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = pathlib.Path(__file__).resolve().parent.parent

HEAD = """
import ctypes, sys
import numpy as np
fail = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
fail.hip_fail_set.argtypes = [ctypes.c_int, ctypes.c_size_t, ctypes.c_long, ctypes.c_long]
fail.hip_fail_calls.restype = ctypes.c_long
HOST_MALLOC, MALLOC_ASYNC, EVENT_RECORD = range(3)
from gpusharesat_amd import _lib, engine as en, serving as sv

ALL = np.uint64(0xFFFFFFFFFFFFFFFF)


def refused(call):
    try:
        call()
    except _lib.GssError as x:
        print("refused:", x, flush=True)
    else:
        raise SystemExit("the call was not refused")


def ones(n):
    return np.ones(n, np.int32)
"""


def run_case(tmp_path, body):
    shim = tmp_path / "hip_fail.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared",
                    str(ROOT / "tests" / "cpp" / "hip_fail.cpp"), "-o", str(shim), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", "-c",
                        textwrap.dedent(HEAD) + textwrap.dedent(body) + "\nprint('ok')", str(shim)],
                       cwd=ROOT, capture_output=True, text=True, timeout=100)
    print(r.stdout + r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok")


def test_calls_after_an_error_of_the_callers_own(tmp_path):
    """An error that another HIP call of the thread has left is not taken for one
    of the engine's launches."""
    run_case(tmp_path, """
        hip = ctypes.CDLL("libamdhip64.so.7")
        e = en.Engine(0)
        e.reset_assignments(64, 1)
        e.append(np.full(100, 2, np.uint32), ones(100))
        every = np.full(1, ALL)
        for k in range(7):
            sv.submit(e, every, records=sv.RECORDS_IDS)
            assert e.step_wait()[0] == 100
            if k > 2:
                assert hip.hipMalloc(None, ctypes.c_size_t(16)) != 0
        print("steps done", flush=True)
        for k in range(3):
            assert e.sweep(every) == 100
            assert hip.hipMalloc(None, ctypes.c_size_t(16)) != 0
    """)


def test_sweep_after_a_sweep_that_was_not_queued(tmp_path):
    """A sweep that claimed chunks past its waves' own, one whose first event is
    refused, one without a valid slot: none of the first one's claims is left."""
    run_case(tmp_path, """
        e = en.Engine(0)
        e.reset_assignments(64, 1)
        n = 2_000_000
        e.append(np.full(n, 2, np.uint32), ones(n))  # undefined: a record per clause
        e.set_tuning(en.TUNE_WAVES_PER_CU, 4)  # ~2,000 records a wave: two chunks
        every = np.full(1, ALL)
        assert e.sweep(every) == n
        fail.hip_fail_set(EVENT_RECORD, 0, 0, 1)
        refused(lambda: e.sweep(every))
        assert e.sweep(np.zeros(1, np.uint64)) == 0
        assert e.sweep(every) == n
        assert np.array_equal(np.sort(e.hits()["row"]), np.arange(n))
        fail.hip_fail_set(EVENT_RECORD, 0, 0, 1)
        refused(lambda: e.sweep(every))
        refused(e.hits)
    """)


def test_records_held_while_a_submit_is_refused(tmp_path):
    """A step's records keep their place until its slot is waited for again, also
    where the slot's next submit is refused first."""
    run_case(tmp_path, """
        e = en.Engine(0)
        e.reset_assignments(64, 1)
        every = np.full(1, ALL)
        e.append(np.full(100, 2, np.uint32), ones(100))
        views = []
        for _ in range(2):
            sv.submit(e, every, records=sv.RECORDS_IDS)
            assert e.step_wait()[0] == 100
            views.append(e.step_ids_view())
        held = [v.copy() for v in views]
        # variable 1 true: of the step's records only the new clauses' are left
        ups = np.zeros(5000, en.VAR_UPDATE_DTYPE)
        ups["var"], ups["is_def"], ups["is_true"] = 1, ALL, ALL
        step = lambda: sv.submit(e, every, lits=np.full(50, 6, np.uint32), lens=ones(50), ups=ups,
                                 records=sv.RECORDS_IDS)
        fail.hip_fail_set(MALLOC_ASYNC, 100_000, 0, 1)  # the device copy of the updates
        refused(step)
        step()
        e.sync()
        for v, h in zip(views, held):
            assert np.array_equal(v, h)
        assert e.step_wait()[0] == 50
        assert np.array_equal(np.sort(e.step_ids_view()["row"]), np.arange(100, 150))
    """)


def test_steps_whose_record_buffers_are_not_page_locked(tmp_path):
    """Neither the buffer of few records nor the one for more: the records are
    copied, to pageable memory."""
    run_case(tmp_path, """
        for times in (1, 1000):
            e = en.Engine(0)
            e.reset_assignments(64, 1)
            e.append(np.full(100, 2, np.uint32), ones(100))
            fail.hip_fail_set(HOST_MALLOC, 500_000, 0, times)
            for _ in range(5):
                sv.submit(e, np.full(1, ALL), records=sv.RECORDS_IDS)
                assert e.step_wait()[0] == 100
                assert np.array_equal(np.sort(e.step_ids_view()["row"]), np.arange(100))
            assert e.sweep(np.full(1, ALL)) == 100
            e.close()
    """)


def test_scorer_pass_without_page_locked_memory(tmp_path):
    """Samples and results then take the device's memory; so they do where the
    engine's page-locked limit is below the samples' size."""
    run_case(tmp_path, """
        from gpusharesat_amd import residency as rs
        rng = np.random.default_rng(3)
        n = 3000
        x = rng.normal(0, 1, (n, 12)).astype(np.float32)
        y = (rng.random(n) < 0.3).astype(np.float32)
        e = en.Engine(0)
        e.enable_tags()
        def grad(at_least, times):
            r = rs.Residency(e, 64, seed=3)
            fail.hip_fail_set(HOST_MALLOC, at_least, 0, times)
            out = [r.grad(x[:m], y[:m]) for m in (n // 2, n, 100)]
            r.close()
            return out, fail.hip_fail_calls(HOST_MALLOC)
        want, calls = grad(70_000, 0)
        assert calls > 0
        for at_least in (70_000, 1):
            got, calls = grad(at_least, 1000)
            assert calls > 0
            for a, b in zip(got, want):
                assert a[0] == b[0] and np.array_equal(a[1], b[1])
        e.set_page_locked_limit(70_000)
        got, calls = grad(70_000, 0)
        assert calls == 0
        for a, b in zip(got, want):
            assert a[0] == b[0] and np.array_equal(a[1], b[1])
    """)
