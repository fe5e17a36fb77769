"""Long runs that take most of the device give it back at intervals: they are several
launches with the results and probe samples of one, and runs of other threads do not wait
for their ends."""
import threading
import time

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl

pytestmark = pytest.mark.gpu
FORMS = {"direct": dict(kind=nh.IMPLICIT, krylov=nh.DIRECT), "explicit": dict(kind=nh.EXPLICIT)}


def _tree(nrt, depth, form):
    geom, run = wl.random_tree(wl.seed_for(3, 2), depth=depth)
    dt = {"dT": run.dT} if form == "direct" else {"dT": None, "dt_factor": 0.8}
    return nrt.setup(geom, **dt)[0]


# (a launch: 1,024 steps of the direct solve, 8,192 explicit ones)
@pytest.mark.parametrize("form,steps", [("direct", 2500), ("explicit", 17000)])
def test_pieces_are_one_run(form, steps, nrt):
    p = _tree(nrt, 13, form)
    with nrt.Solver(p, **FORMS[form]) as s, nrt.Solver(p, **FORMS[form]) as one:
        tr = s.run(1, steps, 5, steps - 100, trace_elem=1, interval=6)
        assert s.stats()["kernel_launches"] == 3 and s.stats()["steps"] == steps
        got, done = [], 0
        while done < steps:  # whole sample periods each
            n = min(700, steps - done)
            got.append(one.run(1 + done, n, 5, steps - 100, trace_elem=1, interval=6))
            assert one.stats()["kernel_launches"] == 1
            done += n
        assert len(tr) == steps // 7 and np.array_equal(tr, np.concatenate(got))
        assert np.array_equal(s.snapshot(), one.snapshot())


def test_batch_pieces_are_one_call(nrt):
    """(a launch: 33,333 steps of so few elements)"""
    p, steps = _tree(nrt, 4, "explicit"), 60000
    with nrt.Solver(p, **FORMS["explicit"]) as s, nrt.Batch(**FORMS["explicit"]) as b:
        tr = s.run(1, steps, 5, 40000, trace_elem=1, interval=6)
        slots = [b.add(p, n, 5, 40000, 1, 6) for n in (steps, 35000, steps + 10)]
        b.step(steps)
        assert b.stats()["launches"] == 2
        for i, n in zip(slots, (steps, 35000, steps)):
            assert b.info(i)["steps_done"] == n
            assert np.array_equal(b.trace(i), tr[:n // 7])
        for i in (slots[0], slots[2]):
            assert np.array_equal(b.snapshot(i), s.snapshot())


def test_a_small_run_beside_a_long_one(nrt):
    large, small = _tree(nrt, 14, "direct"), _tree(nrt, 6, "direct")
    with nrt.Solver(large, **FORMS["direct"]) as a, nrt.Solver(small, **FORMS["direct"]) as b:
        b.run(1, 50, 1, 9)
        a.run(1, 50, 1, 9)
        t0 = time.perf_counter()
        a.run(51, 20000, 1, 9)
        long = time.perf_counter() - t0
        t = threading.Thread(target=lambda: a.run(20051, 20000, 1, 9))
        t.start()
        time.sleep(long / 10)
        t0 = time.perf_counter()
        b.run(51, 50, 1, 9)
        waited = time.perf_counter() - t0
        ended = not t.is_alive()
        t.join()
        # (a launch of the long run is a twentieth of it)
        assert not ended and waited < 0.5 * long
