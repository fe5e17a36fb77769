"""Explicit runs and batches of branching neurites with their elements in registers, at
the sizes where units, groups and halos begin: bit-identical to the same steps taken one
launch at a time (the operations and their order are the same), and within the FP64 bar
of the oracle."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import TOL_V, max_abs_diff
from test_explicit_plan import _random_tree, tree_host

pytestmark = pytest.mark.gpu


def _tree(orc, depth, hh=(1,), seed=0):
    n = _random_tree(orc, depth, seed).N
    return _random_tree(orc, depth, seed, hh=[k % n for k in hh], inputs=(1, 20, n - 4))


def _stepped(nrt, p, steps, a0, a1):
    with nrt.Solver(p, kind=nh.EXPLICIT) as s:
        for i in range(1, steps + 1):
            s.update(a0 <= i <= a1)
            s.calculate()
        return s.snapshot()


# (units of 8 elements, 192 per group: depth 5 has one group, 6 a few, 9 about twenty; HH
# elements at the root, in the middle of a strand, at a branch point and its daughters)
@pytest.mark.parametrize("depth,hh", [(2, (1,)), (3, ()), (3, (1, 2, 3)), (5, (1, 40)), (6, (1,)),
                                      (7, (1, 2, 30, 31, 3100, 3101)), (9, (1, 5)),
                                      (9, (1, 3000, 6000, 9000, 12000, 15000, 18000, 21000))])
def test_runs_equal_single_steps(depth, hh, nrt, orc):
    p = _tree(orc, depth, hh)
    print(f"[gpu-case] tree N={p.N} hh={hh}", flush=True)
    assert not isinstance(tree_host(p, 192, 0, 0, 0), str)
    chunks = (1, 15, 16, 17, 2, 33, 3, 40)  # steps of each run: within and across exchanges
    where = [0, 1, p.N // 2, p.N - 1]
    with nrt.Solver(p, kind=nh.EXPLICIT) as s, nrt.Solver(p, kind=nh.EXPLICIT) as one:
        step = 1
        for i, c in enumerate(chunks):
            k = where[i % 4]
            tr = s.run(step, c, 3, 50, trace_elem=k, interval=0)
            # (one or two steps are a launch each above 8,192 elements)
            assert s.stats()["kernel_launches"] == (c if c <= 2 and p.N > 8192 else 1)
            for j in range(c):
                one.update(3 <= step + j <= 50)
                one.calculate()
                assert tr[j] == one.snapshot()[k]
            step += c
            assert np.array_equal(s.snapshot(), one.snapshot())
        # the two kinds of step may follow each other
        for t in (s, one):
            t.update(True)
            t.calculate()
        s.run(step + 1, 20, 1, 0)
        for _ in range(20):
            one.update(False)
            one.calculate()
        v = s.snapshot()
        assert np.array_equal(v, one.snapshot())
    ref = orc.Explicit(p)
    ref.run(1, step - 1, 3, 50)
    ref.run(step, 1, step, step)
    ref.run(step + 1, 20, 1, 0)
    assert max_abs_diff(v, ref.snapshot()) <= TOL_V


@pytest.mark.parametrize("tree", [0, 240, 480, 4000])
def test_dense_branching(tree, nrt):
    """Segments of a few elements: exchanges every 4 steps (a run ends within, at and after
    one), alone and in a batch."""
    p, _ = nrt.setup(wl.sweep_tree(tree)[0], dT=None, dt_factor=0.8)
    with nrt.Solver(p, kind=nh.EXPLICIT) as s, nrt.Batch(kind=nh.EXPLICIT) as b:
        slot = b.add(p, 1000, 1, 20)
        step = 0
        for c in (3, 4, 5, 30):
            s.run(step + 1, c, 1, 20)
            b.step(c)
            assert b.stats()["launches"] > 0 and s.stats()["kernel_launches"] == 1
            step += c
        v = _stepped(nrt, p, step, 1, 20)
        assert np.array_equal(s.snapshot(), v) and np.array_equal(b.snapshot(slot), v)


def test_batch_slots(nrt, orc):
    """Slots in registers (one group and several) beside slots stepped by launches (more
    HH elements than the form takes), joining, ending and leaving at different steps."""
    probs = [_tree(orc, d, hh, seed) for seed, (d, hh) in enumerate(
        [(3, (1,)), (7, (1, 40)), (9, (1,)), (4, range(1, 12)), (5, (1,)), (8, (1, 2, 3))])]
    steps = [60, 200, 90, 200, 37, 70]
    with nrt.Batch(kind=nh.EXPLICIT) as b:
        ids = [b.add(p, n, 2, 45, 1, 2) for p, n in list(zip(probs, steps))[:4]]
        b.step(25)
        ids += [b.add(p, n, 2, 45, 1, 2) for p, n in list(zip(probs, steps))[4:]]
        b.step(1)
        mid = b.snapshot(ids[2])
        assert np.array_equal(mid, _stepped(nrt, probs[2], 26, 2, 45))
        b.step(50)
        b.remove(ids[3])
        b.step(24)
        done = [60, 100, 90, None, 37, 70]
        for i, n in enumerate(done):
            if n is None:
                continue
            n = min(n, 75) if i >= 4 else n
            assert b.info(ids[i])["steps_done"] == n
            v = b.snapshot(ids[i])
            assert np.array_equal(v, _stepped(nrt, probs[i], n, 2, 45))
            with nrt.Solver(probs[i], kind=nh.EXPLICIT) as s:
                assert np.array_equal(b.trace(ids[i]), s.run(1, n, 2, 45, trace_elem=1, interval=2))


@pytest.mark.parametrize("depth,hh", [(3, ()), (5, (1,)), (7, (1,))])
def test_diverging_runs(depth, hh, nrt, orc):
    """An unstable time step: infinities and NaN come up where the steps alone have them."""
    p = _tree(orc, depth, hh)
    p.dT = 6 * p.dT
    seen = set()
    with nrt.Solver(p, kind=nh.EXPLICIT) as s, nrt.Solver(p, kind=nh.EXPLICIT) as one, \
            nrt.Batch(kind=nh.EXPLICIT) as b:
        slot = b.add(p, 10000, 1, 20)
        for k in range(20):  # (the oracle: NaN from the eighth step on)
            s.run(1 + 3 * k, 3, 1, 20)
            b.step(3)
            for i in range(1 + 3 * k, 4 + 3 * k):
                one.update(i <= 20)
                one.calculate()
            v = one.snapshot()
            seen |= {bool(np.isfinite(v).all())}
            assert np.array_equal(s.snapshot(), v, equal_nan=True), k
            assert np.array_equal(b.snapshot(slot), v, equal_nan=True), k
    assert seen == {True, False}


def test_bounded_wait(nrt, orc):
    """With a wait of one poll the exchanges give up; runs and batches are then where they
    were before, and go on from there with the normal bound."""
    p = _tree(orc, 9)
    want = _stepped(nrt, p, 130, 1, 20)
    with nrt.Solver(p, kind=nh.EXPLICIT) as s, nrt.Batch(kind=nh.EXPLICIT) as b:
        slot = b.add(p, 1000, 1, 20)
        s.run(1, 30, 1, 20)
        b.step(30)
        before = s.snapshot()
        os.environ["NRT_SPIN_LIMIT"] = "1"
        try:
            with pytest.raises(nh.NrtError):
                s.run(31, 800, 1, 20)
            with pytest.raises(nh.NrtError):
                b.step(800)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        assert np.array_equal(s.snapshot(), before)
        assert np.array_equal(b.snapshot(slot), before)
        s.run(31, 100, 1, 20)
        b.step(100)
        assert np.array_equal(s.snapshot(), want)
        assert np.array_equal(b.snapshot(slot), want)
