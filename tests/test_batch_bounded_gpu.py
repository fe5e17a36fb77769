"""Batches whose slots span several workgroups, with a wait that ends early: no slot passes
off rows of two steps for a result, slots of an explicit batch stay in step with each other,
and the batch goes on with the normal bound."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import ghost_mask, max_abs_diff
from test_explicit_tree_gpu import _stepped, _tree

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)


def test_explicit_slots_stay_in_step(nrt, orc):
    """Slots in registers (one group and several) beside slots stepped by launches (more HH
    elements than the form takes)."""
    probs = [_tree(orc, 9, (1,), 2), _tree(orc, 4, range(1, 12), 3), _tree(orc, 3, (1,), 0)]
    with nrt.Batch(kind=nh.EXPLICIT) as b:
        ids = [b.add(p, 1000, 1, 20) for p in probs]
        b.step(30)
        before = [b.snapshot(i) for i in ids]
        launches = b.stats()["launches"]
        os.environ["NRT_SPIN_LIMIT"] = "0"
        try:
            with pytest.raises(nh.NrtError):
                b.step(800)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        assert b.stats()["launches"] >= launches
        for i, v in zip(ids, before):
            assert b.info(i)["steps_done"] == 30 and np.array_equal(b.snapshot(i), v)
        late = b.add(probs[1], 1000, 1, 20)  # joins where the batch stands
        b.step(100)
        for i, p, n in [*zip(ids, probs, (130, 130, 130)), (late, probs[1], 100)]:
            assert b.info(i)["steps_done"] == n
            assert np.array_equal(b.snapshot(i), _stepped(nrt, p, n, 1, 20))


def test_implicit_slots_report(nrt):
    """Single steps with one poll allowed: whichever workgroups of a slot give up, the slot
    says so unless every row took the step."""
    geom, run = wl.random_tree(wl.seed_for(3, 9), depth=10, amp=2e-9)
    p, _ = nrt.setup(geom, dT=run.dT)
    m = ghost_mask(p)
    with nrt.Solver(p, **DIRECT) as s:
        s.run(1, 1, 1, 20)
        want = s.snapshot()
        assert s.stats()["num_blocks"] > 1
    with nrt.Batch(**DIRECT) as b:
        ids = [b.add(p, 10, 1, 20) for _ in range(200)]
        os.environ["NRT_SPIN_LIMIT"] = "0"
        try:
            b.step(1)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        failed = 0
        for i in ids:
            if b.info(i)["status"] != 0:
                failed += 1
            else:
                assert max_abs_diff(b.snapshot(i), want, m) <= 1e-12, i
        assert failed > 0
