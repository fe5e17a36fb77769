"""Batches whose slots span several workgroups, with a wait that ends early: no slot passes
off rows of two steps for a result."""
import os

import pytest

import neurite_hip as nh
import workloads as wl
from common import ghost_mask, max_abs_diff

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)


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
