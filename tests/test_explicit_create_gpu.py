"""Creation of large explicit handles, whose plan is made beside the rest of it: by several
threads at once, and refused for a problem that only the rest finds wrong."""
import threading

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl

pytestmark = pytest.mark.gpu


def test_several_threads_and_a_refusal(nrt):
    geom, _ = wl.random_tree(wl.seed_for(3, 1), depth=10)
    p, _ = nrt.setup(geom, dT=None, dt_factor=0.8)
    assert p.N > 40000
    with nrt.Solver(p, kind=nh.EXPLICIT) as s:
        s.run(1, 40, 1, 20)
        want = s.snapshot()
    bad = nrt.setup(geom, dT=None, dt_factor=0.8)[0]
    j = int(np.nonzero(bad.branching)[0][-1])
    bad.dl = bad.dl.copy()  # (the two share the geometry's)
    bad.dl[j] = bad.N + 5
    got, refused = [], []

    def work(k):
        if k % 3 == 2:
            try:
                nrt.Solver(bad, kind=nh.EXPLICIT)
            except nh.NrtError:
                refused.append(k)
            return
        with nrt.Solver(p, kind=nh.EXPLICIT) as s:
            s.run(1, 40, 1, 20)
            got.append(s.snapshot())

    threads = [threading.Thread(target=work, args=(k,)) for k in range(9)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(refused) == 3 and len(got) == 6
    assert all(np.array_equal(v, want) for v in got)
