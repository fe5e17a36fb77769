"""Snapshots at the sizes where blocks and staging buffers begin, and by several threads
at once, against the potentials they were made from (no step taken: every bit)."""
import threading

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl

pytestmark = pytest.mark.gpu


def _problem(nrt, n):
    geom, _ = wl.squid_axon(n_comp=n - 2, length=1e-5 * (n - 2))
    geom.material[2:] = 0
    prob, _ = nrt.setup(geom, dT=1e-6)
    prob.potential0 = np.random.default_rng(n).uniform(-0.1, 0.1, n)
    prob.potential1 = prob.potential0.copy()
    return prob


@pytest.mark.parametrize("n", [4, 1024, 1025, 262144, 262145, 524289, 800000])
@pytest.mark.parametrize("opt", [dict(kind=nh.EXPLICIT), dict(kind=nh.IMPLICIT, krylov=nh.DIRECT),
                                 dict(kind=nh.IMPLICIT, krylov=nh.DIRECT, num_blocks=1)])
def test_every_element(n, opt, nrt):
    prob = _problem(nrt, n)
    with nrt.Solver(prob, **opt) as s:
        for _ in range(2):
            assert np.array_equal(s.snapshot(), prob.potential0)


def test_several_threads(nrt):
    probs = [_problem(nrt, n) for n in (700, 5000, 300000, 600000, 12345, 40)]
    bad = []

    def work(p):
        with nrt.Solver(p, kind=nh.IMPLICIT, krylov=nh.DIRECT) as s:
            for _ in range(20):
                if not np.array_equal(s.snapshot(), p.potential0):
                    bad.append(p.N)

    threads = [threading.Thread(target=work, args=(p,)) for p in probs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
