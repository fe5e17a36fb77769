"""Single-step calls of explicit batches, between calls of several steps: bit-identical to the
same steps by a solver of each problem, probes and stimulus windows included."""
import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from test_explicit_tree_gpu import _stepped, _tree

pytestmark = pytest.mark.gpu


def test_single_steps(nrt, orc):
    # one group, several, eight HH elements in units' places apart, segments of a few
    # elements (halo of 4), and a slot that the graph steps
    probs = [_tree(orc, 3, (1,), 0), _tree(orc, 7, (1, 2, 30, 31, 3100, 3101), 1),
             _tree(orc, 9, (), 2), nrt.setup(wl.sweep_tree(0)[0], dT=None, dt_factor=0.8)[0],
             _tree(orc, 4, range(1, 12), 3)]
    probes = [0, 1, 2, 5, 3]
    last = 40
    with nrt.Batch(kind=nh.EXPLICIT) as b:
        ids = [b.add(p, last, 3, 22, k, k % 2) for p, k in zip(probs, probes)]
        done = 0
        for k in (1, 1, 1, 17, 1, 4, 1, 1, 3, 1, 1, 8):
            b.step(k)
            done += k
            if done < 24 or done >= last:
                for i, p in zip(ids, probs):
                    assert np.array_equal(b.snapshot(i), _stepped(nrt, p, done, 3, 22)), (i, done)
        for i, p, k in zip(ids, probs, probes):
            assert b.info(i)["steps_done"] == last
            with nrt.Solver(p, kind=nh.EXPLICIT) as s:
                tr = s.run(1, last, 3, 22, trace_elem=k, interval=k % 2)
            assert np.array_equal(b.trace(i), tr)
