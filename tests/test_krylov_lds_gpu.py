"""A handle keeps its workgroup's LDS when handles of other sizes are made: what a kernel
may ask for is the kernel's, not the handle's."""
import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl

pytestmark = pytest.mark.gpu


# (GMRES: 74 and 56 KB of LDS in the same kernel of 8 rows a thread)
def test_large_handle_after_a_smaller_one(nrt):
    opt = dict(kind=nh.IMPLICIT, krylov=nh.GMRES, restart=150, tol=1e-10)

    def cable(n):
        geom, _ = wl.squid_axon(n_comp=n - 2, length=1e-5 * (n - 2))
        return nrt.setup(geom, dT=1e-6)[0]

    large = cable(4096)
    with nrt.Solver(large, **opt) as s, nrt.Solver(large, **opt) as one:
        s.run(1, 2, 1, 10)
        with nrt.Solver(cable(3000), **opt) as t:
            t.run(1, 1, 1, 10)
            s.run(3, 2, 1, 10)
        v = s.snapshot()
        one.run(1, 4, 1, 10)
        assert np.array_equal(v, one.snapshot())
