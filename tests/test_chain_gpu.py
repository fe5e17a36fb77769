"""The chain solve on the GPU: unbranched neurites with more gating rows than the resident
tree solve takes, at the sizes where lanes, waves, the exchange and 16 rows per lane
begin, with stimuli, probes and single steps, against the oracle's exact solve. Bars as
for the other FP64 direct solves: 1e-9 V."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import TOL_V, ghost_mask, max_abs_diff

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)


def _axon(nrt, n, rows, inputs=()):
    """n elements, gating ones at rows, the others passive."""
    geom, _ = wl.squid_axon(n_comp=n - 2, length=1e-5 * (n - 2))
    geom.material[:] = 0
    geom.material[[r for r in rows if 1 <= r <= n - 2]] = 1
    for k in inputs:
        geom.input[k] = 3e-10
    prob, _ = nrt.setup(geom, dT=2.5e-5)
    return prob


# (a lane has 8 rows, a wave 512; 16 and 1,024 above 32,768 rows)
@pytest.mark.parametrize("n,rows", [
    (40, range(1, 39, 3)), (511, range(1, 500, 60)), (512, range(5, 511, 31)),
    (513, range(7, 513, 8)), (514, range(1, 513, 40)), (1024, [*range(440, 503), 1022]),
    (1030, range(1, 1029, 100)), (5000, range(8, 4999, 8)), (20202, range(1, 20201, 101)),
    (32768, range(3, 32767, 700)), (32769, range(15, 32768, 512)), (60602, range(1, 60601, 101)),
    (65536, range(16, 65535, 1000))])
def test_run_and_step(n, rows, nrt, orc):
    prob = _axon(nrt, n, rows, inputs=(1, n // 2, n - 2))
    print(f"[gpu-case] chain N={n} gating={len(prob.hh_elem)}", flush=True)
    probe = n // 3
    with nrt.Solver(prob, **DIRECT) as s:
        for i in range(1, 4):
            s.update(i != 2)
            s.calculate()
        tr = s.run(4, 17, 6, 15, trace_elem=probe, interval=2)
        tr1 = s.run(21, 6, 1, 23, trace_elem=1, interval=0)
        v, st = s.snapshot(), s.stats()
    assert st["tree_form"] == nh.TREE_RESIDENT and st["steps"] == 26
    assert st["num_blocks"] == -(-n // (512 if n <= 32768 else 1024))
    ref = orc.Implicit(prob, variant=orc.VAR_GPU, method=orc.M_DIRECT)
    for i in range(1, 4):
        ref.update(i != 2)
        ref.calculate()
    rtr, _ = ref.run(4, 17, 6, 15, probe, 2)
    rtr1, _ = ref.run(21, 6, 1, 23, 1, 0)
    assert max_abs_diff(v, ref.snapshot(), ghost_mask(prob)) <= TOL_V
    assert len(tr) == len(rtr) and max_abs_diff(tr, rtr) <= TOL_V
    assert len(tr1) == 6 and max_abs_diff(tr1, rtr1) <= TOL_V


@pytest.mark.parametrize("n,rows", [(1002, range(1, 66)), (65537, range(16, 65536, 1000))])
def test_what_the_form_refuses(n, rows, nrt, orc):
    """65 gating rows in a wave, 65 waves: the general solve."""
    prob = _axon(nrt, n, rows)
    with nrt.Solver(prob, **DIRECT) as s:
        s.run(1, 10, 1, 10)
        v = s.snapshot()
        assert s.stats()["tree_form"] != nh.TREE_RESIDENT
    ref = orc.Implicit(prob, variant=orc.VAR_GPU, method=orc.M_DIRECT)
    ref.run(1, 10, 1, 10, 0, -1)
    assert max_abs_diff(v, ref.snapshot(), ghost_mask(prob)) <= TOL_V


def test_bounded_wait(nrt):
    """With a wait of one poll the exchange gives up, the state stays what it was, and a
    run with the normal bound goes on from it; step numbers may begin again."""
    prob = _axon(nrt, 5000, range(1, 4999, 50))
    with nrt.Solver(prob, **DIRECT) as s, nrt.Solver(prob, **DIRECT) as ref:
        s.run(1, 30, 1, 30)
        before = s.snapshot()
        os.environ["NRT_SPIN_LIMIT"] = "0"
        try:
            with pytest.raises(nh.NrtError):
                s.run(1, 400, 1, 20)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        assert np.array_equal(s.snapshot(), before)
        s.run(1, 50, 1, 50)
        ref.run(1, 80, 1, 80)
        assert np.array_equal(s.snapshot(), ref.snapshot())
