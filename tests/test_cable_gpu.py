"""Runs of unbranched neurites by the explicit cable kernel, at the sizes where
workgroups and halos begin: bit-identical to the same steps taken one launch at a time,
and within the FP64 bar of the oracle."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import TOL_V, max_abs_diff

pytestmark = pytest.mark.gpu


def _cable(nrt, n, mix, inputs=()):
    geom, _ = wl.squid_axon(n_comp=n - 2, length=1e-5 * (n - 2))
    if mix:  # HH elements here and there, passive ones between
        geom.material[1:-1] = (np.arange(1, n - 1) % 7 < 2).astype(np.int32)
    for k in inputs:
        geom.input[k] = 3e-10
    prob, _ = nrt.setup(geom, dT=None, dt_factor=0.8)
    return prob


@pytest.mark.parametrize("n,mix", [(4, False), (5, True), (255, False), (256, True), (257, False),
                                   (480, True), (481, False), (488, True), (489, False),
                                   (3000, True), (8192, False)])
def test_runs_equal_single_steps(n, mix, nrt, orc):
    prob = _cable(nrt, n, mix, inputs=(n // 2, n - 2))
    print(f"[gpu-case] cable N={n} mix={mix}", flush=True)
    chunks = (1, 7, 8, 9, 16, 3, 40)  # steps of each run: within and across exchanges
    probes = {k: [] for k in (0, n // 2, n - 1)}
    with nrt.Solver(prob, kind=nh.EXPLICIT) as s, nrt.Solver(prob, kind=nh.EXPLICIT) as one:
        step = 1
        for i, c in enumerate(chunks):
            k = list(probes)[i % 3]
            tr = s.run(step, c, 3, 50, trace_elem=k, interval=0)
            assert s.stats()["kernel_launches"] == 1
            for j in range(c):
                one.update(3 <= step + j <= 50)
                one.calculate()
                assert tr[j] == one.snapshot()[k]
            step += c
            assert np.array_equal(s.snapshot(), one.snapshot())
        # the two kinds of step may follow each other
        s.update(True)
        s.calculate()
        s.run(step + 1, 20, 1, 0)
        one.update(True)
        one.calculate()
        for _ in range(20):
            one.update(False)
            one.calculate()
        v = s.snapshot()
        assert np.array_equal(v, one.snapshot())
    ref = orc.Explicit(prob)
    ref.run(1, step - 1, 3, 50)
    ref.run(step, 1, step, step)
    ref.run(step + 1, 20, 1, 0)
    assert max_abs_diff(v, ref.snapshot()) <= TOL_V


def test_bounded_wait(nrt):
    """With a wait of one poll the exchange gives up, the state stays what it was, and a
    run with the normal bound goes on from it."""
    prob = _cable(nrt, 3000, False)
    with nrt.Solver(prob, kind=nh.EXPLICIT) as s, nrt.Solver(prob, kind=nh.EXPLICIT) as ref:
        s.run(1, 30, 1, 20)
        before = s.snapshot()
        os.environ["NRT_SPIN_LIMIT"] = "1"
        try:
            with pytest.raises(nh.NrtError):
                s.run(31, 400, 1, 20)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        assert np.array_equal(s.snapshot(), before)
        s.run(31, 50, 1, 20)
        ref.run(1, 80, 1, 20)
        assert np.array_equal(s.snapshot(), ref.snapshot())
