"""Gating rates of the direct solves next to their removable singularities (25 mV above
rest for the sodium activation, 10 mV for the potassium one): numerator and denominator
vanish together, so both have to come from one rounded value. The form that keeps its
rows in registers against the general one, which evaluates the same formula: one step from
potentials within rounding of the singular one and up to a microvolt away."""
import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import TOL_V, ghost_mask, max_abs_diff

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)
TOL_SAME = 1e-12  # two eliminations of a few hundred rows, one step, potentials below 0.1 V


def _near(volt):
    """Potentials around `volt`: its neighbours, and farther ones on either side."""
    out = []
    lo = hi = volt
    for _ in range(4):
        lo, hi = np.nextafter(lo, -1), np.nextafter(hi, 1)
        out += [lo, hi]
    for e in (1e-15, 1e-14, 1e-13, 1e-12, 1e-11, 1e-9, 1e-6):
        out += [volt - e, volt + e]
    return out


@pytest.mark.parametrize("mv", [25, 10])
def test_next_to_the_singular_potential(mv, nrt, orc):
    geom, run = wl.random_tree(wl.seed_for(3), depth=4)
    prob, _ = nrt.setup(geom, dT=run.dT)
    k = int(prob.hh_elem[0])
    rest, ls = float(prob.rest_pot[0]), float(prob.ls_Na[0] if mv == 25 else prob.ls_K[0])
    tried = 0
    for v in _near(rest - ls + mv * 1e-3):
        u = ((v + ls) - rest) / 0.001
        lin = (2.5 if mv == 25 else 1.0) - 0.1 * u
        if np.exp(lin) == 1.0:  # 0 / 0 in the formula itself
            continue
        prob.potential0[:] = v
        tried += 1
        ref = orc.Implicit(prob, variant=orc.VAR_GPU, method=orc.M_DIRECT)
        ref.run(1, 1, 1, 1, 0, -1)
        got = []
        for more in ({}, {"num_blocks": 1}):
            with nrt.Solver(prob, **DIRECT, **more) as s:
                s.run(1, 1, 1, 1)
                got.append(s.snapshot())
                assert (s.stats()["tree_form"] == nh.TREE_RESIDENT) == (not more)
        m = ghost_mask(prob)
        assert max_abs_diff(got[0], got[1], m) <= TOL_SAME, (v, u)
        assert abs(got[0][k] - ref.snapshot()[k]) <= TOL_V, (v, u)
    assert tried >= 14
