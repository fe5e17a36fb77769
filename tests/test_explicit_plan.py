"""The resident explicit step's plan (units, groups, cut edges, HH elements apart), its
steps taken on the host in the kernel's order of operations, against the oracle's
explicit step (CPU only): the same operations, so every bit, but for exp() (both host
libm: equal too)."""
import ctypes as C

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import load_golden, problem_from_golden
from test_oracle_math import _problem, _setup


def tree_host(p, T, steps, a0, a1):
    f = nh.lib().nrt_test_explicit_tree_host
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_double),
                  C.POINTER(C.c_int32), C.c_char_p, C.c_int]
    v, info, why = np.full(p.N, np.nan), np.zeros(5, np.int32), C.create_string_buffer(100)
    s = p.struct()
    st = f(C.addressof(s), T, steps, a0, a1, v.ctypes.data_as(C.POINTER(C.c_double)),
           info.ctypes.data_as(C.POINTER(C.c_int32)), why, 100)
    return (v, dict(zip(("G", "T", "slots", "units", "every"), info.tolist()))) if st == 0 else \
        why.value.decode()


def _random_tree(orc, depth, seed=0, hh=(1,), inputs=()):
    geom = wl.random_tree(wl.seed_for(3, seed), depth=depth)[0]
    for k in hh:
        geom.material[k] = 1
    for k in inputs:
        geom.input[k] = 1e-10
    s, bufs, H = _setup(orc, geom)
    p = _problem(geom, s, bufs, H, 1e-7)
    p.dT = 0.8 * float(s.dT_crit)
    rng = np.random.default_rng(seed)
    p.potential0 = p.potential0 + rng.uniform(-1e-3, 1e-3, p.N)
    p.potential1 = p.potential0.copy()
    return p


@pytest.mark.parametrize("depth,T,hh", [(2, 64, (1,)), (3, 64, (1, 2, 3)), (5, 64, (1, 40)),
                                        (6, 512, (1,)), (7, 64, (1, 2, 30, 31)), (9, 128, (1,))])
def test_trees_bitwise(depth, T, hh, orc):
    n = _random_tree(orc, depth).N
    p = _random_tree(orc, depth, hh=hh, inputs=(1, 20, n - 4))
    got = tree_host(p, T, 40, 5, 25)
    assert not isinstance(got, str), got
    assert (got[1]["G"] > 1) == (got[1]["units"] > T) == (got[1]["slots"] > 0)
    ref = orc.Explicit(p)
    ref.run(1, 40, 5, 25)
    assert np.array_equal(got[0], ref.snapshot())


@pytest.mark.parametrize("tree,T", [(0, 192), (0, 64), (240, 64), (480, 192)])
def test_dense_branching_bitwise(tree, T, orc):
    """Segments of a few elements: a halo of 16 elements does not fit, one of 4 does."""
    geom = wl.sweep_tree(tree)[0]
    s, bufs, H = _setup(orc, geom)
    p = _problem(geom, s, bufs, H, 0.8 * float(s.dT_crit))
    got = tree_host(p, T, 30, 1, 20)
    assert not isinstance(got, str), got
    ref = orc.Explicit(p)
    ref.run(1, 30, 1, 20)
    assert np.array_equal(got[0], ref.snapshot())


@pytest.mark.parametrize("name", ["ex4_ct_cable", "ex5_ct_y", "ex6_ct_tree"])
@pytest.mark.parametrize("T", [64, 512])
def test_golden_trees_bitwise(name, T, orc):
    g = load_golden(name)
    p = problem_from_golden(g)
    got = tree_host(p, T, 60, 1, 30)
    assert not isinstance(got, str), got
    ref = orc.Explicit(p)
    ref.run(1, 60, 1, 30)
    assert np.array_equal(got[0], ref.snapshot())


def test_what_the_form_refuses(orc):
    p = _random_tree(orc, 5, hh=range(1, 10))
    assert tree_host(p, 64, 1, 1, 1) == "too many HH elements"
    p = _random_tree(orc, 5)
    p.mother[40] = 10  # an element whose mother knows nothing of it
    assert tree_host(p, 64, 1, 1, 1) in ("mother's daughters", "right daughter")
    p = problem_from_golden(load_golden("ex3_hh_y"))
    assert tree_host(p, 64, 1, 1, 1) == "too many HH elements"
