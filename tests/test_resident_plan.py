"""The resident tree solve's plan (units, pieces, groups, top, dynamic rows), solved on
the host phase by phase as the kernel does, against the oracle's sequential elimination,
the general tree partition solve and dense numpy solves (CPU only).

The systems are diagonally dominant: elimination loses a few ulps a row of the longest
path at most, so 1e-11 relative (1e-12 on the small ones) is far above rounding."""
import ctypes as C

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import load_golden, problem_from_golden
from test_oracle_math import _problem, _setup
from test_tree_plan import _system, tps_host

_dp = C.POINTER(C.c_double)
_ip = C.POINTER(C.c_int32)


def resident_host(rp, col, val, rhs, hh, T):
    """(x, info) or the reason why the form does not apply."""
    f = nh.lib().nrt_test_resident_solve_host
    f.argtypes = [C.c_int, _ip, _ip, _dp, _dp, _ip, C.c_int, C.c_int, _dp, _ip, C.c_char_p,
                  C.c_int]
    rp, col = np.ascontiguousarray(rp, np.int32), np.ascontiguousarray(col, np.int32)
    val, rhs = np.ascontiguousarray(val, np.float64), np.ascontiguousarray(rhs, np.float64)
    hh = np.ascontiguousarray(hh, np.int32)
    x, info = np.full(len(rhs), np.nan), np.zeros(8, np.int32)
    why = C.create_string_buffer(100)
    st = f(len(rhs), rp.ctypes.data_as(_ip), col.ctypes.data_as(_ip), val.ctypes.data_as(_dp),
           rhs.ctypes.data_as(_dp), hh.ctypes.data_as(_ip), len(hh), T, x.ctypes.data_as(_dp),
           info.ctypes.data_as(_ip), why, 100)
    if st != 0:
        return why.value.decode()
    return x, dict(zip(("G", "nt", "nth", "npub", "rounds", "heights", "pieces", "nd"),
                       info.tolist()))


@pytest.mark.parametrize("name", ["ex4_ct_cable", "ex5_ct_y", "ex6_ct_tree", "ex8_neuron"])
@pytest.mark.parametrize("T", [64, 512])
def test_golden_systems(name, T, orc):
    g = load_golden(name)
    p = problem_from_golden(g, dT=g["dT_crit"] * 10)
    rp, col, val, rhs = _system(orc, p)
    got = resident_host(rp, col, val, rhs, [1], T)
    assert not isinstance(got, str), got
    ref = orc.tree_solve(rp, col, val, rhs)
    assert np.max(np.abs(got[0] - ref)) <= 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("depth,T,groups", [(3, 64, 1), (6, 512, 1), (8, 64, 100), (9, 256, 14),
                                            (10, 512, 14), (11, 512, 30)])
def test_dendritic_trees_against_the_general_solve(depth, T, groups, orc):
    geom = wl.random_tree(wl.seed_for(3), depth=depth)[0]
    s, bufs, H = _setup(orc, geom)
    p = _problem(geom, s, bufs, H, 2.5e-5)
    rp, col, val, rhs = _system(orc, p)
    x, info = resident_host(rp, col, val, rhs, p.hh_elem, T)
    assert info["nd"] == 1 and info["G"] >= 1
    assert (info["G"] > 1) == (groups > 1) and info["G"] <= groups * 1.3 + 1, info
    ref = orc.tree_solve(rp, col, val, rhs)
    assert np.max(np.abs(x - ref)) <= 1e-11 * np.max(np.abs(ref))
    general, _, _ = tps_host(rp, col, val, rhs, 8, 8)
    assert np.max(np.abs(x - general)) <= 1e-11 * np.max(np.abs(ref))


def _forest(rng, n, kind):
    """Parent (lower-numbered, at most two children each) of n rows: chains, bushy trees,
    scattered numbering, several components, rows alone."""
    par = np.full(n, -1)
    kids = np.zeros(n, dtype=int)
    for i in range(1, n):
        r = rng.random()
        if r < (0.02 if kind != "forest" else 0.15):
            continue
        open_ = np.nonzero(kids[:i] < 2)[0]
        if kind == "chain":
            p = i - 1 if kids[i - 1] < 2 and r < 0.97 else int(rng.choice(open_))
        elif kind == "bushy":
            p = int(open_[rng.integers(max(0, len(open_) - 6), len(open_))])
        else:
            p = int(rng.choice(open_))
        par[i] = p
        kids[p] += 1
    return par


def _matrix(rng, par):
    """Symmetric diagonally dominant CSR of the forest."""
    n = len(par)
    g = rng.uniform(0.5, 2.0, n)
    diag = rng.uniform(0.01, 0.2, n)
    rows = [[] for _ in range(n)]
    for i in range(n):
        if par[i] >= 0:
            diag[i] += g[i]
            diag[par[i]] += g[i]
            rows[i].append((par[i], -g[i]))
            rows[par[i]].append((i, -g[i]))
    for i in range(n):
        rows[i].append((i, diag[i]))
    rp, col, val = [0], [], []
    for r in rows:
        r.sort()
        col += [c for c, _ in r]
        val += [v for _, v in r]
        rp.append(len(col))
    return np.array(rp), np.array(col), np.array(val)


@pytest.mark.parametrize("kind", ["chain", "bushy", "scattered", "forest"])
@pytest.mark.parametrize("n,T", [(4, 64), (7, 64), (9, 64), (65, 64), (513, 64), (1025, 64),
                                 (1500, 128), (1200, 512)])
def test_random_forests_against_dense(kind, n, T):
    rng = np.random.default_rng([n, T, len(kind)])
    for trial in range(3):
        par = _forest(rng, n, kind)
        rp, col, val = _matrix(rng, par)
        b = rng.uniform(-1, 1, n)
        # dynamic rows: up to three whose root paths are short
        hh = []
        for i in rng.permutation(n)[:40]:
            path = set(hh)
            j = int(i)
            while j >= 0:
                path.add(j)
                j = int(par[j])
            if len(path) <= 8 and len(hh) < trial + 1:
                hh.append(int(i))
        got = resident_host(rp, col, val, b, hh, T)
        if isinstance(got, str):
            assert got == "too many rows change", got  # (paths that add up to more than 8)
            continue
        A = np.zeros((n, n))
        for i in range(n):
            A[i, col[rp[i]:rp[i + 1]]] = val[rp[i]:rp[i + 1]]
        ref = np.linalg.solve(A, b)
        assert np.max(np.abs(got[0] - ref)) <= 1e-11 * np.max(np.abs(ref)), (kind, n, T, trial)


def test_what_the_form_refuses():
    rng = np.random.default_rng(3)
    par = np.arange(-1, 39)
    rp, col, val = _matrix(rng, par)
    b = np.ones(40)
    assert resident_host(rp, col, val, b, [8], 64) == "too many rows change"
    assert not isinstance(resident_host(rp, col, val, b, [7], 64), str)
    bad = val.copy()
    bad[rp[5]] *= 1.0 + 1e-15  # row 5's coupling to row 4, one ulp off its transpose
    assert resident_host(rp, col, bad, b, [0], 64) == "asymmetric coupling"
    par = np.array([-1, 0, 0, 0, 3, 4])
    rp, col, val = _matrix(rng, par)
    assert resident_host(rp, col, val, np.ones(6), [], 64) == "more than two children"
