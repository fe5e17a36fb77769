"""The resident tree solve on the GPU: one workgroup and several, at the sizes where
units, waves, groups or the exchange begin, with stimuli, probes and HH rows in other
places than the soma alone, stepped and run, alone and in batches, against the oracle's
exact solve. Bars as for the other FP64 tree solves: 1e-9 V to the oracle, 1e-12 V
between a slot and the same problem alone."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import TOL_V, ghost_mask, load_golden, max_abs_diff, problem_from_golden

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)


def _tree(nrt, depth, seed=0, hh_rows=1, inputs=()):
    geom, run = wl.random_tree(wl.seed_for(3, seed), depth=depth, amp=2e-9)
    geom.material[1:1 + hh_rows] = 1
    for k in inputs:
        geom.input[k] = 5e-10
    prob, _ = nrt.setup(geom, dT=run.dT)
    return prob


def _oracle(orc, p, steps, a0, a1, trace_elem=0, interval=-1):
    ref = orc.Implicit(p, variant=orc.VAR_GPU, method=orc.M_DIRECT)
    tr, st = ref.run(1, steps, a0, a1, trace_elem, interval)
    assert st == 0
    return ref.snapshot(), tr


@pytest.mark.parametrize("depth,hh_rows", [(2, 1), (3, 2), (5, 1), (6, 8), (7, 1), (8, 3), (10, 1),
                                           (12, 1)])
def test_run_and_step(depth, hh_rows, nrt, orc):
    p0 = _tree(nrt, depth)
    # stimuli at the soma, in the first dendrite and near the last element
    prob = _tree(nrt, depth, hh_rows=hh_rows, inputs=(12, p0.N - 5))
    print(f"[gpu-case] resident depth={depth} N={prob.N} hh={hh_rows}", flush=True)
    probe = prob.N // 3
    with nrt.Solver(prob, **DIRECT) as s:
        for i in range(1, 4):
            s.update(i != 2)
            s.calculate()
        tr = s.run(4, 37, 6, 20, trace_elem=probe, interval=2)
        tr1 = s.run(41, 6, 1, 43, trace_elem=1, interval=0)
        v, st = s.snapshot(), s.stats()
    assert st["tree_form"] == nh.TREE_RESIDENT and st["steps"] == 46
    assert st["krylov_iters"] == 46 and (st["num_blocks"] > 1) == (prob.N > 5000)
    ref = orc.Implicit(prob, variant=orc.VAR_GPU, method=orc.M_DIRECT)
    for i in range(1, 4):
        ref.update(i != 2)
        ref.calculate()
    rtr, _ = ref.run(4, 37, 6, 20, probe, 2)
    rtr1, _ = ref.run(41, 6, 1, 43, 1, 0)
    assert max_abs_diff(v, ref.snapshot(), ghost_mask(prob)) <= TOL_V
    assert len(tr) == len(rtr) and max_abs_diff(tr, rtr) <= TOL_V
    assert len(tr1) == 6 and max_abs_diff(tr1, rtr1) <= TOL_V


def test_repeated_step_numbers(nrt, orc):
    """Runs that count their steps from 1 again (the exchanged values' tags go on)."""
    prob = _tree(nrt, 10)
    with nrt.Solver(prob, **DIRECT) as s:
        for _ in range(5):
            s.run(1, 4, 1, 4)
        v = s.snapshot()
        assert s.stats()["num_blocks"] > 1
    ref, _ = _oracle(orc, prob, 20, 1, 20)
    assert max_abs_diff(v, ref, ghost_mask(prob)) <= TOL_V


@pytest.mark.parametrize("name", ["ex4_ct_cable", "ex5_ct_y", "ex6_ct_tree"])
def test_passive_neurites(name, nrt, orc):
    """No row changes: no dynamic row at all."""
    g = load_golden(name)
    p = problem_from_golden(g, dT=g["dT_crit"] * 10)
    with nrt.Solver(p, **DIRECT) as s:
        s.run(1, 50, 1, 20)
        v = s.snapshot()
        assert s.stats()["tree_form"] == nh.TREE_RESIDENT
    ref, _ = _oracle(orc, p, 50, 1, 20)
    assert max_abs_diff(v, ref, ghost_mask(p)) <= TOL_V


def test_long_unbranched_cable(nrt, orc):
    """One passive chain over several groups: every group is one strand of the top."""
    geom, _ = wl.squid_axon(n_comp=20000)
    geom.material[2:] = 0
    prob, _ = nrt.setup(geom, dT=2.5e-5)
    with nrt.Solver(prob, **DIRECT) as s:
        tr = s.run(1, 60, 1, 30, trace_elem=9000, interval=5)
        v, st = s.snapshot(), s.stats()
    assert st["tree_form"] == nh.TREE_RESIDENT and st["num_blocks"] >= 5
    ref, rtr = _oracle(orc, prob, 60, 1, 30, 9000, 5)
    assert max_abs_diff(v, ref, ghost_mask(prob)) <= TOL_V and max_abs_diff(tr, rtr) <= TOL_V


def test_more_changing_rows_take_the_general_solve(nrt, orc):
    prob = _tree(nrt, 6, hh_rows=9)
    with nrt.Solver(prob, **DIRECT) as s:
        s.run(1, 20, 1, 20)
        v = s.snapshot()
        assert s.stats()["tree_form"] != nh.TREE_RESIDENT
    ref, _ = _oracle(orc, prob, 20, 1, 20)
    assert max_abs_diff(v, ref, ghost_mask(prob)) <= TOL_V


def test_batch_of_resident_and_other_slots(nrt, orc):
    """Resident slots of both workgroup sizes beside slots of the general solve; each
    equals its problem alone, with its own steps, window and probe."""
    probs = [_tree(nrt, d, seed=d) for d in (3, 5, 8, 11)]
    g = load_golden("ex3_hh_y")
    probs.append(problem_from_golden(g, dT=g["dT_crit"] * 50))  # every row HH
    steps = [31, 50, 22, 40, 35]
    with nh.Batch(**DIRECT) as b:
        ids = [b.add(p, n, 2, 17, trace_elem=1, trace_every=2) for p, n in zip(probs, steps)]
        while b.stats()["active_slots"]:
            b.step(9)
        for p, n, sid in zip(probs, steps, ids):
            info = b.info(sid)
            assert info["status"] == 0 and info["steps_done"] == n and info["inner_iters"] == n
            with nrt.Solver(p, **DIRECT) as s:
                tr = s.run(1, n, 2, 17, trace_elem=1, interval=2)
                v = s.snapshot()
            assert max_abs_diff(b.snapshot(sid), v, ghost_mask(p)) <= 1e-12
            assert np.max(np.abs(b.trace(sid) - tr)) <= 1e-12
            ref, _ = _oracle(orc, p, n, 2, 17)
            assert max_abs_diff(v, ref, ghost_mask(p)) <= TOL_V


def test_small_slots_in_a_launch_of_their_own(nrt, orc):
    """Enough small slots to fill the device run beside larger ones in two launches."""
    small = [_tree(nrt, 3, seed=k) for k in range(4)]
    large = _tree(nrt, 9)
    with nh.Batch(**DIRECT) as b:
        ids = [b.add(small[k % 4], 20, 1, 10) for k in range(1500)]
        big = [b.add(large, 20, 1, 10) for _ in range(40)]
        b.step(20)
        assert b.stats()["launches"] == 2
        for p, sid in [(small[k], ids[k]) for k in range(4)] + [(large, big[0]), (large, big[-1])]:
            ref, _ = _oracle(orc, p, 20, 1, 10)
            assert max_abs_diff(b.snapshot(sid), ref, ghost_mask(p)) <= TOL_V
        for k in range(1500):
            assert np.array_equal(b.snapshot(ids[k]), b.snapshot(ids[k % 4]))
        for sid in big:
            assert np.array_equal(b.snapshot(sid), b.snapshot(big[0]))


def test_bounded_wait(nrt, orc):
    """With a wait of one poll the exchange gives up: the call reports it, every
    workgroup ends, and a handle with the normal bound works."""
    prob = _tree(nrt, 11)
    os.environ["NRT_SPIN_LIMIT"] = "1"
    try:
        with nrt.Solver(prob, **DIRECT) as s:
            with pytest.raises(nh.NrtError):
                s.run(1, 50, 1, 20)
    finally:
        del os.environ["NRT_SPIN_LIMIT"]
    with nrt.Solver(prob, **DIRECT) as s:
        s.run(1, 20, 1, 20)
        v = s.snapshot()
    ref, _ = _oracle(orc, prob, 20, 1, 20)
    assert max_abs_diff(v, ref, ghost_mask(prob)) <= TOL_V


def test_handles_of_several_threads(nrt, orc):
    """Large trees, each of which takes half the device or more, run by threads at the
    same time beside a batch: each call gives what it gives alone."""
    import threading
    probs = [_tree(nrt, 13, seed=k) for k in range(3)]
    small = _tree(nrt, 10, seed=7)
    alone, got, failed = [], [[] for _ in range(4)], []
    for p in probs + [small]:
        with nrt.Solver(p, **DIRECT) as s:
            s.run(1, 40, 1, 20)
            alone.append(s.snapshot())

    def work(k):
        try:
            if k < 3:
                with nrt.Solver(probs[k], **DIRECT) as s:
                    for i in range(8):
                        s.run(1 + 5 * i, 5, 1, 20)
                    got[k].append(s.snapshot())
            else:
                with nh.Batch(**DIRECT) as b:
                    ids = [b.add(small, 40, 1, 20) for _ in range(60)]
                    for _ in range(8):
                        b.step(5)
                    got[k] += [b.snapshot(i) for i in ids]
        except Exception as e:  # noqa: BLE001 (reported by the assertion below)
            failed.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for k in range(4):
        assert got[k] and all(np.array_equal(v, alone[k]) for v in got[k])
