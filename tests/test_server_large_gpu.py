"""The server's large requests in the forms that their size and shape take by default
(rows resident in several workgroups, an axon's waves): the same result as alone, beside
batch slots and a second server; and a wait that ends early never passes for a result."""
import os

import numpy as np
import pytest

import neurite_hip as nh
import workloads as wl
from common import ghost_mask, max_abs_diff

pytestmark = pytest.mark.gpu
DIRECT = dict(kind=nh.IMPLICIT, krylov=nh.DIRECT)
TOL_SAME = 1e-12  # as for the server's other requests


def _tree(nrt, depth, seed):
    geom, run = wl.random_tree(wl.seed_for(5, seed), depth=depth, amp=4e-9)
    return nrt.setup(geom, dT=run.dT)[0]


def _axon(nrt, nodes):
    geom, run = wl.myelinated_axon(nodes=nodes)
    return nrt.setup(geom, dT=run.dT)[0]


def _alone(nrt, p, n, a0, a1, te=0, ev=-1):
    with nrt.Solver(p, **DIRECT) as s:
        tr = s.run(1, n, a0, a1, te, ev)
        return s.snapshot(), tr, s.stats()


def test_results_same_alone_and_in_mix(nrt):
    probs = [_tree(nrt, 11, 1), _axon(nrt, 60), _tree(nrt, 5, 2), _tree(nrt, 9, 3),
             _axon(nrt, 130), _tree(nrt, 13, 4)]
    reqs = [(p, 30 + 11 * i, 2, 20, 1, i % 3) for i, p in enumerate(probs)]
    print("[gpu-case] large requests", [p.N for p in probs], flush=True)
    alone = [_alone(nrt, *r) for r in reqs]
    assert all(st["tree_form"] == nh.TREE_RESIDENT for _, _, st in alone)
    assert sum(st["num_blocks"] > 1 and p.N > 6000 for p, (_, _, st) in zip(probs, alone)) >= 4
    srvs = [nh.Server(steps_per_launch=7, big_threshold=6000, **DIRECT) for _ in range(2)]
    try:
        ids = [(s, [s.submit(*r) for r in reqs]) for s in srvs]
        for s, rids in ids:
            s.wait_idle(60.0)
            done = {r["id"]: r for r in s.poll()}
            for rid, r, (v, tr, _) in zip(rids, reqs, alone):
                assert done[rid]["status"] == 0 and done[rid]["steps_done"] == r[1]
                st, got, gtr = s.fetch(rid)
                assert st == 0 and max_abs_diff(got, v, ghost_mask(r[0])) <= TOL_SAME
                assert len(gtr) == len(tr) and np.max(np.abs(gtr - tr)) <= TOL_SAME
    finally:
        for s in srvs:
            s.close()


@pytest.mark.parametrize("shape", ["tree", "axon"])
def test_bounded_wait(shape, nrt):
    """With one poll allowed the exchanges give up: the request fails with the potentials
    of the steps that it reports, and the next one, with the normal bound, is right."""
    p = _tree(nrt, 11, 1) if shape == "tree" else _axon(nrt, 60)
    m = ghost_mask(p)
    with nh.Server(steps_per_launch=400, big_threshold=4000, **DIRECT) as srv:
        os.environ["NRT_SPIN_LIMIT"] = "0"
        try:
            rid = srv.submit(p, 400, 1, 20)
            srv.wait_idle(60.0)
        finally:
            del os.environ["NRT_SPIN_LIMIT"]
        info = srv.poll()[0]
        status, v, _ = srv.fetch(rid)
        assert status != 0 and info["status"] == status and info["steps_done"] == 0
        assert np.array_equal(v, p.potential0)
        rid = srv.submit(p, 50, 1, 20)
        srv.wait_idle(60.0)
        status, v, _ = srv.fetch(rid)
        assert status == 0
        assert max_abs_diff(v, _alone(nrt, p, 50, 1, 20)[0], m) <= TOL_SAME
