"""A tree server's results do not depend on what it served before: the same
burst again on the same server, and a burst larger than the memory pools,
whose rest waits, give bit for bit what a fresh server gives, with the same
step, rejection and projection counts.  The trees are rich in Balls and the
constraint tolerance (5e-7) lies among the quaternion errors of their steps
(median 9e-7), so every instance's projections depend on how many quaternions
its error is averaged over."""
import numpy as np
import pytest

from simbody_amd import models as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _burst(n, seed, nmin, nmax):
    specs = []
    for i in range(n):
        t = M.random_tree(seed, i, nmin=nmin, nmax=nmax)
        rng = np.random.default_rng(seed * 31 + i)
        t.mobilizer[:] = np.where(rng.uniform(size=t.nb) < 0.6, M.BALL, t.mobilizer)
        specs.append(t)
    ys = [M.random_state(t, seed, i) for i, t in enumerate(specs)]
    return specs, [y[0] for y in ys], [y[1] for y in ys], M.Rng(seed, 3).uniform(n, 0.2, 0.4)


def _server(budget, slots):
    from simbody_amd.matter import RungeKuttaMerson
    from simbody_amd.serving import TreeServer
    return TreeServer(RungeKuttaMerson(accuracy=1e-4, constraint_tolerance=5e-7), budget, max_slots=slots)


def _serve(sv, specs, q, u, t_end):
    """All requests in order, as many at a time as the server takes: results
    and the number admitted by each call."""
    out, slot_req, took, i = {}, {}, [], 0
    for _ in range(10000):
        if i < len(specs):
            slots = sv.admit(specs[i:], q[i:], u[i:], t_end[i:])
            for k, s in enumerate(slots):
                slot_req[int(s)] = i + k
            took.append(len(slots))
            i += len(slots)
        sv.advance(20)
        r = sv.collect()
        for j, s in enumerate(r["slots"]):
            out[slot_req.pop(int(s))] = (np.array(r["y"][j]), r["t"][j], r["status"][j], np.array(r["stats"][j]))
        if len(out) == len(specs):
            return out, took
    raise AssertionError("requests did not finish")


def _same(a, b):
    for i in a:
        assert tuple(a[i][3]) == tuple(b[i][3]), (i, a[i][3], b[i][3])
        assert np.array_equal(a[i][0], b[i][0]) and a[i][1] == b[i][1] and a[i][2] == b[i][2] == 1, i


def test_second_burst_is_the_first():
    req = _burst(24, 61, 6, 24)
    sv = _server(1 << 28, 64)
    first, _ = _serve(sv, *req)
    assert sum(first[i][3][3] for i in first) > 24
    again, _ = _serve(sv, *req)
    _same(first, again)
    # other trees in between, in another order of the places
    other = _burst(30, 62, 4, 30)
    _serve(sv, *other)
    _same(first, _serve(sv, *req)[0])


def test_burst_larger_than_the_pools():
    req = _burst(200, 63, 16, 40)
    all_at_once, took = _serve(_server(1 << 28, 256), *req)
    assert took == [200] and sum(all_at_once[i][3][3] for i in all_at_once) > 200
    small, took = _serve(_server(6 << 20, 256), *req)
    # (the pools, not the slots, held them back)
    assert 0 < took[0] < 150 and len(took) > 2
    _same(all_at_once, small)
