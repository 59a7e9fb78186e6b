"""Admission of many requests in one call (their packing is split over host
threads from 4,096 bodies on) against the same requests in small calls, and
the first refused request of a large call."""
import numpy as np
import pytest

from simbody_amd import models as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N, NB = 300, 16


def _requests(tree_server):
    specs = [M.random_tree(50 + i % 7, i, nmin=NB, nmax=NB) for i in range(N)]
    if not tree_server:
        for t in specs:
            t.parent = np.arange(NB, dtype=np.int32)
            t.mobilizer = np.array([M.PIN, M.UNIVERSAL, M.BALL, M.SLIDER] * 4, np.int32)
    ys = [M.random_state(t, 5, i) for i, t in enumerate(specs)]
    return specs, [y[0] for y in ys], [y[1] for y in ys], np.linspace(0.005, 0.01, N)


def _server(tree_server, specs):
    from simbody_amd.matter import RungeKuttaMerson
    from simbody_amd.serving import Server, TreeServer
    integ = RungeKuttaMerson(accuracy=1e-5)
    return TreeServer(integ, 1 << 28, max_slots=512) if tree_server else Server(specs[0], integ, 1 << 28, max_slots=512)


def _admit(srv, tree_server, specs, q, u, t):
    if not tree_server:
        q, u = np.stack(q), np.stack(u)
    return srv.admit(specs, q, u, t)


@pytest.mark.parametrize("tree_server", [False, True])
def test_one_large_call_and_many_small_ones(tree_server):
    specs, q, u, t = _requests(tree_server)
    res = []
    for step in (N, 20):
        srv = _server(tree_server, specs)
        slots = np.concatenate([_admit(srv, tree_server, specs[i:i+step], q[i:i+step], u[i:i+step], t[i:i+step])
                                for i in range(0, N, step)])
        assert len(slots) == N
        srv.advance(10000)
        o = srv.collect()
        y = o["y"] if tree_server else [np.concatenate([a, b]) for a, b in zip(o["q"].copy(), o["u"].copy())]
        at = {int(s): k for k, s in enumerate(o["slots"])}
        res.append([y[at[int(s)]] for s in slots])
    assert all(np.array_equal(a, b) for a, b in zip(*res))


@pytest.mark.parametrize("tree_server", [False, True])
def test_first_refused_request_is_named(tree_server):
    from simbody_amd.matter import TdynError
    specs, q, u, t = _requests(tree_server)
    srv = _server(tree_server, specs)
    for i in (290, 130):
        specs[i].mass = specs[i].mass.copy()
        specs[i].mass[3] = np.nan
    with pytest.raises(TdynError, match="130"):
        _admit(srv, tree_server, specs, q, u, t)
    assert srv.info()["occupied"] == 0
