"""Chain batches on the joint-frame kernels against the oracle: every joint
type alone and mixed, one body and long chains (whose trig values do not fit
the LDS), identity and general joint frames, a Free root, applied forces, and
batches that fill no wavefront, one, and one and a lane.

Tolerances: the FP64 bounds the other parity tests hold (udot 1e-12 relative
per instance; rollouts 1e-8 with identical step counts)."""
import numpy as np
import pytest

from common import rel_inf
from simbody_amd import models as M
from oracle_ctypes import OracleModel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

P, S, U, B, F = M.PIN, M.SLIDER, M.UNIVERSAL, M.BALL, M.FREE
# mobilizers from the base, instances, general frames, applied forces
CASES = {
    "pin1": ([P], 1, False, False),
    "slider2": ([S, S], 3, True, True),
    "universal3": ([U] * 3, 64, True, True),
    "ball2": ([B, B], 65, True, True),
    "free1": ([F], 2, False, True),
    "free_mixed": ([F] + [B, P, S, U] * 3, 63, True, True),
    "mixed_identity": ([P, U, B, S] * 4, 66, False, False),
    "mixed_general": ([S, B, U, P] * 5, 5, True, False),
    "long": ([P, U, B] * 15, 3, False, True),
    "long_general": ([F] + [U, P] * 20, 3, True, False),
}


def _chain(types, frames, seed):
    t = M.random_tree(seed, 1, nmin=len(types), nmax=len(types), general_frames=frames)
    t.parent = np.arange(len(types), dtype=np.int32)
    t.mobilizer = np.array(types, np.int32)
    return t


def _case(name):
    types, n, frames, forces = CASES[name]
    seed = 40 + sorted(CASES).index(name)
    spec = _chain(types, frames, seed)
    Y = M.random_states(spec, seed, np.arange(n))
    fs = [M.random_body_forces(spec, seed, i) for i in range(n)] if forces else None
    from simbody_amd.matter import MatterBatch
    batch = MatterBatch([spec], n_instances=n)
    q, u = batch.pack(Y[:, :spec.nq]), batch.pack(Y[:, spec.nq:])
    return spec, batch, Y, q, u, fs, (batch.pack(fs) if forces else None)


@pytest.mark.parametrize("name", list(CASES))
def test_rollout_derivative(name):
    from simbody_amd.matter import RungeKuttaMerson
    spec, batch, Y, q, u, fs, F_ = _case(name)
    batch.rollout_begin(q, u, RungeKuttaMerson(accuracy=1e-6), 0.1, fapp=F_)
    assert batch.active_evaluator()[0] == 2
    qd, ud = batch.rollout_derivs()
    qds, uds = batch.split_q(qd), batch.split_u(ud)
    o = OracleModel(spec)
    for i in range(len(Y)):
        ref, rqd, _, _ = o.realize_acceleration(Y[i, :spec.nq], Y[i, spec.nq:], fs[i] if fs else None)
        assert rel_inf(uds[i], ref) < 1e-12, i
        assert rel_inf(qds[i], rqd) < 1e-12, i


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("accuracy", [1e-3, 1e-7])
def test_rollout(name, accuracy):
    from simbody_amd.matter import RungeKuttaMerson
    spec, batch, Y, q, u, fs, F_ = _case(name)
    q1, u1, st = batch.stepTo(q, u, RungeKuttaMerson(accuracy=accuracy), 0.08, fapp=F_)
    qs, us, st = batch.split_q(q1), batch.split_u(u1), st.cpu().numpy()
    o = OracleModel(spec)
    for i in range(0, len(Y), max(1, len(Y) // 8)):
        y, s = o.integrate(Y[i], 0.08, accuracy, Fapp=fs[i] if fs else None)
        assert rel_inf(np.concatenate([qs[i], us[i]]), y) < 1e-8, i
        assert (s["attempts"], s["accepted"], s["rejected"], s["projections"]) == tuple(st[i]), (i, st[i], s)


def test_large_angles():
    """Angles near multiples of pi/2, tiny, large, and past the range of the
    kernels' own sine and cosine: udot of single pendulums and of a
    Universal against the oracle."""
    from simbody_amd.matter import MatterBatch, RungeKuttaMerson
    base = np.array([0.0, 1e-300, 1e-9, 0.5, 1.0, 10.0, 1e3, 1e5, 1048575.9, 1048576.1, 3e7, 1e15])
    mult = np.pi / 2 * np.array([1.0, 2.0, 3.0, 7.0, 1001.0, 123456.0])
    qs = np.concatenate([base, -base, mult, np.nextafter(mult, 0), mult + 1e-7, -mult])
    for types in ([P], [U]):
        spec = _chain(types, False, 7)
        n = len(qs)
        Y = np.zeros((n, spec.nq + spec.nu))
        Y[:, 0] = qs
        if types == [U]:
            Y[:, 1] = qs[::-1]
        Y[:, spec.nq:] = 0.3
        batch = MatterBatch([spec], n_instances=n)
        batch.rollout_begin(batch.pack(Y[:, :spec.nq]), batch.pack(Y[:, spec.nq:]), RungeKuttaMerson(accuracy=1e-6), 0.1)
        uds = batch.split_u(batch.rollout_derivs()[1])
        o = OracleModel(spec)
        for i in range(n):
            ref = o.realize_acceleration(Y[i, :spec.nq], Y[i, spec.nq:])[0]
            assert np.abs(uds[i] - ref).max() < 1e-12 * max(1.0, np.abs(ref).max()), (types, qs[i])
