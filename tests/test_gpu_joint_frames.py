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


@pytest.mark.parametrize("name", list(CASES))
def test_operators(name):
    spec, batch, Y, q, u, _, _ = _case(name)
    n = len(Y)
    rng = np.random.default_rng(len(name))
    v = rng.normal(size=(n, spec.nu)); f = rng.normal(size=(n, spec.nu))
    fs = [M.random_body_forces(spec, 3, i) for i in range(n)]
    V, f_, F_ = batch.pack(v), batch.pack(f), batch.pack(fs)
    X, Vb, qd, E = batch.realizeKinematics(q, u)
    E = E.cpu().numpy().reshape(-1, 2)
    X, Vb, qd = batch.split_b(X, 12), batch.split_b(Vb, 6), batch.split_q(qd)
    acc, accq = batch.realizeAcceleration(q, u, F_)
    acc, accq, acc0 = batch.split_u(acc), batch.split_q(accq), batch.split_u(batch.realizeAcceleration(q, u)[0])
    ud, A, qdd = batch.calcAccelerationIgnoringConstraints(q, u, f_, F_)
    ud, A, qdd = batch.split_u(ud), batch.split_b(A, 6), batch.split_q(qdd)
    minv = batch.split_u(batch.multiplyByMInv(q, f_))
    res = batch.split_u(batch.calcResidualForceIgnoringConstraints(q, u, f_, F_, V))
    res0 = batch.split_u(batch.calcResidualForceIgnoringConstraints(q, u))
    mv = batch.split_u(batch.multiplyByM(q, V))
    jv = batch.split_b(batch.multiplyBySystemJacobian(q, V), 6)
    jt = batch.split_u(batch.multiplyBySystemJacobianTranspose(q, F_))
    ba = batch.split_b(batch.calcBodyAccelerationFromUDot(q, u, V), 6)
    ba0 = batch.split_b(batch.calcBodyAccelerationFromUDot(q, u), 6)
    abi, abip = (batch.split_b(x, 21) for x in batch.realizeArticulatedBodyInertias(q))
    cbi = batch.split_b(batch.calcCompositeBodyInertias(q), 10)
    rf = batch.split_b(batch.calcMobilizerReactionForces(q, u, f_, F_), 6)
    assert int(batch.op_status().abs().sum()) == 0
    o = OracleModel(spec)
    for i in range(0, n, max(1, n // 8)):
        qi, ui = Y[i, :spec.nq].copy(), Y[i, spec.nq:].copy()
        k = o.kinematics(qi, ui)
        oud, oqdd, oA, _ = o.forward(qi, ui, f[i], fs[i])
        oP, oPP = o.abi(qi, spec.dofs())[:2]
        r1, rq = o.realize_acceleration(qi, ui, fs[i])[:2]
        oc = o.composite_inertias(qi)
        got = dict(X=X, V=Vb, qd=qd, acc=acc, accq=accq, acc0=acc0, ud=ud, A=A, qdd=qdd, minv=minv, res=res, res0=res0,
                   mv=mv, jv=jv, jt=jt, ba=ba, ba0=ba0, abi=[a[1:] for a in abi], rf=rf)
        ref = dict(X=k["X_GB"], V=k["V_GB"], qd=k["qdot"], acc=r1, accq=rq, acc0=o.realize_acceleration(qi, ui)[0],
                   ud=oud, A=oA, qdd=oqdd, minv=o.minv(qi, f[i]), res=o.residual(qi, ui, f[i], fs[i], v[i]),
                   res0=o.residual(qi, ui), mv=o.multiply_by_m(qi, v[i]), jv=o.jacobian(qi, v[i]),
                   jt=o.jacobian_transpose(qi, fs[i]), ba=o.body_acceleration(qi, ui, v[i]),
                   ba0=o.body_acceleration(qi, ui), abi=oP, rf=o.reactions(qi, ui, f[i], fs[i]))
        for key in got:
            # scaled by max(|ref|, 1): a lone Pin's velocity torque about its
            # axis is zero, the oracle's value for it rounding
            err = np.abs(np.ravel(got[key][i]) - np.ravel(ref[key])).max() / max(1.0, np.abs(ref[key]).max())
            assert err < (1e-11 if key == "rf" else 1e-12), (key, i, err)
        # P+ of a lone Free body is zero: compared on P's scale
        assert np.abs(np.ravel(abip[i][1:]) - np.ravel(oPP)).max() < 1e-12 * np.abs(oP).max(), i
        c = np.asarray(cbi[i]).reshape(-1, 10)
        assert np.isinf(c[0, 0]) and np.array_equal(c[0, 1:], oc[0, 1:]), i
        assert rel_inf(c[1:], oc[1:]) < 1e-12, i
        for e, key in ((0, "ke"), (1, "pe")):
            assert abs(E[i, e] - k[key]) <= 1e-12 * max(abs(k[key]), 1.0), (key, i)
