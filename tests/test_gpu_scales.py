"""Badly scaled models and states, each quantity on its own scale: a light fast
distal link; a fast balanced wheel at the end of slow arms; angles next to
the zeros of their cosine; a branch that is not a number beside one that is;
a small last body whose joint lies far from it; a small body that turns
about itself.

Tolerances.  A recursion that forms every body's own values from its parent's
is off by a few roundings of the quantity's own terms: with chains of three
bodies and at most 32 terms of rounding 1.1e-16, 1e-13 of an entry's terms
covers it; where a vector is compared on its largest entry, 1e-12."""
import numpy as np
import pytest

from simbody_amd import models as M
from oracle_ctypes import OracleModel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _planar(mobilizer, masses, parent=None):
    """Links along x, joints about z at their inner end, mass center halfway;
    the last body a wheel about its own joint where its mass is negative."""
    n = len(mobilizer)
    m = np.abs(np.array(masses, float))
    com = np.zeros((n, 3)); I = np.zeros((n, 6)); XF = np.tile(M._xform(), (n, 1)); XM = np.tile(M._xform(), (n, 1))
    parent = np.arange(n) if parent is None else np.array(parent)
    for b in range(n):
        if masses[b] > 0:
            com[b, 0] = 0.5
            I[b] = m[b] * np.array([0.01, 0.01 + 0.25, 0.02 + 0.25, 0, 0, 0])
        else:
            I[b] = m[b] * np.array([0.02, 0.02, 0.04, 0, 0, 0])
        if parent[b] > 0:
            XF[b, 9] = 1.0
    return M.TreeSpec(parent=parent.astype(np.int32), mobilizer=np.array(mobilizer, np.int32), mass=m, com_B=com,
                      inertia_B=I, X_PF=XF, X_BM=XM)


def _residual(spec, q, u, udot):
    """H^T of the forces that give udot, in extended precision: the recursion
    in Ground, one hinge axis after the other; and the sum of the magnitudes
    of the terms that make up each entry."""
    L = np.longdouble
    x3 = np.zeros(3, L)
    R, p, w, al, a = np.eye(3).astype(L), x3, x3, x3, x3         # frame; its origin's acceleration
    hinges, bodies, qi, ui = [], [], 0, 0
    for b in range(spec.nb):
        r = R @ spec.X_PF[b, 9:].astype(L)
        a = a + np.cross(al, r) + np.cross(w, np.cross(w, r))
        p = p + r
        ty = int(spec.mobilizer[b])

        def turn(axis, k, w, al):
            rate = L(u[k]) * axis
            return w + rate, al + L(udot[k]) * axis + np.cross(w, rate)

        if ty == M.SLIDER:
            ax, x = R[:, 0].copy(), L(q[qi])
            hinges.append((ui, None, ax, len(bodies)))
            a = a + np.cross(al, x * ax) + np.cross(w, np.cross(w, x * ax)) + 2 * L(u[ui]) * np.cross(w, ax) + L(udot[ui]) * ax
            p = p + x * ax
        elif ty == M.BALL:
            F = R.copy()
            rate, acc = F @ np.array(u[ui:ui + 3], L), F @ np.array(udot[ui:ui + 3], L)
            hinges += [(ui + k, p, F[:, k], len(bodies)) for k in range(3)]
            w, al = w + rate, al + acc + np.cross(w, rate)
            n = np.array(q[qi:qi + 4], L)
            c, s = (n / np.sqrt(n @ n))[0], (n / np.sqrt(n @ n))[1:]
            S = np.array([[0, -s[2], s[1]], [s[2], 0, -s[0]], [-s[1], s[0], 0]], L)
            R = R @ (np.eye(3) + 2 * c * S + 2 * S @ S)
        else:
            for k, i in enumerate([2] if ty == M.PIN else [0, 1]):
                hinges.append((ui + k, p, R[:, i].copy(), len(bodies)))
                w, al = turn(R[:, i], ui + k, w, al)
                c, s = np.cos(L(q[qi + k])), np.sin(L(q[qi + k]))
                m, n = (i + 1) % 3, (i + 2) % 3
                T = np.eye(3).astype(L)
                T[m, m] = T[n, n] = c
                T[m, n], T[n, m] = -s, s
                R = R @ T
        m, cb, I6 = L(spec.mass[b]), spec.com_B[b].astype(L), spec.inertia_B[b].astype(L)
        I = np.array([[I6[0], I6[3], I6[4]], [I6[3], I6[1], I6[5]], [I6[4], I6[5], I6[2]]])
        I = R @ (I - m * (cb @ cb * np.eye(3) - np.outer(cb, cb))) @ R.T
        c = R @ cb
        bodies.append((p + c, m * (a + np.cross(al, c) + np.cross(w, np.cross(w, c))), I @ al + np.cross(w, I @ w)))
        qi += M.NQ[ty]
        ui += M.DOF[ty]
    out, terms = np.zeros(spec.nu, L), np.zeros(spec.nu, L)
    for k, o, ax, first in hinges:
        for at, f, n in bodies[first:]:
            x = f if o is None else n + np.cross(at - o, f)
            y = f if o is None else np.abs(n) + np.abs(np.cross(at - o, f))
            out[k] += ax @ x
            terms[k] += np.abs(ax) @ np.abs(y)
    return out.astype(np.float64), terms.astype(np.float64)


def _comp(a, ref):
    b, terms = ref
    return float(np.max(np.abs(np.ravel(a) - b) / terms))


@pytest.mark.parametrize("m_tip", [1.0, 1e-4, 1e-8])
@pytest.mark.parametrize("types", [[M.PIN, M.PIN], [M.PIN, M.UNIVERSAL, M.PIN], [M.SLIDER, M.BALL, M.PIN]])
def test_light_fast_tip(types, m_tip):
    """M v, the residual and the reactions where the tip's share of the base
    torque is small although its acceleration is large."""
    from simbody_amd.matter import MatterBatch
    spec = _planar(types, [1.0] * (len(types) - 1) + [m_tip])
    batch = MatterBatch([spec], n_instances=2)
    q = np.zeros(spec.nq); u = np.zeros(spec.nu); v = np.zeros(spec.nu)
    qi, ui = spec.offsets()
    for b, t in enumerate(types):
        if t == M.BALL:
            q[qi[b]:qi[b] + 4] = M.Rng(5, b).normal(4)
            q[qi[b]:qi[b] + 4] /= np.linalg.norm(q[qi[b]:qi[b] + 4])
        else:
            q[qi[b]] = 0.3 + 0.2 * b
    v[0] = 1.0 / 3.0
    v[-1] = 1.0 / (7.0 * m_tip)
    u[0] = 0.1
    o = OracleModel(spec)
    Q, U, V = (batch.pack([x, x]) for x in (q, u, v))
    assert _comp(batch.split_u(batch.multiplyByM(Q, V))[1], _residual(spec, q, 0 * u, v)) < 1e-13
    got = batch.split_u(batch.calcResidualForceIgnoringConstraints(Q, U, udot=V))[1]
    assert _comp(got, _residual(spec, q, u, v)) < 1e-13
    # a torque that gives the tip that acceleration
    f = np.zeros(spec.nu)
    f[-1] = 0.01
    F = np.zeros((spec.nb + 1, 6))
    F[1] = [0.1, 0.2, 0.3, 1.0, 2.0, 3.0]
    got = np.reshape(batch.split_b(batch.calcMobilizerReactionForces(Q, U, batch.pack([f, f]), batch.pack([F, F])), 6)[1],
                     (-1, 6))
    ref = np.reshape(o.reactions(q, u, f, F), (-1, 6))
    for b in range(1, spec.nb + 1):
        scale = np.abs(ref[b]).max()
        assert np.abs(got[b] - ref[b]).max() < 1e-12 * scale, (b, got[b], ref[b])


def _wheel(tree):
    spec = (_planar([M.PIN, M.PIN, M.PIN, M.PIN], [1.0, 1.0, -0.5, 1.0], parent=[0, 1, 2, 1]) if tree
            else _planar([M.PIN, M.PIN, M.PIN], [1.0, 1.0, -0.5]))
    q = np.array([0.4, -0.7, 0.2, 1.1])[:spec.nq]
    u = np.array([0.9, -1.3, 1e7, 0.5])[:spec.nu]
    return spec, q, u


def _batch(spec, tree):
    from simbody_amd.matter import MatterBatch
    if not tree:
        return MatterBatch([spec], n_instances=3)
    # another tree beside it: a batch of different trees
    return MatterBatch([spec, _planar([M.PIN], [1.0])], tree_of=np.array([0, 1, 0], np.int32))


def _pack(batch, tree, x):
    return batch.pack([x, np.zeros(1) if tree else x, x])


@pytest.mark.parametrize("tree", [False, True])
def test_fast_wheel_accelerations(tree):
    from simbody_amd.matter import RungeKuttaMerson
    spec, q, u = _wheel(tree)
    batch = _batch(spec, tree)
    Q, U = _pack(batch, tree, q), _pack(batch, tree, u)
    ref = OracleModel(spec).realize_acceleration(q, u)[0]
    ud = batch.split_u(batch.realizeAcceleration(Q, U)[0])
    assert np.abs(ud[2] - ref).max() < 1e-12 * np.abs(ref).max()
    batch.rollout_begin(Q, U, RungeKuttaMerson(accuracy=1e-6), 0.1)
    ud = batch.split_u(batch.rollout_derivs()[1])
    assert np.abs(ud[2] - ref).max() < 1e-12 * np.abs(ref).max()
    fm, F = np.zeros(spec.nu), np.zeros((spec.nb + 1, 6))
    if not tree:
        got = batch.calcAccelerationIgnoringConstraints(Q, U, batch.pack([fm] * 3), batch.pack([F] * 3))[0]
        ref = OracleModel(spec).forward(q, u, fm, F)[0]
        assert np.abs(batch.split_u(got)[2] - ref).max() < 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("tree", [False, True])
@pytest.mark.parametrize("forces", [False, True])
def test_fast_wheel_rollout(tree, forces):
    """The arms' own motion over 100 fixed steps: its change against the
    oracle's, 100 x 5 evaluations of 1e-13 each."""
    from simbody_amd.matter import RungeKuttaMerson
    spec, q, u = _wheel(tree)
    batch = _batch(spec, tree)
    F = np.zeros((spec.nb + 1, 6))
    F[2, 5] = F[1, 2] = 0.25
    fapp = (batch.pack([F, np.zeros((2, 6)) if tree else F, F]) if forces else None)
    q1, u1, _ = batch.stepTo(_pack(batch, tree, q), _pack(batch, tree, u),
                             RungeKuttaMerson(accuracy=1e-3, fixed_step=1e-3), 0.1, fapp=fapp)
    y, _ = OracleModel(spec).integrate(np.concatenate([q, u]), 0.1, 1e-3, fixed_h=1e-3, Fapp=F if forces else None)
    arms = [0, 1] + ([3] if tree else [])
    for got, start, ref in ((batch.split_q(q1)[2], q, y[:spec.nq]), (batch.split_u(u1)[2], u, y[spec.nq:])):
        for k in arms:
            assert abs(got[k] - ref[k]) < 5e-11 * abs(ref[k] - start[k]), (k, got[k], ref[k])


def test_cosine_next_to_its_zeros():
    """A pendulum's udot is a constant times the cosine of its angle where
    gravity is along the link's normal at zero: relative accuracy at and
    beside multiples of pi/2 up to 2^20 (three roundings of the result)."""
    from simbody_amd.matter import MatterBatch
    spec = _planar([M.PIN], [1.0])
    k = np.unique(np.concatenate([np.arange(1, 400, 2), np.geomspace(401, 667000, 3000).astype(np.int64) | 1]))
    x0 = (k.astype(np.longdouble) * (np.longdouble("3.14159265358979323846264338327950288") / 2)).astype(np.float64)
    x = np.concatenate([x0, np.nextafter(x0, 0), np.nextafter(x0, np.inf), -x0, [0.0]])
    batch = MatterBatch([spec], n_instances=len(x))
    ud = batch.realizeAcceleration(batch.to_device(x), batch.to_device(np.zeros(len(x))))[0].cpu().numpy()
    c = np.cos(x.astype(np.longdouble))
    err = np.abs(ud / ud[-1] - c) / np.abs(c)
    worst = int(np.argmax(err))
    assert err[worst] < 1e-15, (x[worst], float(err[worst]))


def test_branch_beside_one_that_is_not_a_number():
    """Base branches do not touch each other: a Weld of one reads nothing of
    the other's coordinates."""
    from simbody_amd.matter import MatterBatch
    spec = _planar([M.PIN, M.WELD, M.PIN], [1.0, 1.0, 1.0], parent=[0, 1, 0])
    one = _planar([M.PIN], [1.0])
    batch = MatterBatch([spec, one], tree_of=np.array([0, 1, 0], np.int32))
    q = [np.array([0.3, np.nan]), np.zeros(1), np.array([0.3, 0.2])]
    u = [np.array([0.1, 0.2]), np.zeros(1), np.array([0.1, 0.2])]
    ud = batch.split_u(batch.realizeAcceleration(batch.pack(q), batch.pack(u))[0])
    assert ud[0][0] == ud[2][0] and np.isnan(ud[0][1])


@pytest.mark.parametrize("last", [M.PIN, M.UNIVERSAL, M.BALL, M.SLIDER])
def test_leaf_inertias(last):
    """Body frames at the mass center, joints 3 away, inertias of radius 0.001:
    composite and articulated inertias about the body origins, the last body's
    inertia blocks on their own size (what the joint's distance would add is 1e7
    times as large)."""
    from simbody_amd.matter import MatterBatch
    spec = _planar([M.BALL, M.PIN, last], [1.0, 1.0, 1.0])
    spec.com_B[:] = 0.0
    spec.inertia_B[:] = 1e-6 * np.array([2.0, 3.0, 4.0, 0.1, 0.2, 0.3])
    spec.X_BM[:, 9:] = [0.0, 3.0, 0.0]
    q = np.concatenate([[0.5, 0.5, -0.5, 0.5], [0.3], [0.8, 0.0, 0.6, 0.0] if last == M.BALL else [0.7, -0.4][:M.NQ[last]]])
    batch = MatterBatch([spec], n_instances=2)
    Q = batch.pack([q, q])
    P, PP = (np.reshape(batch.split_b(x, 21)[1], (-1, 21)) for x in batch.realizeArticulatedBodyInertias(Q))
    C = np.reshape(batch.split_b(batch.calcCompositeBodyInertias(Q), 10)[1], (-1, 10))
    o = OracleModel(spec)
    oP, oPP = o.abi(q, spec.dofs())[:2]
    oC = o.composite_inertias(q)
    for got, ref in ((P[1:], oP), (PP[1:], oPP), (C[1:], oC[1:])):
        assert np.abs(got - ref).max() < 1e-12 * np.abs(ref).max()
    for got, ref in ((P[3, 6:12], oP[2, 6:12]), (PP[3, 6:12], oPP[2, 6:12]), (C[3, 4:], oC[3, 4:])):
        assert np.abs(got - ref).max() < 1e-13 * np.abs(ref).max(), (got, ref)


def test_kinetic_energy_of_a_spinning_leaf():
    """A body of radius 0.001 that turns about its own mass center, the body
    origin, while its Free joint's frame, 3 away, moves: the energy is that of
    the turning alone, 1e-7 of what the joint frame's motion would suggest."""
    from simbody_amd.matter import MatterBatch
    spec = _planar([M.FREE], [1.0])
    spec.com_B[:] = 0.0
    spec.inertia_B[:] = 1e-6 * np.array([2.0, 3.0, 4.0, 0.1, 0.2, 0.3])
    spec.X_BM[:, 9:] = [0.0, 3.0, 0.0]
    batch = MatterBatch([spec], n_instances=2)
    q = np.array([1.0, 0, 0, 0, 0.1, 0.2, 0.3])
    w = np.array([0.75, -1.25, 0.5])
    u = np.concatenate([w, np.cross(w, [0.0, 3.0, 0.0])])
    E = batch.realizeKinematics(batch.pack([q, q]), batch.pack([u, u]))[3].cpu().numpy()
    I = 1e-6 * np.array([[2.0, 0.1, 0.2], [0.1, 3.0, 0.3], [0.2, 0.3, 4.0]])
    assert abs(E[2] - 0.5 * w @ I @ w) < 1e-13 * E[2]
