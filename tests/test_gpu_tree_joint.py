"""Level-parallel trees against the oracle where the evaluator's rules change:
one body, a level wider than the LDS ring (a far parent), a chain among
trees, several base bodies, a Free base, Welds only, every mobilizer of the
padded form, identity and general joint frames, with and without body forces;
as one tree in many instances and as a batch of different trees.  Bounds as
in the other parity tests: udot and qdot 1e-12 relative per instance,
rollouts 1e-8 with the oracle's step counts."""
import numpy as np
import pytest

from common import rel_inf
from simbody_amd import models as M
from oracle_ctypes import OracleModel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

G10 = [M.PIN, M.SLIDER, M.UNIVERSAL, M.BALL, M.TRANSLATION, M.PLANAR, M.CYLINDER, M.SCREW, M.GIMBAL, M.WELD]


def _tree(seed, parent, mobilizer, frames):
    n = len(parent)
    t = M.random_tree(seed, 1, nmin=n, nmax=n, general_frames=frames)
    t.parent = np.array(parent, np.int32)
    t.mobilizer = np.array(mobilizer, np.int32)
    if M.SCREW in mobilizer:
        t.pitch = np.full(n, 0.3)
    return t


def _trees(frames):
    rng = np.random.default_rng(17)
    mob = lambda n, types=G10: [types[i % len(types)] for i in rng.permutation(n)]
    return [
        _tree(1, [0], [M.BALL], frames),
        _tree(2, [0, 1, 1], [M.FREE, M.PIN, M.UNIVERSAL], frames),
        _tree(3, [0] + [1] * 70, [M.PIN] + mob(70), frames),                     # one wide level
        _tree(4, list(range(21)), [M.UNIVERSAL] + mob(20), frames),              # a chain
        _tree(5, [0, 0, 0, 1, 2, 3, 3], [M.FREE, M.SLIDER, M.BALL] + mob(4), frames),
        _tree(6, [0] + [1 + i // 2 for i in range(62)], [M.GIMBAL] + mob(62), frames),
        _tree(7, [0] + [1 + i // 40 for i in range(130)], [M.FREE] + mob(130), frames),
    ]


def _states(per):
    ys = [M.random_state(t, 23, i) for i, t in enumerate(per)]
    fs = [M.random_body_forces(t, 29, i) for i, t in enumerate(per)]
    return [y[0] for y in ys], [y[1] for y in ys], fs


@pytest.mark.parametrize("frames", [False, True])
@pytest.mark.parametrize("forces", [False, True])
@pytest.mark.parametrize("which", ["different", 2, 4, 6])
def test_acceleration_and_rollout(frames, forces, which):
    from simbody_amd.matter import MatterBatch, RungeKuttaMerson
    trees = _trees(frames)
    if which == "different":
        per = [trees[i % len(trees)] for i in range(2 * len(trees) + 3)]
        batch = MatterBatch(trees, tree_of=np.arange(len(per), dtype=np.int32) % len(trees))
    else:
        per = [trees[which]] * 3
        batch = MatterBatch([trees[which]], n_instances=3)
    qs, us, fs = _states(per)
    q, u, F = batch.pack(qs), batch.pack(us), (batch.pack(fs) if forces else None)
    ud, qd = batch.realizeAcceleration(q, u, F)
    assert int(batch.op_status().abs().sum()) == 0
    uds, qds = batch.split_u(ud), batch.split_q(qd)
    for i, t in enumerate(per):
        ref, rqd = OracleModel(t).realize_acceleration(qs[i], us[i], fs[i] if forces else None)[:2]
        assert rel_inf(uds[i], ref) < 1e-12, i
        assert rel_inf(qds[i], rqd) < 1e-12, i
    q1, u1, st = batch.stepTo(q, u, RungeKuttaMerson(accuracy=1e-5), 0.03, fapp=F)
    q1, u1, st = batch.split_q(q1), batch.split_u(u1), st.cpu().numpy()
    for i in range(0, len(per), 2):
        y, s = OracleModel(per[i]).integrate(np.concatenate([qs[i], us[i]]), 0.03, 1e-5, Fapp=fs[i] if forces else None)
        assert rel_inf(np.concatenate([q1[i], u1[i]]), y) < 1e-8, i
        assert (s["attempts"], s["accepted"], s["rejected"], s["projections"]) == tuple(st[i]), i


def test_large_angles():
    """Half the angles of the padded form go through the kernels' own sine and
    cosine up to 2^20, through the library's beyond."""
    from simbody_amd.matter import MatterBatch
    angles = np.array([0.0, 1e-300, np.pi, -np.pi, 2 * np.pi, 10.0, -1e3, 1e5, 2097151.9, 2097152.1, -3e7, 1e15])
    trees = [_tree(8, [0, 1], [ty, M.PIN], False) for ty in (M.PIN, M.UNIVERSAL, M.GIMBAL, M.PLANAR)]
    per = [t for t in trees for _ in angles]
    batch = MatterBatch(trees, tree_of=np.repeat(np.arange(len(trees), dtype=np.int32), len(angles)))
    qs, us = [], []
    for i, t in enumerate(per):
        q = np.full(t.nq, 0.4)
        q[0] = angles[i % len(angles)]
        if t.mobilizer[0] in (M.UNIVERSAL, M.GIMBAL):
            q[1] = 0.3 + angles[(i + 1) % len(angles)] * (t.mobilizer[0] == M.UNIVERSAL)
        qs.append(q); us.append(np.full(t.nu, 0.3))
    uds = batch.split_u(batch.realizeAcceleration(batch.pack(qs), batch.pack(us))[0])
    for i, t in enumerate(per):
        ref = OracleModel(t).realize_acceleration(qs[i], us[i])[0]
        assert np.abs(uds[i] - ref).max() < 1e-12 * max(1.0, np.abs(ref).max()), i
