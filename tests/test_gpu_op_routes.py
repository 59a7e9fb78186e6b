"""realizeAcceleration of trees at the sizes and shapes where the evaluator and
its lanes change, against the oracle (1e-12 relative per instance, as the other
parity tests hold): more different narrow trees than groups of 16 lanes, with a
wide one and a long one among them; and one tree, narrow or wide, with and
without room for its steps."""
import numpy as np
import pytest

from common import rel_inf
from simbody_amd import models as M
from oracle_ctypes import OracleModel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TYPES = [M.PIN, M.BALL, M.UNIVERSAL, M.SLIDER, M.GIMBAL, M.SCREW, M.PLANAR, M.WELD]


def _tree(seed, parent, frames, free=False):
    n = len(parent)
    t = M.random_tree(seed, 1, nmin=n, nmax=n, general_frames=frames)
    t.parent = np.array(parent, np.int32)
    t.mobilizer = np.array([M.FREE if free else M.PIN] + [TYPES[(seed + b) % len(TYPES)] for b in range(1, n)], np.int32)
    t.pitch = np.full(n, 0.3)
    return t


def _check(batch, per, forces, sample):
    ys = [M.random_state(t, 23, i) for i, t in enumerate(per)]
    fs = [M.random_body_forces(t, 29, i) for i, t in enumerate(per)]
    q, u = batch.pack([y[0] for y in ys]), batch.pack([y[1] for y in ys])
    ud, qd = batch.realizeAcceleration(q, u, batch.pack(fs) if forces else None)
    assert int(batch.op_status().abs().sum()) == 0
    uds, qds = batch.split_u(ud), batch.split_q(qd)
    for i in sample:
        ref, rqd = OracleModel(per[i]).realize_acceleration(*ys[i], fs[i] if forces else None)[:2]
        assert rel_inf(uds[i], ref) < 1e-12, i
        assert rel_inf(qds[i], rqd) < 1e-12, i


@pytest.mark.parametrize("frames,forces", [(False, False), (True, True)])
def test_more_narrow_trees_than_groups(frames, forces):
    from simbody_amd.matter import MatterBatch
    narrow = [_tree(k, [0] + [max(0, b - (k % 3 == 2 and b % 4 == 3)) for b in range(1, 3 + k)], frames, free=k % 4 == 1)
              for k in range(8)]
    trees = narrow + [_tree(8, [0] + [1] * 90, frames), _tree(9, list(range(70)), frames)]
    n = 4500
    tree_of = np.arange(n, dtype=np.int32) % len(narrow)
    tree_of[1234], tree_of[4321] = 8, 9
    batch = MatterBatch(trees, tree_of=tree_of)
    _check(batch, [trees[t] for t in tree_of], forces, [0, 1, 2, 3, 4, 5, 6, 7, 1234, 4321, 2047, n - 1])


@pytest.mark.parametrize("shape", ["narrow", "wide"])
@pytest.mark.parametrize("n", [1, 65, 4096])
@pytest.mark.parametrize("nb", [3, 20])
def test_one_tree(shape, n, nb):
    from simbody_amd.matter import MatterBatch
    parent = [0, 0] + list(range(2, nb)) if shape == "narrow" else [0] + [1 + b // 7 for b in range(nb - 1)]
    t = _tree(11, parent, True, free=shape == "wide")
    batch = MatterBatch([t], n_instances=n)
    _check(batch, [t] * n, True, sorted({0, n // 2, n - 1}))
