"""The work that is measured: batched tree dynamics through the Python mirror
of the C ABI (simbody_amd.matter, simbody_amd.serving).

Kinds of case:
  op       one or several operators of a MatterBatch at one state
  rollout  MatterBatch.stepTo from a state to a final time
  serve    a Server (chains, each request with its own constants) that admits
           requests from host memory, advances and collects them
  tserve   the same with a TreeServer (each request its own tree)

Models: "pendulum" (planar Pin links), "chain" (one spatial chain, mobilizers
Pin/Universal/Ball in turn), "free" (the same with a Free root and Sliders
among the links), "stiff" (link masses spread over four decades), "trees"
(uneven branched trees, up to 4,096 different ones in a batch).  Sizes follow
bench.py's rows and the tests: 65,536 x 32-body chains, 16,384 uneven trees of
8 to 128 bodies, one 10-link pendulum, servers of 32-body chains and of trees
of 8 to 64 bodies.
"""
import math

import numpy as np
import torch

from simbody_amd import models as M
from simbody_amd.matter import MatterBatch, RungeKuttaMerson
from simbody_amd.serving import Requests, Server, TreeRequests, TreeServer, serve

DEV = "cuda:0"
CHAIN_TYPES = (M.PIN, M.UNIVERSAL, M.BALL)
FREE_TYPES = (M.BALL, M.PIN, M.SLIDER, M.UNIVERSAL)
MAX_TREES = 4096
OPS = ("accel", "inverse", "given", "minv", "mass", "jac", "jact", "bacc", "kin", "abi", "cbi", "react")


def listed():
    return [
        # One small model stepped at high accuracy, as an interactive program
        # or a single optimizer evaluation does: launches and latency only.
        dict(name="pendulum_rollout_1x10", kind="rollout", model="pendulum", n=1, nb=10, accuracy=1e-8, h=0.0,
             t=0.1, forces=False, precision=0),
        # One realize(Acceleration) of one 32-body chain: the smallest operator call.
        dict(name="accel_chain_1x32", kind="op", ops="accel", model="chain", n=1, nb=32, forces=False),
        # Forward dynamics of a large ensemble (reinforcement learning, sampling).
        dict(name="accel_chain_65536x32", kind="op", ops="accel", model="chain", n=65536, nb=32, forces=False),
        # Inverse dynamics of the same ensemble.
        dict(name="inverse_chain_65536x32", kind="op", ops="inverse", model="chain", n=65536, nb=32, forces=False),
        # What a controller asks of one state: kinematics, forward dynamics
        # under given forces, M^-1 f, M v, J v, J^T F; an odd batch of chains
        # with a Free root, body forces, Sliders.
        dict(name="controller_free_4999x17", kind="op", ops="kin,given,minv,mass,jac,jact", model="free", n=4999,
             nb=17, forces=True),
        # Forward dynamics of an ensemble of different trees.
        dict(name="accel_trees_16384", kind="op", ops="accel", model="trees", n=16384, nb=128, forces=True),
        # Long-horizon simulation of the ensemble at a fixed step: the
        # headline rollout, sixteen steps of it.
        dict(name="rollout_chain_65536x32", kind="rollout", model="chain", n=65536, nb=32, accuracy=1e-3, h=1e-3,
             t=0.016, forces=False, precision=0),
        # Error-controlled rollout of a mid-sized odd batch with a Free root,
        # Sliders and body forces.
        dict(name="rollout_free_4001x23", kind="rollout", model="free", n=4001, nb=23, accuracy=1e-6, h=0.0, t=0.05,
             forces=True, precision=0),
        # Error-controlled rollout of 16,384 uneven trees under body forces.
        dict(name="rollout_trees_16384", kind="rollout", model="trees", n=16384, nb=128, accuracy=1e-6, h=0.0,
             t=0.02, forces=True, precision=0),
        # The ensemble rollout with the mixed-precision option.
        dict(name="mixed_chain_16384x32", kind="rollout", model="chain", n=16384, nb=32, accuracy=1e-3, h=1e-3,
             t=0.008, forces=False, precision=1),
        # A burst of rollout requests, each its own 32-body chain.
        dict(name="serve_chains_2048x32", kind="serve", model="chain", n=2048, nb=32, t=0.05),
        # A burst of rollout requests of different trees.
        dict(name="serve_trees_1024", kind="tserve", model="trees", n=1024, nb=64, t=0.05),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["op", "op", "op", "rollout", "rollout", "rollout", "serve", "tserve"])
    if kind == "op":
        model = rng.choice(["chain", "chain", "free", "trees", "pendulum", "stiff"])
        nb = _log_int(rng, 8, 128) if model == "trees" else _log_int(rng, 2, 64)
        n = _log_int(rng, 1, min(65536, (1 << 20) // nb if model == "trees" else (1 << 21) // nb))
        ops = rng.choice(["accel", "inverse", ",".join(rng.sample(OPS, 4))])
        return dict(kind=kind, ops=ops, model=model, n=n, nb=nb, forces=rng.random() < 0.5)
    if kind == "rollout":
        model = rng.choice(["chain", "chain", "free", "trees", "trees", "pendulum", "stiff"])
        nb = _log_int(rng, 8, 128) if model == "trees" else _log_int(rng, 2, 64)
        n = _log_int(rng, 1, min(65536, (1 << 20) // nb if model == "trees" else (1 << 21) // nb))
        fixed = model == "chain" and rng.random() < 0.5
        t = rng.uniform(0.005, 0.016) if fixed else rng.uniform(0.01, 0.02)
        return dict(kind=kind, model=model, n=n, nb=nb, accuracy=1e-3 if fixed else rng.choice([1e-4, 1e-6]),
                    h=1e-3 if fixed else 0.0, t=t, forces=rng.random() < 0.5,
                    precision=1 if fixed and rng.random() < 0.2 else 0)
    if kind == "serve":
        return dict(kind=kind, model="chain", n=_log_int(rng, 16, 2048), nb=_log_int(rng, 4, 40),
                    t=rng.uniform(0.02, 0.05))
    return dict(kind=kind, model="trees", n=_log_int(rng, 16, 1024), nb=_log_int(rng, 16, 64),
                t=rng.uniform(0.02, 0.05))


# ----------------------------------------------------------------------------
# Models and states
# ----------------------------------------------------------------------------
def _types(case):
    if case["model"] == "free":
        return [M.FREE] + [FREE_TYPES[i % 4] for i in range(case["nb"] - 1)]
    return [CHAIN_TYPES[i % 3] for i in range(case["nb"])]


def _tree_params(rng, count, nmin, nmax):
    """`count` uneven trees as padded arrays: bodies, parents, mobilizers (the
    same for every seed, so that results have one shape) and link constants."""
    links = _links(rng, count, nmax)
    rng = np.random.default_rng([count, nmin, nmax])
    nb = rng.integers(nmin, nmax + 1, count)
    parent = np.zeros((count, nmax), np.int32)
    for b in range(1, nmax):
        parent[:, b] = 1 + (rng.random(count) * b).astype(np.int32)
    root = rng.choice([M.PIN, M.SLIDER, M.UNIVERSAL, M.BALL, M.FREE], p=[.40, .10, .20, .25, .05], size=count)
    mob = rng.choice([M.PIN, M.SLIDER, M.UNIVERSAL, M.BALL], p=np.array([.40, .10, .20, .25]) / .95,
                     size=(count, nmax)).astype(np.int32)
    mob[:, 0] = root
    return (nb, parent, mob) + links


def _links(rng, count, nb):
    """Link constants: masses LogNormal(0, 0.5), joints U(0.2, 1) from the body
    origin, mass centers halfway, positive principal moments."""
    s = (count, nb)
    m = np.exp(0.5 * rng.standard_normal(s))
    d = rng.standard_normal(s + (3,))
    p = rng.uniform(0.2, 1.0, s + (1,)) * d / np.linalg.norm(d, axis=-1, keepdims=True)
    c = 0.5 * p
    x = rng.uniform(0.02, 0.2, s + (3,))
    mom = np.stack([x[..., 1] + x[..., 2], x[..., 0] + x[..., 2], x[..., 0] + x[..., 1]], -1)
    R = _quat_R(rng.standard_normal(s + (4,)), np)
    Ic = ((R * mom[..., None, :])[..., :, None, :] * R[..., None, :, :]).sum(-1)
    Io = m[..., None, None] * (Ic + (c * c).sum(-1)[..., None, None] * np.eye(3) - c[..., :, None] * c[..., None, :])
    I6 = np.stack([Io[..., 0, 0], Io[..., 1, 1], Io[..., 2, 2], Io[..., 0, 1], Io[..., 0, 2], Io[..., 1, 2]], -1)
    X_BM = np.zeros(s + (12,)); X_BM[..., [0, 4, 8]] = 1.0; X_BM[..., 9:] = p
    X_PF = np.zeros(s + (12,)); X_PF[..., [0, 4, 8]] = 1.0
    return m, c, I6, X_PF, X_BM


def _quat_R(q, xp):
    q = q / xp.sqrt((q * q).sum(-1))[..., None]
    w, x, y, z = q[..., 0], q[..., 1], q[..., 2], q[..., 3]
    r = [1 - 2*(y*y + z*z), 2*(x*y - w*z), 2*(x*z + w*y), 2*(x*y + w*z), 1 - 2*(x*x + z*z), 2*(y*z - w*x),
         2*(x*z - w*y), 2*(y*z + w*x), 1 - 2*(x*x + y*y)]
    return xp.stack(r, -1).reshape(tuple(w.shape) + (3, 3))


def _specs(case, rng, own=False):
    """The case's trees, and which one each instance has (None: one tree)."""
    n, nb = case["n"], case["nb"]
    if case["model"] == "pendulum":
        return [M.pendulum_chain(nb)], None
    if case["model"] == "trees" or own:
        k = n if own else min(n, MAX_TREES)
        if case["model"] == "trees":
            nbs, par, mob, m, c, I6, X_PF, X_BM = _tree_params(rng, k, min(8, nb), nb)
        else:
            nbs, par = np.full(k, nb), np.tile(np.arange(nb, dtype=np.int32), (k, 1))
            mob = np.tile(np.array(_types(case), np.int32), (k, 1))
            m, c, I6, X_PF, X_BM = _links(rng, k, nb)
        return [M.TreeSpec(parent=par[i, :b], mobilizer=mob[i, :b], mass=m[i, :b], com_B=c[i, :b],
                           inertia_B=I6[i, :b], X_PF=X_PF[i, :b], X_BM=X_BM[i, :b])
                for i, b in enumerate(nbs)], np.arange(n, dtype=np.int32) % k
    m, c, I6, X_PF, X_BM = (a[0] for a in _links(rng, 1, nb))
    if case["model"] == "stiff":
        f = 1e4 ** rng.random(nb)
        m, I6 = m * f, I6 * f[:, None]
    return [M.TreeSpec(parent=np.arange(nb, dtype=np.int32), mobilizer=np.array(_types(case), np.int32), mass=m,
                       com_B=c, inertia_B=I6, X_PF=X_PF, X_BM=X_BM)], None


def _state(rng, spec, n):
    """States of n instances of one tree: angles U(-pi, pi), translations
    U(-1, 1), unit quaternions, u ~ N(0, 1)."""
    cols = []
    for t in spec.mobilizer:
        if t in (M.BALL, M.FREE):
            q = rng.standard_normal((n, 4))
            cols.append(q / np.linalg.norm(q, axis=1, keepdims=True))
            if t == M.FREE:
                cols.append(rng.uniform(-1, 1, (n, 3)))
        elif t == M.SLIDER:
            cols.append(rng.uniform(-1, 1, (n, 1)))
        else:
            cols.append(rng.uniform(-math.pi, math.pi, (n, M.NQ[int(t)])))
    return np.concatenate(cols, 1), rng.standard_normal((n, spec.nu))


def _states(rng, specs, tree_of, n):
    """Packed q, u (instance after instance) and each instance's sizes."""
    if tree_of is None:
        q, u = _state(rng, specs[0], n)
        return q.ravel(), u.ravel()
    kinds = [s.mobilizer[np.newaxis] for s in specs]
    nq = np.array([M.NQ[t] for t in range(5)])
    dof = np.array([M.DOF[t] for t in range(5)])
    seq = np.concatenate([kinds[t][0] for t in tree_of])          # mobilizers, instance after instance
    q = np.zeros(int(nq[seq].sum()))
    at = np.concatenate([[0], np.cumsum(nq[seq])])[:-1]
    for t in range(5):
        w = at[seq == t]
        if t in (M.BALL, M.FREE):
            v = rng.standard_normal((len(w), 4))
            v /= np.linalg.norm(v, axis=1, keepdims=True)
            for j in range(4):
                q[w + j] = v[:, j]
            for j in range(4, nq[t]):
                q[w + j] = rng.uniform(-1, 1, len(w))
        else:
            for j in range(nq[t]):
                q[w + j] = rng.uniform(-1, 1, len(w)) * (1.0 if t == M.SLIDER else math.pi)
    return q, rng.standard_normal(int(dof[seq].sum()))


def _inputs(case, seed):
    """Everything a pass reads, on the host, from the seed alone."""
    rng = np.random.default_rng([seed, 20])
    own = case["kind"] in ("serve", "tserve")
    specs, tree_of = _specs(case, rng, own)
    n = case["n"]
    q, u = _states(rng, specs, tree_of, n)
    x = dict(specs=specs, tree_of=tree_of, q=q, u=u)
    if own:
        x["t_end"] = case["t"] * rng.uniform(0.2, 1.0, n)
        return x
    bodies = n * (specs[0].nb + 1) if tree_of is None else int(sum(specs[t].nb + 1 for t in tree_of))
    if case["kind"] == "op":
        x["v"] = rng.standard_normal(len(u))       # udot, f or v
        x["f"] = rng.standard_normal(len(u))       # mobility forces
    needs = case["kind"] == "op" and any(o in case["ops"] for o in ("jact", "given", "react"))
    if case["forces"] or needs:
        x["F"] = rng.standard_normal(6 * bodies)   # body forces; Ground's entries are ignored
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    specs, tree_of, n = x["specs"], x["tree_of"], case["n"]
    if case["kind"] == "serve":
        integ = RungeKuttaMerson(accuracy=1e-6)
        req = Requests(specs, x["q"].reshape(n, -1), x["u"].reshape(n, -1), x["t_end"])
        return dict(kind="serve", server=Server(specs[0], integ, 1 << 30, max_slots=max(64, n), device=DEV), req=req, n=n)
    if case["kind"] == "tserve":
        integ = RungeKuttaMerson(accuracy=1e-6)
        qo = np.concatenate([[0], np.cumsum([s.nq for s in specs])])
        uo = np.concatenate([[0], np.cumsum([s.nu for s in specs])])
        req = TreeRequests(specs, [x["q"][a:b] for a, b in zip(qo, qo[1:])],
                           [x["u"][a:b] for a, b in zip(uo, uo[1:])], x["t_end"])
        return dict(kind="tserve", server=TreeServer(integ, 1 << 30, max_slots=max(64, n), device=DEV), req=req, n=n)
    B = MatterBatch(specs, tree_of=tree_of, n_instances=n, device=DEV)
    s = dict(kind=case["kind"], B=B)
    for k in ("q", "u", "v", "f", "F"):
        s[k] = torch.as_tensor(x[k], device=DEV) if k in x else None
    if case["kind"] == "op":
        s["ops"] = case["ops"].split(",")
    else:
        s["t"] = case["t"]
        s["integ"] = RungeKuttaMerson(accuracy=case["accuracy"], fixed_step=case["h"], precision=case["precision"])
    return s


def run(s):
    if s["kind"] in ("serve", "tserve"):
        r = serve(s["server"], s["req"], np.zeros(s["n"]))
        if s["kind"] == "serve":
            return {"q": r["q"], "u": r["u"], "status": r["status"], "stats": r["stats"]}
        return {"y": np.concatenate(r["y"]), "status": r["status"], "stats": r["stats"]}
    B = s["B"]
    if s["kind"] == "rollout":
        q, u, stats = B.stepTo(s["q"], s["u"], s["integ"], s["t"], fapp=s["F"])
        return {"q": q, "u": u, "stats": stats}
    q, u, v, f, F = (s[k] for k in ("q", "u", "v", "f", "F"))
    out = {}
    for op in s["ops"]:
        if op == "accel":
            out[op] = B.realizeAcceleration(q, u, fapp=F)
        elif op == "inverse":
            out[op] = B.calcResidualForceIgnoringConstraints(q, u, F=F, udot=v)
        elif op == "given":
            out[op] = B.calcAccelerationIgnoringConstraints(q, u, f, F)
        elif op == "minv":
            out[op] = B.multiplyByMInv(q, f)
        elif op == "mass":
            out[op] = B.multiplyByM(q, v)
        elif op == "jac":
            out[op] = B.multiplyBySystemJacobian(q, v)
        elif op == "jact":
            out[op] = B.multiplyBySystemJacobianTranspose(q, F)
        elif op == "bacc":
            out[op] = B.calcBodyAccelerationFromUDot(q, u, v)
        elif op == "kin":
            out[op] = B.realizeKinematics(q, u)
        elif op == "abi":
            out[op] = B.realizeArticulatedBodyInertias(q)
        elif op == "cbi":
            # Ground's entry holds an infinite mass
            out[op] = B.calcCompositeBodyInertias(q)
        else:
            out[op] = B.calcMobilizerReactionForces(q, u, f, F)
    return out


# Flops per body that the reference quotes for its own sweeps (position,
# velocity, articulated inertia, forward dynamics, inverse dynamics, M v) for
# two-dof joints, and doubles per body of the inputs and outputs.
_POS, _VEL, _ABI, _FWD, _INV, _MASS = 90, 100, 390, 132, 141, 121
_OP_FLOPS = dict(accel=_POS + _VEL + _ABI + _FWD, given=_POS + _VEL + _ABI + _FWD, react=_POS + _VEL + _ABI + _FWD,
                 inverse=_POS + _VEL + _INV, minv=_POS + _ABI + _FWD, mass=_POS + _MASS, jac=_POS + 60,
                 jact=_POS + 60, bacc=_POS + _VEL + 60, kin=_POS + _VEL, abi=_POS + _ABI, cbi=_POS + 90)


def work(case):
    n, nb, model = case["n"], case["nb"], case["model"]
    if model == "trees":
        bodies, nq, nu = n * (min(8, nb) + nb) / 2, 2.2, 1.85       # per body, on average
        bodies_const = bodies if case["kind"] == "tserve" else min(n, MAX_TREES) * (min(8, nb) + nb) / 2
    else:
        bodies, bodies_const = n * nb, n * nb if case["kind"] == "serve" else nb
        ty = [M.PIN] * nb if model == "pendulum" else _types(case)
        nq, nu = sum(M.NQ[t] for t in ty) / nb, sum(M.DOF[t] for t in ty) / nb
    deriv = _OP_FLOPS["accel"]
    const = 23 * bodies_const                   # mass, center, inertia, frames
    force = 6 * bodies if case.get("forces") else 0
    if case["kind"] in ("serve", "tserve", "rollout"):
        # five derivatives a step; error control at 1e-6 takes about 300 steps a second
        steps = case["t"] / case["h"] if case.get("h") else 300 * case["t"] * (0.6 if "serve" in case["kind"] else 1)
        return {"bytes": 8 * (const + force + 2 * bodies * (nq + nu)), "flops": max(1, steps) * 5 * bodies * deriv}
    moved = dict(accel=2*nq + 2*nu, inverse=nq + 3*nu, given=2*nq + 3*nu + 6, minv=nq + 2*nu, mass=nq + 2*nu,
                 jac=nq + nu + 6, jact=nq + nu + 6, bacc=nq + 2*nu + 6, kin=2*nq + nu + 18, abi=nq + 42, cbi=nq + 10,
                 react=nq + 2*nu + 6)
    ops = case["ops"].split(",")
    return {"bytes": 8 * (const + sum(force * (o in ("accel", "given", "inverse", "react")) + bodies * moved[o]
                                      for o in ops)),
            "flops": sum(_OP_FLOPS[o] for o in ops) * bodies}


# ----------------------------------------------------------------------------
# The same results in plain 64-bit torch: body by body over all instances at
# once (a tree's bodies padded to the widest), dense 6x6 spatial algebra in
# Ground about each body's origin.
# ----------------------------------------------------------------------------
def _mm(A, B):
    return (A[..., :, :, None] * B[..., None, :, :]).sum(-2)


def _mv(A, x):
    return (A * x[..., None, :]).sum(-1)


def _x(a):
    z = torch.zeros_like(a[..., 0])
    return torch.stack([z, -a[..., 2], a[..., 1], a[..., 2], z, -a[..., 0], -a[..., 1], a[..., 0], z],
                       -1).reshape(a.shape[:-1] + (3, 3))


def _cr(a, b):
    return torch.linalg.cross(a, b)


class _Exact:
    """Instances of the given trees, with packed states padded to rows."""

    def __init__(self, specs, tree_of, n):
        self.dev = "cuda:0" if torch.cuda.is_available() else "cpu"
        T, nb = len(specs), max(s.nb for s in specs)
        self.nb = nb
        a = dict(parent=np.zeros((T, nb), np.int64), ty=np.full((T, nb), -1, np.int64), m=np.zeros((T, nb)),
                 c=np.zeros((T, nb, 3)), I=np.zeros((T, nb, 6)), PF=np.zeros((T, nb, 12)), BM=np.zeros((T, nb, 12)),
                 qi=np.zeros((T, nb), np.int64), ui=np.zeros((T, nb), np.int64), g=np.zeros((T, 3)))
        for i, s in enumerate(specs):
            k = s.nb
            a["parent"][i, :k], a["ty"][i, :k], a["m"][i, :k], a["c"][i, :k] = s.parent, s.mobilizer, s.mass, s.com_B
            a["I"][i, :k], a["PF"][i, :k], a["BM"][i, :k], a["g"][i] = s.inertia_B, s.X_PF, s.X_BM, s.gravity
            a["qi"][i, :k], a["ui"][i, :k] = s.offsets()
        of = np.zeros(n, np.int64) if tree_of is None else np.asarray(tree_of, np.int64)
        self.one = tree_of is None          # one topology: no gathers by instance
        self.of = torch.as_tensor(of, device=self.dev)
        self.t = {k: torch.as_tensor(v, device=self.dev) for k, v in a.items()}
        self.n = n
        self.nq = np.array([s.nq for s in specs])[of]; self.nu = np.array([s.nu for s in specs])[of]
        self.nbs = np.array([s.nb for s in specs])[of]
        self.rows = torch.arange(n, device=self.dev)
        self.live = torch.as_tensor(self.nbs, device=self.dev)

    def pad(self, packed, sizes, width=1):
        sizes = np.asarray(sizes) * width
        off = np.concatenate([[0], np.cumsum(sizes)[:-1]])
        k = int(sizes.max()) if len(sizes) else 0
        idx = off[:, None] + np.arange(max(k, 1))[None, :]
        ok = np.arange(max(k, 1))[None, :] < sizes[:, None]
        x = np.asarray(packed)[np.where(ok, idx, 0)] * ok
        return torch.as_tensor(x, device=self.dev)

    def pack(self, x, sizes, width=1):
        sizes = torch.as_tensor(np.asarray(sizes) * width, device=self.dev)
        return x[torch.arange(x.shape[1], device=self.dev)[None, :] < sizes[:, None]]

    def const(self, key, b):
        return self.t[key][:, b][self.of]

    def parent_of(self, X, b):
        return X[self.rows, self.const("parent", b)]

    def kin(self, q, u):
        """Sweeps base to tip; keeps R, p, V, H, the shift and the bias
        accelerations per body (index 0 is Ground).  Returns qdot."""
        n, nb, dev = self.n, self.nb, self.dev
        z = lambda *s: torch.zeros((n, nb + 1) + s, dtype=torch.float64, device=dev)  # noqa: E731
        self.R, self.p, self.V, self.H, self.l, self.a = z(3, 3), z(3), z(6), z(6, 6), z(3), z(6)
        self.P, self.bias = z(6, 6), z(6)
        self.R[:, 0] = torch.eye(3, dtype=torch.float64, device=dev)
        qd = torch.zeros_like(q)
        pad7 = torch.cat([q, torch.zeros(n, 7, dtype=q.dtype, device=dev)], 1)
        pad6 = torch.cat([u, torch.zeros(n, 6, dtype=q.dtype, device=dev)], 1)
        e = torch.eye(3, dtype=torch.float64, device=dev)
        self.dof = torch.zeros((n, nb + 1), dtype=torch.int64, device=dev)
        for b in range(nb):
            ty, qi, ui = self.const("ty", b), self.const("qi", b), self.const("ui", b)
            x = pad7.gather(1, qi[:, None] + torch.arange(7, device=dev))
            w = pad6.gather(1, ui[:, None] + torch.arange(6, device=dev))
            pin, sl, un, ball, free = (ty == k for k in range(5))
            quat = ball | free
            d = torch.tensor([1, 1, 2, 3, 6, 0], device=dev)[ty]
            self.dof[:, b + 1] = d
            w = w * (torch.arange(6, device=dev)[None, :] < d[:, None])
            ax = torch.where(un, x[:, 0], torch.zeros_like(x[:, 0])); ay = torch.where(un, x[:, 1], ax * 0)
            az = torch.where(pin, x[:, 0], ax * 0)
            o, zz = torch.ones_like(ax), torch.zeros_like(ax)
            cx, sx, cy, sy, cz, sz = ax.cos(), ax.sin(), ay.cos(), ay.sin(), az.cos(), az.sin()
            Rx = torch.stack([o, zz, zz, zz, cx, -sx, zz, sx, cx], -1).reshape(n, 3, 3)
            Ry = torch.stack([cy, zz, sy, zz, o, zz, -sy, zz, cy], -1).reshape(n, 3, 3)
            Rz = torch.stack([cz, -sz, zz, sz, cz, zz, zz, zz, o], -1).reshape(n, 3, 3)
            Rq = _quat_R(torch.where(quat[:, None], x[:, :4], torch.tensor([1., 0, 0, 0], dtype=q.dtype, device=dev)),
                         torch)
            R_FM = _mm(_mm(_mm(Rx, Ry), Rz), Rq)
            p_FM = torch.where(free[:, None], x[:, 4:7], torch.where(sl[:, None], x[:, :1] * e[0], zz[:, None]))
            H = torch.zeros((n, 6, 6), dtype=torch.float64, device=dev)      # [spatial, dof]
            H[:, :3, 0] = torch.where(pin[:, None], e[2], torch.where((un | quat)[:, None], e[0], zz[:, None]))
            H[:, :3, 1] = torch.where(un[:, None], R_FM[:, :, 1], torch.where(quat[:, None], e[1], zz[:, None]))
            H[:, :3, 2] = torch.where(quat[:, None], e[2], zz[:, None])
            H[:, 3:, 0] = torch.where(sl[:, None], e[0], zz[:, None])
            for k in range(3):
                H[:, 3:, 3 + k] = torch.where(free[:, None], e[k], zz[:, None])
            PF, BM = self.const("PF", b), self.const("BM", b)
            R_PF, p_PF = PF[:, :9].reshape(n, 3, 3), PF[:, 9:]
            R_MB = BM[:, :9].reshape(n, 3, 3).transpose(1, 2)
            p_MB = -_mv(R_MB, BM[:, 9:])
            r = _mv(R_FM, p_MB)
            R_P, p_P, V_P = self.parent_of(self.R, b), self.parent_of(self.p, b), self.parent_of(self.V, b)
            R_GF = _mm(R_P, R_PF)
            lv = _mv(R_P, p_PF) + _mv(R_GF, p_FM + r)
            Hw = _mm(R_GF, H[:, :3]); Hv = _mm(R_GF, H[:, 3:] - _mm(_x(r), H[:, :3]))
            HG = torch.cat([Hw, Hv], 1)
            wF, vF = _mv(H[:, :3], w), _mv(H[:, 3:], w)
            ab = torch.where(un[:, None], _cr(wF, H[:, :3, 1]) * w[:, 1:2], zz[:, None])     # HDot u, angular
            wP = V_P[:, :3]
            rel = _mv(HG, w)
            V = torch.cat([wP + rel[:, :3], V_P[:, 3:] + _cr(wP, lv) + rel[:, 3:]], 1)
            aw = _mv(R_GF, ab) + _cr(wP, rel[:, :3])
            # parent's centripetal term, Coriolis term and the joint's own
            av = (_cr(wP, _cr(wP, lv)) + 2 * _cr(wP, rel[:, 3:]) + _mv(R_GF, _cr(wF, _cr(wF, r)) + _cr(ab, r)))
            Rb = _mm(_mm(R_GF, R_FM), R_MB)
            c = _mv(Rb, self.const("c", b)); m = self.const("m", b)
            I = self.const("I", b)
            Ib = torch.stack([I[:, 0], I[:, 3], I[:, 4], I[:, 3], I[:, 1], I[:, 5], I[:, 4], I[:, 5], I[:, 2]],
                             -1).reshape(n, 3, 3)
            Ig = _mm(_mm(Rb, Ib), Rb.transpose(1, 2))
            cx_ = m[:, None, None] * _x(c)
            P = torch.cat([torch.cat([Ig, cx_], 2), torch.cat([-cx_, m[:, None, None] * e.expand(n, 3, 3)], 2)], 1)
            bg = torch.cat([_cr(V[:, :3], _mv(Ig, V[:, :3])), m[:, None] * _cr(V[:, :3], _cr(V[:, :3], c))], 1)
            k = b + 1
            self.R[:, k], self.p[:, k], self.V[:, k], self.H[:, k], self.l[:, k] = Rb, p_P + lv, V, HG, lv
            self.a[:, k], self.P[:, k], self.bias[:, k] = torch.cat([aw, av], 1), P, bg
            x0, x1, x2, x3 = (0.5 * x[:, j] for j in range(4))
            w0, w1, w2 = w[:, 0], w[:, 1], w[:, 2]
            Nq = torch.stack([-x1*w0 - x2*w1 - x3*w2, x0*w0 + x3*w1 - x2*w2, -x3*w0 + x0*w1 + x1*w2,
                              x2*w0 - x1*w1 + x0*w2], -1)
            full = torch.where(quat[:, None], torch.cat([Nq, w[:, 3:6]], 1), torch.cat([w, w[:, :1] * 0], 1))
            nqk = torch.tensor([1, 1, 2, 4, 7, 0], device=dev)[ty]
            for j in range(7):
                ok = nqk > j
                qd[self.rows[ok], qi[ok] + j] = full[ok, j]
        return qd

    def shift(self, b):
        S = torch.eye(6, dtype=torch.float64, device=self.dev).repeat(self.n, 1, 1)
        S[:, :3, 3:] = _x(self.l[:, b])
        return S

    def gravity(self, b):
        m = self.P[:, b, 5, 5]
        f = m[:, None] * self.t["g"][self.of]
        c = torch.stack([self.P[:, b, 2, 4], self.P[:, b, 0, 5], self.P[:, b, 1, 3]], -1)
        return torch.cat([_cr(c, self.t["g"][self.of]), f], 1), c

    def take(self, x, b, width):
        """The dof-padded entries of body b (0-based) of padded rows x."""
        xx = torch.cat([x, torch.zeros(self.n, 6, dtype=x.dtype, device=self.dev)], 1)
        v = xx.gather(1, self.const("ui", b)[:, None] + torch.arange(6, device=self.dev))
        return v * (torch.arange(6, device=self.dev)[None, :] < self.dof[:, b + 1][:, None])

    def put(self, out, b, v):
        for j in range(6):
            ok = self.dof[:, b + 1] > j
            out[self.rows[ok], self.const("ui", b)[ok] + j] = v[ok, j]

    def forward(self, f, F, gravity=True, bias=True):
        """Articulated-body algorithm on the last kin().  Returns udot, A_GB,
        P, P+ and the forces transmitted at each body's origin."""
        n, nb, dev = self.n, self.nb, self.dev
        P = self.P.clone()
        z = torch.zeros((n, nb + 1, 6), dtype=torch.float64, device=dev)
        PP, zp = torch.zeros_like(P), torch.zeros_like(z)
        G, DIe, DI = torch.zeros_like(P), torch.zeros_like(z), None
        for k in range(nb, 0, -1):
            b = k - 1
            H = self.H[:, k]
            if bias:
                z[:, k] += _mv(P[:, k], self.a[:, k]) + self.bias[:, k]
            if F is not None:
                z[:, k] -= F[:, 6*k:6*k + 6]
            if gravity:
                z[:, k] -= self.gravity(k)[0]
            PH = _mm(P[:, k], H)
            D = _mm(H.transpose(1, 2), PH)
            pad = (torch.arange(6, device=dev)[None, :] >= self.dof[:, k][:, None]).double()
            DI = torch.linalg.inv(D + torch.diag_embed(pad))
            G[:, k] = _mm(PH, DI)
            eps = (self.take(f, b, 6) if f is not None else 0.0) - _mv(H.transpose(1, 2), z[:, k])
            DIe[:, k] = _mv(DI, eps)
            X = P[:, k] - _mm(G[:, k], PH.transpose(1, 2))
            PP[:, k] = 0.5 * (X + X.transpose(1, 2))       # asymmetry would grow from body to body
            zp[:, k] = z[:, k] + _mv(G[:, k], eps)
            S, par = self.shift(k), self.const("parent", b)
            live = (self.live >= k).double()
            P[self.rows, par] += live[:, None, None] * _mm(_mm(S, PP[:, k]), S.transpose(1, 2))
            z[self.rows, par] += live[:, None] * _mv(S, zp[:, k])
        A, udot = torch.zeros_like(z), torch.zeros((n, int(self.nu.max())), dtype=torch.float64, device=dev)
        T = torch.zeros_like(z)
        for k in range(1, nb + 1):
            Ap = _mv(self.shift(k).transpose(1, 2), self.parent_of(A, k - 1))
            ud = DIe[:, k] - _mv(G[:, k].transpose(1, 2), Ap)
            A[:, k] = Ap + _mv(self.H[:, k], ud) + (self.a[:, k] if bias else 0.0)
            T[:, k] = _mv(PP[:, k], Ap) + zp[:, k]
            self.put(udot, k - 1, ud)
        return udot, A, P, PP, T

    def outward(self, v, bias):
        A = torch.zeros((self.n, self.nb + 1, 6), dtype=torch.float64, device=self.dev)
        for k in range(1, self.nb + 1):
            Ap = _mv(self.shift(k).transpose(1, 2), self.parent_of(A, k - 1))
            A[:, k] = Ap + _mv(self.H[:, k], self.take(v, k - 1, 6)) + (self.a[:, k] if bias else 0.0)
        return A

    def inward(self, F):
        """H^T of the forces F [n, nb+1, 6] gathered tip to base."""
        F = F.clone()
        tau = torch.zeros((self.n, int(self.nu.max())), dtype=torch.float64, device=self.dev)
        for k in range(self.nb, 0, -1):
            self.put(tau, k - 1, _mv(self.H[:, k].transpose(1, 2), F[:, k]))
            live = (self.live >= k).double()
            F[self.rows, self.const("parent", k - 1)] += live[:, None] * _mv(self.shift(k), F[:, k])
        return tau

    def derivative(self, q, u, F):
        qd = self.kin(q, u)
        return qd, self.forward(None, F)[0]


def _exact_op(E, case, q, u, v, f, F, F_packed):
    n, nb = E.n, E.nb
    out = {}
    body = lambda X, w: E.pack(X.reshape(n, -1), E.nbs + 1, w)  # noqa: E731
    sym = [(0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)]

    def abi(P):
        cols = [P[..., 3 + i, 3 + j] for i, j in sym] + [P[..., i, j] for i, j in sym]
        return torch.stack(cols + [P[..., i, 3 + j] for i in range(3) for j in range(3)], -1)

    for op in case["ops"].split(","):
        qd = E.kin(q, u if op in ("accel", "given", "inverse", "bacc", "kin", "react") else u * 0)
        if op == "accel":
            out[op] = (E.pack(E.forward(None, F)[0], E.nu), E.pack(qd, E.nq))
        elif op == "given":
            ud, A = E.forward(f, F, gravity=False)[:2]
            qdd = torch.zeros_like(q)
            pad7 = torch.cat([q, torch.zeros(n, 7, dtype=q.dtype, device=q.device)], 1)
            for b in range(nb):
                ty, qi = E.const("ty", b), E.const("qi", b)
                a, w = E.take(ud, b, 6), E.take(u, b, 6)
                x = pad7.gather(1, qi[:, None] + torch.arange(7, device=q.device))
                quat = (ty == M.BALL) | (ty == M.FREE)
                h = [0.5 * x[:, j] for j in range(4)]
                s = -0.25 * (w[:, :3] * w[:, :3]).sum(-1)
                N = torch.stack([-h[1]*a[:, 0] - h[2]*a[:, 1] - h[3]*a[:, 2], h[0]*a[:, 0] + h[3]*a[:, 1] - h[2]*a[:, 2],
                                 -h[3]*a[:, 0] + h[0]*a[:, 1] + h[1]*a[:, 2], h[2]*a[:, 0] - h[1]*a[:, 1] + h[0]*a[:, 2]],
                                -1) + s[:, None] * x[:, :4]
                full = torch.where(quat[:, None], torch.cat([N, a[:, 3:6]], 1), torch.cat([a, a[:, :1] * 0], 1))
                nqk = torch.tensor([1, 1, 2, 4, 7, 0], device=q.device)[ty]
                for j in range(7):
                    ok = nqk > j
                    qdd[E.rows[ok], qi[ok] + j] = full[ok, j]
            out[op] = (E.pack(ud, E.nu), body(A, 6), E.pack(qdd, E.nq))
        elif op == "minv":
            out[op] = E.pack(E.forward(f, None, gravity=False, bias=False)[0], E.nu)
        elif op in ("mass", "inverse"):
            A = E.outward(v, op == "inverse")
            W = _mv(E.P, A)
            if op == "inverse":
                W = W + E.bias
                if F is not None:
                    W = W - F.reshape(n, nb + 1, 6)
            out[op] = E.pack(E.inward(W), E.nu)
        elif op in ("jac", "bacc"):
            out[op] = body(E.outward(v, op == "bacc"), 6)
        elif op == "jact":
            out[op] = E.pack(E.inward(F_packed.reshape(n, nb + 1, 6)), E.nu)
        elif op == "kin":
            ke = 0.5 * (E.V * _mv(E.P, E.V)).sum((-1, -2))
            pe = sum(-(E.P[:, k, 5, 5][:, None] * E.t["g"][E.of] * (E.p[:, k] + E.gravity(k)[1]
                       / E.P[:, k, 5, 5].clamp_min(1e-300)[:, None])).sum(-1) for k in range(1, nb + 1))
            X = torch.cat([E.R.reshape(n, nb + 1, 9), E.p], -1)
            out[op] = (body(X, 12), body(E.V, 6), E.pack(qd, E.nq), torch.stack([ke, pe], -1).reshape(-1))
        elif op == "abi":
            P, PP = E.forward(None, None, gravity=False, bias=False)[2:4]
            P[:, 0] = 0
            out[op] = (body(abi(P), 21), body(abi(PP), 21))
        elif op == "react":
            T = E.forward(f, F, gravity=False)[4]
            for k in range(1, nb + 1):
                pm = _mv(E.R[:, k], E.const("BM", k - 1)[:, 9:])
                T[:, k, :3] -= _cr(pm, T[:, k, 3:])
            T[:, 0] = 0
            out[op] = body(T, 6)
        else:
            out[op] = None
    return out


def _norm(e, y1, E):
    """Sums over each instance's q of the weighted error estimate: quaternion
    entries through N N^-1, the others as they are."""
    n, dev = E.n, E.dev
    e7 = torch.cat([e, torch.zeros(n, 7, dtype=e.dtype, device=dev)], 1)
    y7 = torch.cat([y1, torch.zeros(n, 7, dtype=e.dtype, device=dev)], 1)
    total = torch.zeros(n, dtype=e.dtype, device=dev)
    for b in range(E.nb):
        ty, idx = E.const("ty", b), E.const("qi", b)[:, None] + torch.arange(7, device=dev)
        quat = (ty == M.BALL) | (ty == M.FREE)
        nqk = torch.tensor([1, 1, 2, 4, 7, 0], device=dev)[ty]
        ee = e7.gather(1, idx) * (torch.arange(7, device=dev)[None, :] < nqk[:, None])
        y = y7.gather(1, idx)[:, :4]
        # N N^-1 e = |q|^2 e - q (q . e)
        w = (y * y).sum(-1, keepdim=True) * ee[:, :4] - y * (y * ee[:, :4]).sum(-1, keepdim=True)
        total += torch.where(quat, (w * w).sum(-1) + (ee[:, 4:] ** 2).sum(-1), (ee * ee).sum(-1))
    return total


def exact(case, seed):
    n, nb = case["n"], case["nb"]
    if case["kind"] in ("serve", "tserve") or n * (nb + 1) > 2.5e6:
        return None
    most = 20 if case["kind"] == "op" else 1600 // nb          # attempted steps within about 20 s
    x = _inputs(case, seed)
    E = _Exact(x["specs"], x["tree_of"], n)
    q, u = E.pad(x["q"], E.nq), E.pad(x["u"], E.nu)
    F = E.pad(x["F"], E.nbs + 1, 6) if "F" in x else None
    with torch.no_grad():
        if case["kind"] == "op":
            pad = lambda k: E.pad(x[k], E.nu)  # noqa: E731
            return _exact_op(E, case, q, u, pad("v"), pad("f"), F, F)
        # Merson's method under the reference's step control; the quaternions
        # of a state are normalized where their error passes the tolerance.
        acc, fixed, end = case["accuracy"], case["h"], case["t"]
        tol = acc / 10
        quats = torch.stack([(E.const("ty", b) == M.BALL) | (E.const("ty", b) == M.FREE) for b in range(nb)], 1)
        qis = torch.stack([E.const("qi", b) for b in range(nb)], 1)
        nquat = quats.sum(1)
        dev, f8 = E.dev, torch.float64
        nq, nu = (torch.as_tensor(s, device=dev).to(f8) for s in (E.nq, E.nu))
        t = torch.zeros(n, dtype=f8, device=dev)
        h = torch.full((n,), fixed or 0.01, dtype=f8, device=dev)
        for _ in range(most):
            go = t < end
            if not bool(go.any()):
                return {"q": E.pack(q, E.nq), "u": E.pack(u, E.nu), "stats": None}
            limited = end < t + 0.95 * h
            t1 = torch.where(~limited & (end > t + 1.001 * h), t + h, torch.full_like(t, end))
            step = torch.where(go, t1 - t, torch.zeros_like(t))[:, None]

            def at(*terms):
                return tuple(y + step * sum(c * f[j] for c, f in terms) for j, y in enumerate((q, u)))

            f0 = E.derivative(q, u, F)
            f1 = E.derivative(*at((1/3, f0)), F)
            f2 = E.derivative(*at((1/6, f0), (1/6, f1)), F)
            f3 = E.derivative(*at((1/8, f0), (3/8, f2)), F)
            ys = at((1/2, f0), (-3/2, f2), (2, f3))
            f4 = E.derivative(*ys, F)
            q1, u1 = at((1/6, f0), (4/6, f3), (1/6, f4))
            eq, eu = 0.2 * (q1 - ys[0]).abs(), 0.2 * (u1 - ys[1]).abs()
            eu = eu / u.abs().clamp_min(1.0)
            un = ((eu * eu).sum(1) / nu).sqrt()
            e1 = torch.maximum((_norm(eq, q1, E) / nq).sqrt(), un)
            err = e1.clone()
            gate = (e1 <= 16 * acc) & (nquat > 0)
            q7 = torch.cat([q1, torch.ones(n, 4, dtype=f8, device=dev)], 1)
            idx = qis[:, :, None] + torch.arange(4, device=dev)
            quat = q7.gather(1, idx.reshape(n, -1)).reshape(n, nb, 4)
            off = torch.where(quats, quat.square().sum(-1).sqrt() - 1, torch.zeros_like(quat[..., 0]))
            qe = (off.square().sum(1) / nquat.clamp_min(1)).sqrt()
            err[gate & (qe > max(2 * tol, math.sqrt(tol)))] = math.inf
            proj = gate & (qe > tol) & (qe <= max(2 * tol, math.sqrt(tol)))
            if bool(proj.any()):
                for b in range(nb):
                    w = (proj & quats[:, b]).nonzero()[:, 0]
                    i = qis[w, b][:, None] + torch.arange(4, device=dev)
                    z = q1[w].gather(1, i)
                    z = z / z.square().sum(-1, keepdim=True).sqrt()
                    e = eq[w].gather(1, i)
                    q1[w[:, None], i] = z
                    eq[w[:, None], i] = e - z * (z * e).sum(-1, keepdim=True)
                err = torch.where(proj, torch.maximum((_norm(eq, q1, E) / nq).sqrt(), un), err)
            new = torch.where(err == 0, 5 * h, 0.9 * h * (acc / err).pow(0.25))
            new = torch.where(torch.isfinite(err), new, 0.1 * h)
            new = torch.where((new > h) & (limited | (new < 1.2 * h)), h, new)
            new = torch.where(new < h, torch.where(err <= acc, h, torch.minimum(new, 0.9 * h)), new)
            new = torch.maximum(torch.minimum(new, 5 * h), 0.1 * h)
            if fixed:
                new = torch.full_like(h, fixed)
            ok = go & (new >= h)
            h = torch.where(go, new, h)
            t = torch.where(ok, t1, t)
            q, u = torch.where(ok[:, None], q1, q), torch.where(ok[:, None], u1, u)
    return None
