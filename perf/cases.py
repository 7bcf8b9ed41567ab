"""Performance cases: what a user of the framework has it do, through its public entry points.

Kinds of case
  step      frames of AffineBodySimulator: its native frame driver, or the driver that calls
            the stages one by one from Python ("driver": "python").  One pass restores the frame-start
            state (a checkpoint) and advances "frames" frames; the outputs are the
            advanced state, the posed vertices and the Newton iterations of every frame.
  rollout   a simulated trajectory and its gradient with respect to the initial velocities
            (RolloutFunction forward and backward).
  collide   the collision set of a state (boxes, body pairs, PT / EE / VG lists) and the CCD
            step bound of a given Newton step.
  assemble  energies, gradient and Hessian of the frame energy over given candidate lists.
  solve     one Newton system (BSR) solved by a named method.

Scenes are columns of bodies, a gap of about one contact distance (dhat) between neighbours
and above the floor, so that contacts are active from the first Newton iterations on.
Mesh mixes: "cube" (8 vertices), "sphere" (icosphere-3, 642), "coarse" (cube, icosphere-2,
6x6x6 box: the batched benchmark's), "fine" (cube, icosphere-3, icosphere-4 ellipsoid: the
1024-body benchmark's).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "abd-warp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from abd_hip import scenes as _scenes  # noqa: E402
from abd_hip.const_params import ContactParams  # noqa: E402

DHAT = 1e-3
DEV = "cuda"


def listed():
    return [
        # the reference's own configuration: two unit cubes, one on the other, its solver and
        # Hessian (BiCGSTAB, unprojected): the smallest call, all latency
        dict(name="step 2 cubes", kind="step", driver="native", scenes=1, bodies_lo=2, bodies_hi=2, mix="cube",
             psd=0, solver=0, frames=4),
        # an interactive scene: 64 spheres, the stable mode with the direct solve
        dict(name="step 64 spheres", kind="step", driver="native", scenes=1, bodies_lo=64, bodies_hi=64,
             mix="sphere", psd=1, solver=3, frames=2),
        # the headline workload: 256 independent scenes of 2 to 64 bodies advanced together
        dict(name="step 256 scenes", kind="step", driver="native", scenes=256, bodies_lo=2, bodies_hi=64,
             mix="coarse", psd=1, solver=3, frames=3),
        # an ordinary batch with the reference's solver (Jacobi CG)
        dict(name="step 61 scenes cg", kind="step", driver="native", scenes=61, bodies_lo=2, bodies_hi=40,
             mix="coarse", psd=1, solver=1, frames=2),
        # one large scene: 1024 bodies and a million vertices (above the direct solve's 64 bodies)
        dict(name="step pile 1024", kind="step", driver="native", scenes=1, bodies_lo=1024, bodies_hi=1024,
             mix="fine", psd=1, solver=3, frames=2),
        # a few large scenes advanced together
        dict(name="step 8 piles of 128", kind="step", driver="native", scenes=8, bodies_lo=128, bodies_hi=128,
             mix="fine", psd=1, solver=3, frames=2),
        # the full IPC contact model (closest features, mollified edges, per-contact projection)
        dict(name="step full ipc", kind="step", driver="native", scenes=24, bodies_lo=4, bodies_hi=32,
             mix="coarse", psd=3, solver=3, frames=2),
        # the driver written against the stage entry points (the reference's own call shapes)
        dict(name="step python 27 spheres", kind="step", driver="python", scenes=1, bodies_lo=27, bodies_hi=27,
             mix="sphere", psd=1, solver=3, frames=1),
        # optimisation through the simulation: a drop onto the floor and its adjoint
        dict(name="rollout 16 spheres", kind="rollout", bodies=16, frames=20),
        # culling and CCD of a large scene called as stages
        dict(name="collide 1024", kind="collide", bodies=1024, mix="fine"),
        # gradient and Hessian assembly of a large scene called as a stage
        dict(name="assemble 700", kind="assemble", bodies=700, mix="coarse"),
        # one direct solve at the largest size it takes
        dict(name="solve 64 bodies", kind="solve", bodies=64, method="ldlt"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(["plain", "plain", "batch", "batch", "python", "rollout", "collide", "assemble", "solve"])
    if k == "plain":
        mix = rng.choice(["cube", "sphere", "coarse", "fine"])
        n = _log_int(rng, 2, 900 if mix != "sphere" else 400)
        psd = rng.choice([1, 1, 1, 3]) if n > 2 else 0
        return dict(kind="step", driver="native", scenes=1, bodies_lo=n, bodies_hi=n, mix=mix, psd=psd,
                    solver=0 if psd == 0 else rng.choice([2, 3, 3]), frames=rng.randint(1, 3))
    if k == "batch":
        s = _log_int(rng, 3, 230)
        lo = rng.randint(2, 12)
        return dict(kind="step", driver="native", scenes=s, bodies_lo=lo, bodies_hi=lo + rng.randint(0, 50),
                    mix=rng.choice(["cube", "coarse", "coarse"]), psd=rng.choice([1, 1, 1, 3]),
                    solver=rng.choice([1, 2, 3, 3, 3]), frames=rng.randint(1, 3))
    if k == "python":
        n = _log_int(rng, 3, 60)
        return dict(kind="step", driver="python", scenes=1, bodies_lo=n, bodies_hi=n,
                    mix=rng.choice(["sphere", "coarse"]), psd=1, solver=rng.choice([1, 3]), frames=1)
    if k == "rollout":
        return dict(kind="rollout", bodies=rng.randint(3, 24), frames=rng.randint(8, 20))
    if k == "collide":
        return dict(kind="collide", bodies=_log_int(rng, 20, 1000), mix=rng.choice(["coarse", "fine"]))
    if k == "assemble":
        return dict(kind="assemble", bodies=_log_int(rng, 20, 700), mix=rng.choice(["coarse", "sphere"]))
    method = rng.choice(["ldlt", "cg", "cg_block"])
    return dict(kind="solve", bodies=rng.randint(5, 64) if method == "ldlt" else _log_int(rng, 20, 1000),
                method=method)


# ------------------------------------------------------------------------------- scenes
_LIB = {}


def _mesh(name):
    """(vertices, triangles, edges) of a base mesh, built once per process."""
    if name not in _LIB:
        V, F = {"cube": _scenes.cube_mesh, "ico2": lambda: _scenes.icosphere_mesh(2, 0.5),
                "ico3": lambda: _scenes.icosphere_mesh(3, 0.5), "ico4": lambda: _scenes.icosphere_mesh(4, 1.0),
                "box6": lambda: _scenes.subdivided_box_mesh(6)}[name]()
        _LIB[name] = (V, F, _scenes.edges_of(F))
    return _LIB[name]


_MIX = {"cube": ["cube"], "sphere": ["ico3"], "coarse": ["cube", "ico2", "box6"], "fine": ["cube", "ico3", "ico4"]}


def _bodies(case):
    """(scene, mesh name) of every body: a function of the case alone, so that states of
    different seeds have the same sizes."""
    if case["kind"] == "step":
        s, lo, hi, mix = case["scenes"], case["bodies_lo"], case["bodies_hi"], case["mix"]
    else:
        s, lo, hi, mix = 1, case["bodies"], case["bodies"], case["mix"]
    rng = np.random.default_rng([7, s, lo, hi])
    out = []
    for k in range(s):
        names = _MIX[mix]
        pick = rng.integers(0, len(names), size=int(rng.integers(lo, hi + 1)))
        out += [(k, names[int(i)]) for i in pick]
    return out


def _columns(case, seed, gap, speed):
    """A SceneSpec of the case's bodies in columns (see the module's docstring)."""
    rng = np.random.default_rng([seed, 11])
    bodies = _bodies(case)
    nb = len(bodies)
    scene = np.array([s for s, _ in bodies], np.int32)
    per_scene = np.bincount(scene)
    fine = case["mix"] == "fine"
    pitch = 1.75 if fine else 1.2
    xs, fs, es = [], [], []
    p = np.zeros((nb, 3))
    A = np.zeros((nb, 3, 3))
    yaw = rng.uniform(-0.1, 0.1, nb)
    tilt = rng.uniform(-1e-4, 1e-4, (nb, 2))
    shift = rng.uniform(-0.01, 0.01, (nb, 2))
    gaps = rng.uniform(gap[0], gap[1], nb) * DHAT
    radii = rng.uniform(0.3, 0.8, (nb, 3))
    where = rng.random(nb)
    # rotations: a yaw, then a tilt too small to matter but for the contacts' generality
    c, w, z, o = np.cos(yaw), np.sin(yaw), np.zeros(nb), np.ones(nb)
    tx, tz = tilt[:, 0], tilt[:, 1]
    R = np.stack([c, z, w, z, o, z, -w, z, c], 1).reshape(-1, 3, 3)
    Q, U = np.linalg.qr(R @ np.stack([o, -tz, z, tz, o, -tx, z, tx, o], 1).reshape(-1, 3, 3))
    A[:] = Q * np.sign(np.diagonal(U, axis1=1, axis2=2))[:, None, :]
    heights = {}
    for b, (s, name) in enumerate(bodies):
        V, F, E = _mesh(name)
        if name == "ico4":
            V = V * radii[b][None, :]
        side = max(1, int(math.sqrt(per_scene[s] / (10.0 if per_scene[s] > 200 else 4.0))))
        cell = int(where[b] * side * side)
        y = V @ A[b][:, 1]
        y0, y1 = float(y.min()), float(y.max())
        top = heights.get((s, cell), 0.0) + gaps[b]
        p[b] = (pitch * (cell % side) + shift[b, 0] + 40.0 * s, top - y0, pitch * (cell // side) + shift[b, 1])
        heights[(s, cell)] = top + (y1 - y0)
        xs.append(V)
        fs.append(F)
        es.append(E)
    off = lambda a: np.concatenate([[0], np.cumsum([len(v) for v in a])]).astype(np.int32)  # noqa: E731
    d = rng.normal(size=(nb, 3))
    pdot = d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(0.0, speed, (nb, 1))
    return _scenes.SceneSpec(
        x0=np.ascontiguousarray(np.concatenate(xs)), tris=np.concatenate(fs).astype(np.int32),
        edges=np.concatenate(es).astype(np.int32), voff=off(xs), foff=off(fs), eoff=off(es), A=A, p=p,
        Adot=np.zeros((nb, 3, 3)), pdot=pdot, mass=np.full(nb, 1e3), I0=np.full(nb, 1e2), body_scene=scene,
        ground=0.0, name="columns")


def _drop(case, seed):
    """Spheres above a floor, each falling freely until it lands."""
    rng = np.random.default_rng([seed, 12])
    n = case["bodies"]
    V, F, E = _mesh("ico2")
    side = int(math.ceil(math.sqrt(n)))
    p = np.array([[1.5 * (i % side), 0.5 + rng.uniform(0.02, 0.1), 1.5 * (i // side)] for i in range(n)])
    off = lambda m: (np.arange(n + 1) * m).astype(np.int32)  # noqa: E731
    return _scenes.SceneSpec(
        x0=np.tile(V, (n, 1)), tris=np.tile(F, (n, 1)), edges=np.tile(E, (n, 1)), voff=off(len(V)), foff=off(len(F)),
        eoff=off(len(E)), A=np.stack([np.eye(3)] * n), p=p, Adot=np.zeros((n, 3, 3)),
        pdot=rng.uniform(-0.5, 0.5, (n, 3)), mass=np.full(n, 1e3), I0=np.full(n, 1e2),
        body_scene=np.zeros(n, np.int32), ground=0.0, name="drop")


def _pose(spec, A, p):
    body = np.repeat(np.arange(spec.n_bodies), np.diff(spec.voff))
    return np.einsum("vr,vrk->vk", spec.x0, A[body]) + p[body]


# -------------------------------------------------- candidates, without the framework
def _body_pairs(spec, x, x1=None):
    """Pairs i < j of bodies whose boxes, dilated by dhat / 2, overlap, sorted by (i, j)."""
    at = spec.voff[:-1]
    lo, hi = np.minimum.reduceat(x, at) - 0.5 * DHAT, np.maximum.reduceat(x, at) + 0.5 * DHAT
    if x1 is not None:
        lo = np.minimum(lo, np.minimum.reduceat(x1, at) - 0.5 * DHAT)
        hi = np.maximum(hi, np.maximum.reduceat(x1, at) + 0.5 * DHAT)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    hit = np.ones((spec.n_bodies,) * 2, bool)
    for k in range(3):
        hit &= (lo[:, None, k] <= hi[None, :, k]) & (lo[None, :, k] <= hi[:, None, k])
    return np.argwhere(np.triu(hit, 1)).astype(np.int32)


def _lists(spec, x, x1=None):
    """Body pairs and the PT / EE / VG tuples whose boxes (over both poses) overlap, in the
    framework's layouts and order."""
    ij = _body_pairs(spec, x, x1)
    plo, phi = (x, x) if x1 is None else (np.minimum(x, x1), np.maximum(x, x1))

    def prim(topo, off, b, dil):
        t = topo[off[b]:off[b + 1]] + spec.voff[b]
        return plo[t].min(1) - dil, phi[t].max(1) + dil

    def point(b):
        v = slice(spec.voff[b], spec.voff[b + 1])
        return plo[v] - DHAT, phi[v] + DHAT

    def meet(a, b):
        """index pairs (sorted) of overlapping boxes of the two sets"""
        (alo, ahi), (blo, bhi) = a, b
        ia = np.nonzero(np.all((alo <= bhi.max(0)) & (ahi >= blo.min(0)), 1))[0]
        if not len(ia):
            return np.zeros((0, 2), np.int64)
        ib = np.nonzero(np.all((blo <= ahi[ia].max(0)) & (bhi >= alo[ia].min(0)), 1))[0]
        h = np.ones((len(ia), len(ib)), bool)
        for k in range(3):
            h &= (alo[ia, None, k] <= bhi[None, ib, k]) & (blo[None, ib, k] <= ahi[ia, None, k])
        w = np.argwhere(h)
        return np.stack([ia[w[:, 0]], ib[w[:, 1]]], 1)

    pts, ees = [], []
    for n, (i, j) in enumerate(ij):
        for a, b in ((i, j), (j, i)):
            m = meet(point(a), prim(spec.tris, spec.foff, b, 0.0))
            pts.append(np.concatenate([np.tile([a, b, n], (len(m), 1)), m], 1))
        m = meet(prim(spec.edges, spec.eoff, i, 0.5 * DHAT), prim(spec.edges, spec.eoff, j, 0.5 * DHAT))
        ees.append(np.concatenate([np.tile([i, j, n], (len(m), 1)), m], 1))
    cat = lambda a: (np.concatenate(a) if a else np.zeros((0, 5))).astype(np.int32).reshape(-1, 5)  # noqa: E731
    body = np.repeat(np.arange(spec.n_bodies), np.diff(spec.voff))
    v = np.nonzero(plo[:, 1] - DHAT <= spec.ground)[0]
    vg = np.stack([body[v], v - spec.voff[body[v]]], 1).astype(np.int32)
    return ij, cat(pts), cat(ees), vg


def _structure(nb, ij):
    """(ji, row_ptr, cols, slots) of the body-pair structure of `ij`."""
    n = len(ij)
    order = np.lexsort((ij[:, 0], ij[:, 1])) if n else np.zeros(0, np.int64)
    r = np.concatenate([np.arange(nb), ij[:, 0], ij[:, 1]])
    c = np.concatenate([np.arange(nb), ij[:, 1], ij[:, 0]])
    s = np.concatenate([np.arange(nb), nb + np.arange(n), nb + n + np.arange(n)])
    o = np.lexsort((c, r))
    row_ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=nb))])
    return ij[order], row_ptr.astype(np.int32), c[o].astype(np.int32), s[o].astype(np.int32)


def _dev(a, dtype=None):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


# ------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    return {"step": _prepare_step, "rollout": _prepare_rollout, "collide": _prepare_collide,
            "assemble": _prepare_assemble, "solve": _prepare_solve}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_step(case, seed):
    from abd_hip.abd import AffineBodySimulator
    spec = _columns(case, seed, (1.0, 1.3), 0.3)
    cp = ContactParams(ground=spec.ground, psd=case["psd"], solver=case["solver"])
    sim = AffineBodySimulator(spec, cp, DEV, native=case["driver"] == "native")
    st = sim.states
    saved = [t.clone() for t in (st.A0, st.p0, st.Adot, st.pdot, sim.dq)]
    return dict(run=_run_step, sim=sim, saved=saved, frames=case["frames"])


def _run_step(s):
    sim, st = s["sim"], s["sim"].states
    for t, c in zip((st.A0, st.p0, st.Adot, st.pdot, sim.dq), s["saved"]):
        t.copy_(c)
    iters = [sim.step(f) for f in range(s["frames"])]
    return dict(A=st.A0, p=st.p0, Adot=st.Adot, pdot=st.pdot, x=sim.meshes.x_view, iters=iters)


def _prepare_rollout(case, seed):
    from abd_hip.adjoint import Rollout, rest_centroids
    spec = _drop(case, seed)
    # converged Newton and linear solves: the adjoint is exact for the minimiser of a frame
    cp = ContactParams(ground=0.0, psd=2, solver=1, solver_tol=1e-12, solver_maxiter=20000, tol=1e-8, max_iter=100)
    rng = np.random.default_rng([seed, 13])
    return dict(run=_run_rollout, rollout=Rollout(spec, cp, DEV), frames=case["frames"], v0=_dev(spec.pdot),
                c=rest_centroids(spec, DEV), target=_dev(spec.p + rng.uniform(-0.3, 0.3, spec.p.shape)))


def _run_rollout(s):
    from abd_hip.adjoint import RolloutFunction, centre_of_mass
    v0 = s["v0"].detach().requires_grad_(True)
    A, p = RolloutFunction.apply(v0, s["rollout"], s["frames"])
    loss = ((centre_of_mass(A, p, s["c"]) - s["target"]) ** 2).sum()
    loss.backward()
    return dict(A=A.detach(), p=p.detach(), loss=loss.detach(), grad=v0.grad)


def _newton_step(spec, seed):
    """A Newton step dq of a few contact distances per body ([4 nb, 3]: p, then the rows of A)."""
    rng = np.random.default_rng([seed, 14])
    dq = np.zeros((spec.n_bodies, 4, 3))
    dq[:, 0] = rng.uniform(-1.0, 1.0, (spec.n_bodies, 3)) * 3.0 * DHAT
    dq[:, 0, 1] += 4.0 * DHAT
    dq[:, 1:] = rng.uniform(-1.0, 1.0, (spec.n_bodies, 3, 3)) * DHAT
    return dq.reshape(-1, 3)


def _prepare_collide(case, seed):
    from abd_hip.abd import AffineBodySimulator
    spec = _columns(case, seed, (0.5, 1.2), 0.0)
    sim = AffineBodySimulator(spec, ContactParams(ground=spec.ground), DEV)
    # the program's own fixed-size lists, rows past a list's end -1
    nb = spec.n_bodies
    own = {k: torch.full((n, w), -1, dtype=torch.int32, device=DEV) for k, n, w in (
        ("ij", 2 * nb + 16, 2), ("ee", 200 * nb + 1000, 5), ("pt", 60 * nb + 500, 5), ("vg", 10 * nb + 300, 2))}
    return dict(run=_run_collide, sim=sim, dq=_dev(_newton_step(spec, seed)), own=own)


def _run_collide(s):
    sim, own = s["sim"], s["own"]
    sim.dq.copy_(s["dq"])
    sim.q_gets_q0()
    sim.update_mesh_vertex("xk")
    pairs, ee, pt, vg = sim.collision_set()
    for k, t in (("ij", pairs.ij), ("ee", ee), ("pt", pt), ("vg", vg)):
        own[k][:t.shape[0]].copy_(t)
        own[k][t.shape[0]:].fill_(-1)
    return dict(step=sim.ccd(sim.states, sim.dq), **own)


def _slots(nb):
    return 5 * nb + 32


def _assembly_state(case, seed):
    """Scene, positions (A near a rotation, p) and rates of an assembly: q is one Newton
    iterate, (A0, p0) the frame's start."""
    spec = _columns(case, seed, (0.5, 1.2), 0.3)
    rng = np.random.default_rng([seed, 15])
    A0 = spec.A + rng.uniform(-1e-3, 1e-3, spec.A.shape)
    p0 = spec.p - 0.01 * spec.pdot
    Adot = rng.uniform(-0.1, 0.1, spec.A.shape)
    return spec, spec.A, spec.p, A0, p0, Adot, spec.pdot


def _prepare_assemble(case, seed):
    from abd_hip.affine_body import Meshes
    from abd_hip.culling import BodyPairs
    from abd_hip.ipc import IPCContactEnergy
    from abd_hip.orthogonal_energy import InertialEnergy
    spec, A, p, A0, p0, Adot, pdot = _assembly_state(case, seed)
    x = _pose(spec, A, p)
    ij, pt, ee, vg = _lists(spec, x)
    cp = ContactParams(ground=spec.ground, psd=1)
    m = Meshes(spec, DEV)
    m.x.copy_(_dev(x))
    m.xk.copy_(m.x)
    st = m.states()
    for name, v in (("A", A), ("p", p), ("Ak", A), ("pk", p), ("A0", A0), ("p0", p0), ("Adot", Adot), ("pdot", pdot)):
        getattr(st, name).copy_(_dev(v))
    nb = spec.n_bodies
    ji, row_ptr, cols, slots = _structure(nb, ij)
    pairs = BodyPairs(_dev(ij), _dev(ji), _dev(row_ptr), _dev(cols), _dev(slots))
    m.pairs = pairs
    g = torch.zeros((4 * nb, 3), dtype=torch.float64, device=DEV)
    # slots for two pairs a body (a program sizes them once, above its pairs)
    blocks = torch.zeros((16 * _slots(nb), 3, 3), dtype=torch.float64, device=DEV)
    return dict(run=_run_assemble, m=m, st=st, ipc=IPCContactEnergy(cp), inertia=InertialEnergy(cp, m), g=g,
                blocks=blocks, pairs=pairs, pt=_dev(pt), ee=_dev(ee), vg=_dev(vg))


def _run_assemble(s):
    m, st, g, blocks = s["m"], s["st"], s["g"], s["blocks"]
    Ec = s["ipc"].energy_device([s["ee"], s["pt"], s["vg"], m])
    Ei = s["inertia"].energy_device(st)
    g.zero_()
    blocks.zero_()
    s["inertia"].gradient(g, st)
    s["inertia"].hessian(blocks, st)
    _, n = s["ipc"].gh([s["pt"], s["ee"], s["vg"], s["pairs"], m, g, blocks], return_active=True)
    return dict(Ec=Ec, Ei=Ei, g=g, blocks=blocks, active=n)


def _system(case, seed):
    """A Newton system: bodies' inertia and orthogonality stiffness on the diagonal, stiff
    rank-one contacts between neighbours of columns of about ten bodies and with the floor."""
    rng = np.random.default_rng([seed, 16])
    nb = case["bodies"]
    i = np.arange(nb - 1)
    i = i[i % 10 != 9]
    ij = np.stack([i, i + 1], 1).astype(np.int32)
    cross = np.stack([np.arange(max(0, nb - 10)), np.arange(10, max(10, nb))], 1).astype(np.int32)
    ij = np.concatenate([ij, cross[rng.random(len(cross)) < 0.3]]) if len(cross) else ij
    ij = ij[np.lexsort((ij[:, 1], ij[:, 0]))]
    n = len(ij)
    D = np.zeros((nb, 12, 12))
    O = np.zeros((n, 12, 12))
    D[:, range(3), range(3)] = 1e3
    for b in range(nb):
        M = rng.normal(size=(9, 9))
        D[b, 3:, 3:] = 1e2 * np.eye(9) + 4e4 * (np.eye(9) + 0.02 * (M @ M.T))
    for k, (a, b) in enumerate(ij):
        V = rng.normal(size=(4, 24)) * math.sqrt(10.0 ** rng.uniform(4.0, 7.0))
        V[:, 12:15] = -V[:, :3]  # a translation of both bodies feels no contact
        H = V.T @ V
        D[a] += H[:12, :12]
        D[b] += H[12:, 12:]
        O[k] = H[:12, 12:]
    B = np.concatenate([D, O, O.transpose(0, 2, 1)])
    b = rng.normal(size=12 * nb) * 1e3
    return nb, ij, B, b


def _prepare_solve(case, seed):
    from abd_hip.sparse import BsrMatrix, SolveInfo
    nb, ij, B, b = _system(case, seed)
    _, row_ptr, cols, slots = _structure(nb, ij)
    # 3x3 sub-block (ii, jj) of a slot at 16 slot + ii + 4 jj
    blocks = B.reshape(-1, 4, 3, 4, 3).transpose(0, 3, 1, 2, 4).reshape(-1, 3, 3)
    A = BsrMatrix(nb, _dev(row_ptr), _dev(cols), _dev(slots), _dev(blocks))
    x = torch.zeros((4 * nb, 3), dtype=torch.float64, device=DEV)
    return dict(run=_run_solve, A=A, b=_dev(b.reshape(-1, 3)), x=x, info=SolveInfo(x.device), method=case["method"])


def _run_solve(s):
    from abd_hip.sparse import bsr_cg, bsr_ldlt
    x = s["x"].zero_()
    if s["method"] == "ldlt":
        bsr_ldlt(s["A"], x, s["b"], info=s["info"])
    else:
        bsr_cg(s["A"], x, s["b"], tol=1e-9, info=s["info"], block_precond=s["method"] == "cg_block")
    return dict(x=x, iters=s["info"].iters)


# --------------------------------------------------------------------------------- work
_VFE = {"cube": (8, 12, 18), "ico2": (162, 320, 480), "ico3": (642, 1280, 1920), "ico4": (2562, 5120, 7680),
        "box6": (218, 432, 648)}


def work(case):
    k = case["kind"]
    if k == "rollout":  # forward: the posed vertices of every frame; backward: a system per frame
        n, f = case["bodies"], case["frames"]
        return dict(bytes=f * n * (48 * 162 + 384 + 1152 + 192), flops=f * n * (18 * 162 + 2 * 144))
    if k == "solve":
        nb = case["bodies"]
        nnzb = 3.4 * nb
        return dict(bytes=1152 * nnzb + 192 * nb, flops=2 * 144 * nnzb * (12 if case["method"] == "ldlt" else 20))
    size = [_VFE[name] for _, name in _bodies(case)]
    nb, V, F, E = len(size), sum(s[0] for s in size), sum(s[1] for s in size), sum(s[2] for s in size)
    if k == "collide":  # both poses of every vertex and the topology once, the state once
        return dict(bytes=72 * V + 12 * F + 8 * E + 192 * nb, flops=40 * V)
    if k == "assemble":  # the state, about one pair a body: gradient and three 12x12 blocks a body, contacts' terms
        return dict(bytes=nb * (288 + 96 + 3 * 1152) + 20.0 * 60 * nb, flops=nb * 20 * 3000.0)
    f = case["frames"]  # the rest shape read and the posed vertices written, the state, per frame
    return dict(bytes=f * (48 * V + 384 * nb), flops=f * 18 * V)


# -------------------------------------------------------------------------------- exact
def exact(case, seed):
    if case["kind"] == "solve":
        return _exact_solve(case, seed)
    if case["kind"] == "assemble":
        return _exact_assemble(case, seed)
    if case["kind"] == "collide":
        return _exact_collide(case, seed)
    # step, rollout: a frame ends where its own Newton loop stops (a tolerance or an
    # iteration cap, line search included), so it has no value apart from that loop's iterates
    return None


def _exact_solve(case, seed):
    nb, ij, B, b = _system(case, seed)
    H = torch.zeros((nb, nb, 12, 12), dtype=torch.float64)
    n = len(ij)
    H[range(nb), range(nb)] = torch.as_tensor(B[:nb])
    H[ij[:, 0], ij[:, 1]] = torch.as_tensor(B[nb:nb + n])
    H[ij[:, 1], ij[:, 0]] = torch.as_tensor(B[nb + n:])
    H = H.permute(0, 2, 1, 3).reshape(12 * nb, 12 * nb)
    H = H.cuda() if nb > 100 else H
    x = torch.linalg.solve(H, torch.as_tensor(b, device=H.device))
    return dict(x=x.reshape(-1, 3).cpu(), iters=None)


def _contact_vertices(spec, t, kind):
    """Scene vertex ids [n, 4] of PT (kind 0) or EE (kind 1) tuples."""
    I, J = t[:, 0], t[:, 1]
    if kind == 0:
        tri = spec.tris[spec.foff[J] + t[:, 4]] + spec.voff[J][:, None]
        return np.concatenate([(spec.voff[I] + t[:, 3])[:, None], tri], 1)
    return np.concatenate([spec.edges[spec.eoff[I] + t[:, 3]] + spec.voff[I][:, None],
                           spec.edges[spec.eoff[J] + t[:, 4]] + spec.voff[J][:, None]], 1)


def _edges3(v, kind):
    """(e0, e1, e2): the two spanning edges and the separation; beta, gamma: the closest
    point's coordinates along them."""
    if kind == 0:
        e0, e1, e2 = v[:, 1] - v[:, 2], v[:, 3] - v[:, 2], v[:, 0] - v[:, 2]
    else:
        e0, e1, e2 = v[:, 1] - v[:, 0], v[:, 3] - v[:, 2], v[:, 2] - v[:, 0]
    d = lambda a, b: (a * b).sum(-1)  # noqa: E731
    a, b, c, r, s = d(e0, e0), d(e0, e1), d(e1, e1), d(e0, e2), d(e1, e2)
    det = a * c - b * b
    inv = torch.where(det.abs() > 0, 1.0 / det, torch.zeros_like(det))
    return e0, e1, e2, (c * r - b * s) * inv, (a * s - b * r) * inv, b / a


def _inside(be, ga, kind):
    if kind == 0:
        return (be > 0) & (be < 1) & (ga > 0) & (ga < 1) & (be + ga > 0) & (be + ga < 1)
    return (be > 0) & (be < 1) & (-ga > 0) & (-ga < 1)


def _exact_assemble(case, seed):
    spec, A, p, A0, p0, Adot, pdot = _assembly_state(case, seed)
    cp = ContactParams(ground=spec.ground, psd=1)
    x = _pose(spec, A, p)
    ij, pt, ee, vg = _lists(spec, x)
    nb, nij, dt, k = spec.n_bodies, len(ij), cp.dt, cp.stiffness
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64)  # noqa: E731
    eye3 = torch.eye(3, dtype=torch.float64)
    # inertia and orthogonality: 1/2 |q - q~|_M^2 + dt^2 k |A A^T - 1|^2
    At, tA = T(A), T(A0) + dt * T(Adot)
    dp = T(p) - (T(p0) + dt * T(pdot) + dt * dt * T([0.0, cp.gravity, 0.0]))
    S = At @ At.transpose(1, 2) - eye3
    Ei = (0.5 * (1e3 * (dp ** 2).sum() + 1e2 * ((At - tA) ** 2).sum()) + dt * dt * k * (S ** 2).sum()).reshape(1)
    g = torch.zeros((nb, 4, 3), dtype=torch.float64)
    g[:, 0] = 1e3 * dp
    g[:, 1:] = 1e2 * (At - tA) + 4.0 * k * dt * dt * (S @ At)
    # slots as [slot, jj, ii, 3, 3] (block ii + 4 jj)
    B = torch.zeros((_slots(nb), 4, 4, 3, 3), dtype=torch.float64)
    for a in range(4):
        B[:nb, a, a] += (1e3 if a == 0 else 1e2) * eye3
    AtA = At.transpose(1, 2) @ At
    for a in range(3):
        for b in range(3):
            h = At[:, b, :, None] * At[:, a, None, :] + S[:, a, b, None, None] * eye3
            B[:nb, b + 1, a + 1] += 4.0 * k * dt * dt * (h + AtA if a == b else h)
    Ec = torch.zeros(1, dtype=torch.float64)
    active = 0
    d2, kap = cp.d2hat, cp.kappa
    b0 = lambda s: -kap * (s / d2 - 1.0) ** 2 * torch.log(s / d2)  # noqa: E731
    b1 = lambda s: kap * (d2 - s) * (2.0 * torch.log(s / d2) + (s - d2) / s) / d2 ** 2  # noqa: E731
    b2 = lambda s: -kap * (2.0 * torch.log(s / d2) + (s - d2) / s + (s - d2) * (2.0 / s + d2 / s ** 2)) / d2 ** 2  # noqa: E731,E501
    for kind, t in ((0, pt), (1, ee)):
        vid = _contact_vertices(spec, t, kind)
        v, r = T(x[vid]), T(spec.x0[vid])
        e0, e1, e2, be, ga, al = _edges3(v, kind)
        w = e2 - be[:, None] * e0 - ga[:, None] * e1
        s = (w * w).sum(1)
        on = _inside(be, ga, kind) & (s < d2)
        Ec = Ec + b0(s[on]).sum()
        active += int(on.sum())
        if not bool(on.any()):
            continue
        t, r, e0, e1, w, be, ga, al, s = t[on.numpy()], r[on], e0[on], e1[on], w[on], be[on], ga[on], al[on], s[on]
        n = len(s)
        u1 = e1 - al[:, None] * e0
        nn = torch.linalg.cross(e0, u1)
        l = (w * nn).sum(1) / nn.norm(dim=1)
        # d2(l^2)/dc2 in the contact coordinates c = (e0, u1, w)
        q0, q1, q2 = (e0 ** 2).sum(1), (u1 ** 2).sum(1), (w ** 2).sum(1)
        out = lambda a, b: a[:, :, None] * b[:, None, :]  # noqa: E731
        e = lambda c: c[:, None, None]  # noqa: E731
        blk = eye3 - out(e0, e0) / e(q0) - out(u1, u1) / e(q1)
        H9 = torch.zeros((n, 9, 9), dtype=torch.float64)
        H9[:, 0:3, 0:3] = -e(l / q0) * blk
        H9[:, 3:6, 3:6] = -e(l / q1) * blk
        H9[:, 0:3, 6:9] = -e(l / (q2 * q0)) * out(w, e0)
        H9[:, 3:6, 6:9] = -e(l / (q2 * q1)) * out(w, u1)
        H9[:, 6:9, 0:6] = H9[:, 0:6, 6:9].transpose(1, 2)
        gl = w * (l / q2)[:, None]
        H9 = 2.0 * e(l) * H9
        H9[:, 6:9, 6:9] += 2.0 * out(gl, gl)
        g9 = torch.zeros((n, 9), dtype=torch.float64)
        g9[:, 6:9] = 2.0 * l[:, None] * gl
        # the whole barrier Hessian in contact space, negative eigenvalues set to zero
        lam, Q = torch.linalg.eigh(e(b1(s)) * H9 + e(b2(s)) * out(g9, g9))
        H9 = (Q * lam.clamp(min=0.0)[:, None, :]) @ Q.transpose(1, 2)
        z, o = torch.zeros_like(be), torch.ones_like(be)
        if kind == 0:
            D = [[z, o, -o, z], [z, -al, al - 1.0, o], [o, -be, be + ga - 1.0, -ga]]
        else:
            D = [[-o, o, z, z], [al, -al, -o, o], [be - 1.0, -be, ga + 1.0, -ga]]
        D = torch.stack([torch.stack(row, 1) for row in D], 1)  # [n, 3, 4]
        side = torch.tensor([0, 1, 1, 1] if kind == 0 else [0, 0, 1, 1])
        r1 = torch.cat([torch.ones((n, 4, 1), dtype=torch.float64), r], 2)  # (1, rest) of each vertex
        J = torch.zeros((n, 4, 2, 4), dtype=torch.float64)  # vertex by (body, coordinate row)
        J[:, torch.arange(4), side] = r1
        C = (D @ J.reshape(n, 4, 8))  # [n, 3, 8]: contact coordinates by affine rows
        G = torch.kron(C.reshape(-1, 8), eye3).reshape(n, 9, 24)
        g24 = b1(s)[:, None] * (G.transpose(1, 2) @ g9[:, :, None])[:, :, 0]
        H24 = G.transpose(1, 2) @ H9 @ G
        I, Jb, m = (torch.as_tensor(t[:, c].astype(np.int64)) for c in (0, 1, 2))
        g.index_add_(0, I, g24[:, :12].reshape(n, 4, 3))
        g.index_add_(0, Jb, g24[:, 12:].reshape(n, 4, 3))
        sub = lambda M: M.reshape(n, 4, 3, 4, 3).permute(0, 3, 1, 2, 4)  # noqa: E731  [jj, ii]
        B.index_add_(0, I, sub(H24[:, :12, :12]))
        B.index_add_(0, Jb, sub(H24[:, 12:, 12:]))
        up = (I < Jb)
        Hij = torch.where(up[:, None, None], H24[:, :12, 12:], H24[:, 12:, :12])
        B.index_add_(0, nb + m, sub(Hij))
        B.index_add_(0, nb + nij + m, sub(Hij.transpose(1, 2)))
    d = T(x[spec.voff[vg[:, 0]] + vg[:, 1], 1] - spec.ground)
    on = d * d < d2
    d, vb = d[on], vg[on.numpy()]
    s = d * d
    Ec = Ec + b0(s).sum()
    th = torch.cat([torch.ones((len(d), 1), dtype=torch.float64), T(spec.x0[spec.voff[vb[:, 0]] + vb[:, 1]])], 1)
    b = torch.as_tensor(vb[:, 0].astype(np.int64))
    gv = torch.zeros((len(d), 4, 3), dtype=torch.float64)
    gv[:, :, 1] = th * (2.0 * d * b1(s))[:, None]
    g.index_add_(0, b, gv)
    Bv = torch.zeros((len(d), 4, 4, 3, 3), dtype=torch.float64)
    Bv[:, :, :, 1, 1] = th[:, :, None] * th[:, None, :] * (4.0 * s * b2(s))[:, None, None]
    B.index_add_(0, b, Bv)
    return dict(Ec=Ec, Ei=Ei, g=g.reshape(-1, 3), blocks=B.reshape(-1, 3, 3), active=None)


def _exact_collide(case, seed):
    """The earliest verified time at which a candidate of the step touches, times 0.9."""
    spec = _columns(case, seed, (0.5, 1.2), 0.0)
    dq = _newton_step(spec, seed).reshape(-1, 4, 3)
    x, x1 = _pose(spec, spec.A, spec.p), _pose(spec, spec.A - dq[:, 1:], spec.p - dq[:, 0])
    _, pt, ee, vg = _lists(spec, x, x1)
    y0, y1 = x[spec.voff[vg[:, 0]] + vg[:, 1], 1], x1[spec.voff[vg[:, 0]] + vg[:, 1], 1]
    low = y1 < spec.ground
    toi = min([1.0] + list((y0 - spec.ground)[low] / (y0 - y1)[low]))
    for kind, t in ((0, pt), (1, ee)):
        vid = _contact_vertices(spec, t, kind)
        a, b = torch.as_tensor(x[vid]), torch.as_tensor(x1[vid])
        # det(u, v, w)(t) with u = u0 + t u1: the cubic's coefficients
        u0, d = a[:, 1:] - a[:, :1], (b - a)[:, 1:] - (b - a)[:, :1]
        det = lambda p, q, r: (torch.linalg.cross(p, q) * r).sum(1)  # noqa: E731
        U, W = [u0[:, k] for k in range(3)], [d[:, k] for k in range(3)]
        c0, c3 = det(*U), det(*W)
        c1 = det(W[0], U[1], U[2]) + det(U[0], W[1], U[2]) + det(U[0], U[1], W[2])
        c2 = det(U[0], W[1], W[2]) + det(W[0], U[1], W[2]) + det(W[0], W[1], U[2])
        bern = torch.stack([c0, c0 + c1 / 3.0, c0 + (2.0 * c1 + c2) / 3.0, c0 + c1 + c2 + c3], 1)
        on = (bern.amin(1) <= 0.0) & (bern.amax(1) >= 0.0) & (c0 != 0)  # else no root in [0, 1]
        if not bool(on.any()):
            continue
        a, b = a[on], b[on]
        c = torch.stack([c0, c1, c2, c3], 1)[on]
        M = torch.zeros((len(c), 3, 3), dtype=torch.float64)  # companion of z^3 c0 + z^2 c1 + z c2 + c3, z = 1 / t
        M[:, 0] = -c[:, 1:] / c[:, :1]
        M[:, 1, 0] = M[:, 2, 1] = 1.0
        z = torch.linalg.eigvals(M)
        real = (z.imag.abs() <= 1e-9 * z.abs()) & (z.real >= 1.0 - 1e-12)
        root = torch.where(real, 1.0 / z.real, torch.full_like(z.real, 2.0))
        for r in root.unbind(1):
            f = lambda r: c[:, 0] + r * (c[:, 1] + r * (c[:, 2] + r * c[:, 3]))  # noqa: E731
            for _ in range(2):  # polish
                df = c[:, 1] + r * (2.0 * c[:, 2] + 3.0 * r * c[:, 3])
                r = torch.where((r <= 1.0) & (df != 0), r - f(r) / df, r)
            v = a * (1.0 - r)[:, None, None] + b * r[:, None, None]
            _, _, _, be, ga, _ = _edges3(v, kind)
            ok = (r >= 0.0) & (r < 1.0) & _inside(be, ga, kind)
            if bool(ok.any()):
                toi = min(toi, float(r[ok].min()))
    return dict(ij=None, ee=None, pt=None, vg=None, step=float(toi * 0.9 if toi < 1.0 else toi))
