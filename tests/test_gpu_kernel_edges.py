"""Kernels at the sizes where their work splits can go wrong (one item, remainders, one more
than a full grid), against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import full_ipc_config, near_contact_ee, near_contact_pt, params, rel_err, rest_of
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("psd", [2, 3])
@pytest.mark.parametrize("n", [1, 2, 65, 4099])
def test_dense_contacts_one_wave_each(psd, n):
    """The dense modes' contacts, one wave each: one contact to more than the grid's waves.
    1e-9 relative, the bound of every Hessian comparison with the oracle."""
    import abd_hip
    from abd_hip.ipc import pair_gh
    abd_hip.load()
    rng = np.random.default_rng(40 + psd)
    cp = params(psd=psd)
    prm = O.params(cp)
    for kind in (0, 1):
        X, R = [], []
        for k in range(min(n, 37)):
            d = rng.uniform(0.05, 1.2) * 1e-3
            if psd == 3:
                feats = ("face", "edge", "vertex") if kind == 0 else ("line", "pe", "pp", "parallel")
                x4 = full_ipc_config(rng, kind, feats[k % len(feats)], d)
            else:
                x4 = near_contact_pt(rng, d) if kind == 0 else near_contact_ee(rng, d)
            X.append(x4)
            R.append(rest_of(x4, rng, 0.05))
        ref = [O.pair_gh(kind, prm, x, r) for x, r in zip(X, R)]
        pick = np.arange(n) % len(X)
        act, g24, H24 = pair_gh(kind, cp, torch.as_tensor(np.array(X)[pick], device="cuda"),
                                torch.as_tensor(np.array(R)[pick], device="cuda"))
        torch.cuda.synchronize()
        act, g24, H24 = act.cpu().numpy(), g24.cpu().numpy(), H24.cpu().numpy()
        for i in range(n):
            a, s, g, Hi, Hj, Hij = ref[pick[i]]
            assert bool(act[i]) == a, i
            if not a:
                assert not g24[i].any() and not H24[i].any()
                continue
            if i >= len(X):  # a repeated contact: the same bits wherever it ran
                assert np.array_equal(g24[i], g24[pick[i]]) and np.array_equal(H24[i], H24[pick[i]])
                continue
            assert rel_err(g24[i], g) <= 1e-9
            assert rel_err(H24[i], np.block([[Hi, Hij], [Hij.T, Hj]])) <= 1e-9


@pytest.mark.parametrize("nb,seed", [(2, 0), (3, 1), (9, 2)])
def test_line_search_prunes_nothing_active(nb, seed):
    """Frames whose line searches halve and whose steps are cut short by contacts: iterations
    and energies of the native driver (which evaluates only the candidates that can be active
    at a trial) against the oracle's, which evaluates every one.  1e-7, the drivers' bound."""
    from abd_hip import scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    rng = np.random.default_rng(seed)
    lib = [scenes.cube_mesh(), scenes.icosphere_mesh(1, 0.5), scenes.subdivided_box_mesh(2)]
    meshes = [lib[k % 3] for k in range(nb)]
    # columns of three with gaps of 1 to 1.3 dhat, thrown at each other
    p, y = np.zeros((nb, 3)), {}
    for b, (V, F) in enumerate(meshes):
        c = b // 3
        base = y.get(c, 0.0) + rng.uniform(1.0, 1.3) * 1e-3
        p[b] = (1.5 * c + rng.uniform(-0.01, 0.01), base - V[:, 1].min(), rng.uniform(-0.01, 0.01))
        y[c] = base + np.ptp(V[:, 1])
    pdot = rng.uniform(-0.3, 0.3, (nb, 3))
    spec = scenes.build_scene(meshes, np.stack([np.eye(3)] * nb), p, np.zeros((nb, 3, 3)), pdot, ground=0.0)
    cp = ContactParams(ground=0.0, psd=1, solver=3)
    sim = AffineBodySimulator(spec, cp, native=True)
    ref = O.OracleSim(spec, cp)
    for f in range(3):
        n = sim.step(f)
        before = int(ref.stats[0])
        ref.step()
        assert n == int(ref.stats[0]) - before
    torch.cuda.synchronize()
    assert np.abs(sim.states.A.cpu().numpy() - ref.A).max() <= 1e-7
    assert np.abs(sim.states.p.cpu().numpy() - ref.p).max() <= 1e-7
    assert sim.stats["energy_evals"] > sim.stats["newton_iters"] + 3  # some search halved


@pytest.mark.parametrize("mesh", ["cube", "ico2", "ico3"])
def test_body_passes_by_mesh_size(mesh):
    """The per-body passes with one wave a body (8 and 162 vertices) and with four (642):
    the vertices placed by a frame, and a frame after the rest shape was changed in place,
    against the oracle (1e-7, the drivers' bound)."""
    from abd_hip import scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    m = {"cube": scenes.cube_mesh, "ico2": lambda: scenes.icosphere_mesh(2, 0.5),
         "ico3": lambda: scenes.icosphere_mesh(3, 0.5)}[mesh]()
    h = m[0][:, 1].max() - m[0][:, 1].min()
    p = np.array([[0.0, 5e-4 - m[0][:, 1].min() + k * (h + 1.1e-3), 0.01 * k] for k in range(3)])
    spec = scenes.build_scene([m] * 3, np.stack([np.eye(3)] * 3), p, np.zeros((3, 3, 3)), np.zeros((3, 3)), ground=0.0)
    cp = ContactParams(ground=0.0, psd=1, solver=3)
    sim = AffineBodySimulator(spec, cp, native=True)
    for scale in (1.0, 0.999):
        if scale != 1.0:  # another rest shape in the same buffers, the state kept
            sim.meshes.x0.mul_(scale)
        st = sim.states
        sp = scenes.build_scene([(m[0] * scale, m[1])] * 3, *(t.cpu().numpy() for t in (st.A0, st.p0, st.Adot, st.pdot)),
                                ground=0.0)
        ref = O.OracleSim(sp, cp)
        ref.dq[...] = sim.dq.cpu().numpy()
        sim.step()
        ref.step()
        torch.cuda.synchronize()
        A, q = st.A0.cpu().numpy(), st.p0.cpu().numpy()
        assert np.abs(A - ref.A).max() <= 1e-7 and np.abs(q - ref.p).max() <= 1e-7
        body = np.repeat(np.arange(3), np.diff(sp.voff))
        x = np.einsum("vr,vrk->vk", sp.x0, A[body]) + q[body]
        assert np.abs(sim.meshes.x_view.cpu().numpy() - x).max() <= 1e-13


@pytest.mark.parametrize("sizes", [(1, 1, 1, 1), (256, 257, 255, 0), (2049, 16385, 16384, 513),
                                   (65536, 2048, 1, 2047), (65793, 40003, 30001, 3001)])
@pytest.mark.parametrize("with_ji", [True, False])
def test_keep_filter_block_edges(sizes, with_ji):
    """The superset filter (abd_cull_keep) at the edges of its blocks (256 entries), of its
    super-blocks (64 blocks) and of the pair blocks it sums in LDS (65536 pairs): the kept
    entries in their order with the kept pairs' indices, exactly."""
    from abd_hip import _lib, scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    nij, npt, nee, nvg = sizes
    rng = np.random.default_rng(nij)
    nb = 400
    spec = scenes.build_scene([scenes.cube_mesh()] * nb, np.stack([np.eye(3)] * nb), np.zeros((nb, 3)),
                              np.zeros((nb, 3, 3)), np.zeros((nb, 3)), ground=0.0)
    m = AffineBodySimulator(spec, ContactParams(ground=0.0), native=False).meshes

    def boxes(n):
        lo = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
        return lo, lo + rng.uniform(0, 2, (n, 3)).astype(np.float32)

    def hit(a, i, b, j):
        return ((a[0][i] <= b[1][j]) & (a[1][i] >= b[0][j])).all(1)

    body, pnt, edg, tri = boxes(nb), boxes(8 * nb), boxes(18 * nb), boxes(12 * nb)
    I, J = np.triu_indices(nb, 1)
    sel = np.sort(rng.choice(len(I), nij, replace=False))
    ij = np.stack([I[sel], J[sel]], 1).astype(np.int32)
    ji = ij[:, ::-1].copy()
    keep_ij = hit(body, ij[:, 0], body, ij[:, 1])
    new = np.cumsum(keep_ij) - 1

    def tuples(n, na, nbm, first, A, B):
        q = np.sort(rng.integers(0, nij, n))
        t = np.stack([ij[q, 0], ij[q, 1], q, rng.integers(0, na, n), rng.integers(0, nbm, n)], 1).astype(np.int32)
        k = keep_ij[q] & hit(A, na * t[:, 0] + t[:, 3], B, nbm * t[:, 1] + t[:, 4])
        out = t[k].copy()
        out[:, 2] = new[out[:, 2]]
        return t, out

    pt, pt_ref = tuples(npt, 8, 12, 0, pnt, tri)
    ee, ee_ref = tuples(nee, 18, 18, 0, edg, edg)
    vg = np.stack([np.sort(rng.integers(0, nb, nvg)), rng.integers(0, 8, nvg)], 1).astype(np.int32)
    dhat, ground = 0.01, 0.1
    v = 8 * vg[:, 0] + vg[:, 1]
    q = (np.float32([-1e3, -1e3, -1e3]), np.array([1e3, ground, 1e3], np.float32))
    keep_vg = (body[0][vg[:, 0], 1].astype(np.float64) < 0.5 * dhat + ground) & (
        (pnt[0][v] <= q[1]) & (pnt[1][v] >= q[0])).all(1)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ins = [d(x) for x in (ij, ji, pt, ee, vg)]
    bx = [d(x) for b in (body, pnt, edg, tri) for x in b]
    outs = [torch.full_like(x, -7) for x in ins]
    P = _lib.ptr
    cnt = (ctypes.c_int64 * 5)()
    _lib.call("abd_cull_keep", _lib.stream_handle(), m.c, P(ins[0]), P(ins[1]) if with_ji else None, nij, P(ins[2]),
              npt, P(ins[3]), nee, P(ins[4]), nvg, *[P(b) for b in bx], dhat, ground, P(outs[0]),
              P(outs[1]) if with_ji else None, P(outs[2]), P(outs[3]), P(outs[4]), cnt)
    refs = [ij[keep_ij], ji[keep_ij] if with_ji else ji[:0], pt_ref, ee_ref, vg[keep_vg]]
    assert list(cnt) == [len(r) for r in refs]
    for o, r in zip(outs, refs):
        o = o.cpu().numpy()
        assert np.array_equal(o[:len(r)], r) and (o[len(r):] == -7).all()


@pytest.mark.parametrize("method", [0, 1])
def test_krylov_in_registers_edges(method):
    """BiCGSTAB and Jacobi CG where the workgroup's size and the rows kept in registers change
    (n = 12 bodies <= 64, 256, 1024 threads; 12, 6 or 4 threads a block): a batch of the sizes
    gives each system the bits of its solve alone, and the dense solution.  The residual is
    below 1e-10 of b and the matrices' condition below 2: 1e-9."""
    import abd_hip
    from abd_hip import _lib
    from abd_hip.sparse import BsrMatrix, SolveInfo, bicgstab, bsr_cg
    abd_hip.load()
    rng = np.random.default_rng(5)
    sizes = [(1, 0), (4, 6), (5, 3), (8, 28), (9, 0), (21, 32), (22, 32), (42, 64), (43, 64), (64, 96), (65, 96),
             (85, 20), (86, 20)]
    boff = np.concatenate([[0], np.cumsum([m for m, _ in sizes])]).astype(np.int32)
    nb = int(boff[-1])
    pairs = []
    for (m, k), r0 in zip(sizes, boff):
        a, b = np.triu_indices(m, 1)
        sel = rng.choice(len(a), k, replace=False) if k else []
        pairs += [(int(a[q] + r0), int(b[q] + r0)) for q in sel]
    ij = np.array(sorted(pairs), np.int32)
    nij = len(ij)
    blocks = np.zeros(((nb + 2 * nij), 16, 3, 3))
    dense = np.zeros((12 * nb, 12 * nb))

    def put(slot, i, j, M):
        blocks[slot] = M.reshape(4, 3, 4, 3).transpose(2, 0, 1, 3).reshape(16, 3, 3)
        dense[12 * i:12 * i + 12, 12 * j:12 * j + 12] = M

    for k, (i, j) in enumerate(ij):
        M = 0.3 * rng.normal(size=(12, 12))
        put(nb + k, i, j, M)
        put(nb + nij + k, j, i, M.T)
    for i in range(nb):
        Q = rng.normal(size=(12, 12))
        put(i, i, i, Q @ Q.T + 600.0 * np.eye(12))
    rhs, x0 = rng.normal(size=(12 * nb)), 0.01 * rng.normal(size=(12 * nb))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()

    def structure(n, p):
        q = p[np.lexsort((p[:, 0], p[:, 1]))]
        out = [torch.empty(s, dtype=torch.int32, device="cuda") for s in (n + 1, n + 2 * len(p), n + 2 * len(p))]
        tp, tq = d(p.astype(np.int32)), d(q.astype(np.int32))
        _lib.call("abd_bsr_structure", _lib.stream_handle(), n, _lib.ptr(tp), _lib.ptr(tq), len(p),
                  *[_lib.ptr(o) for o in out])
        torch.cuda.synchronize()
        return out

    rp, cl, sl = structure(nb, ij)
    tboff, tbs = d(boff), d(np.repeat(np.arange(len(sizes)), [m for m, _ in sizes]).astype(np.int32))
    sc = _lib.AbdScene()
    sc.n_bodies, sc.n_scenes = nb, len(sizes)
    sc.scene_boff, sc.body_scene = tboff.data_ptr(), tbs.data_ptr()
    tb, tr, x = d(blocks), d(rhs), d(x0)
    active = torch.ones(len(sizes), dtype=torch.uint8, device="cuda")
    iters = torch.zeros(len(sizes), dtype=torch.int32, device="cuda")
    resid = torch.zeros(len(sizes), dtype=torch.float64, device="cuda")
    tol = 1e-11 if method == 0 else 1e-12
    _lib.call("abd_bsr_solve_scenes", _lib.stream_handle(), method, ctypes.byref(sc), 86, _lib.ptr(rp), _lib.ptr(cl),
              _lib.ptr(sl), _lib.ptr(tb), _lib.ptr(tr), _lib.ptr(x), tol, 500, 10, _lib.ptr(active),
              _lib.ptr(iters), _lib.ptr(resid))
    xb = x.cpu().numpy()
    assert rel_err(xb, np.linalg.solve(dense, rhs)) <= 1e-9
    for s, (m, k) in enumerate(sizes):
        r0, r1 = boff[s], boff[s + 1]
        q = np.nonzero((ij[:, 0] >= r0) & (ij[:, 0] < r1))[0]
        slots = np.concatenate([np.arange(r0, r1), nb + q, nb + nij + q])
        A = BsrMatrix(m, *structure(m, ij[q] - r0), d(blocks[slots].reshape(-1, 3, 3)))
        xs, info = d(x0[12 * r0:12 * r1].reshape(-1, 3)), SolveInfo("cuda")
        bs = d(rhs[12 * r0:12 * r1].reshape(-1, 3))
        if method == 0:
            bicgstab(A, bs, xs, tol, 500, 10, info)
        else:
            bsr_cg(A, xs, bs, 500, tol, 10, info)
        assert np.array_equal(xs.cpu().numpy().ravel(), xb[12 * r0:12 * r1]), (m, k)
        assert int(info.iters[0]) == int(iters[s]) and float(info.resid[0]) == float(resid[s])


def _ldlt_pairs(kind, m):
    if kind == "dense":
        return [(i, j) for i in range(m) for j in range(i + 1, m)]
    if kind == "star":  # the last body coupled to all: the others are one level
        return [(i, m - 1) for i in range(m - 1)]
    if kind == "pairs":
        return [(2 * i, 2 * i + 1) for i in range(m // 2)]
    return [(i, i + w) for i in range(m) for w in (1, 9, 10) if i + w < m]  # "band"


@pytest.mark.parametrize("kind,m", [("dense", 3), ("dense", 13), ("dense", 14), ("dense", 15), ("dense", 51),
                                    ("dense", 52), ("dense", 64), ("star", 43), ("star", 44), ("star", 64),
                                    ("pairs", 63), ("band", 64)])
def test_ldlt_chunk_edges(kind, m):
    """The direct solve where its storage changes (the factor in LDS, in memory with staged
    chunks, in memory unstaged) and where a level takes several chunks (1024 columns): against
    the oracle's same sums, 1e-14 (the bound of the batched comparison)."""
    import abd_hip
    from abd_hip.sparse import BsrMatrix, SolveInfo, bsr_ldlt
    from test_gpu_ldlt import _structure, _system
    lib = abd_hip.load()
    rng = np.random.default_rng(m)
    ij = np.array(sorted(_ldlt_pairs(kind, m)), np.int32).reshape(-1, 2)
    blocks, dense = _system(m, ij, rng)
    b = rng.normal(size=(4 * m, 3))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = BsrMatrix(m, *_structure(lib, m, ij), d(blocks))
    x, info = d(np.zeros((4 * m, 3))), SolveInfo("cuda")
    bsr_ldlt(A, x, d(b), info=info)
    ref, st = O.bsr_ldlt(m, ij, blocks, b, np.zeros((4 * m, 3)))
    assert st == 1 and int(info.iters[0]) == 1
    assert rel_err(x.cpu().numpy(), ref) <= 1e-14
    assert rel_err(x.cpu().numpy().ravel(), np.linalg.solve(dense, b.ravel())) <= 1e-10


@pytest.mark.parametrize("psd,total", [(1, 255), (1, 256), (1, 257), (1, 16385), (1, 40000), (3, 600)])
def test_gh_over_repeated_candidates(psd, total):
    """The contact gradient and Hessian over lists in which every candidate is repeated until
    they pass the edges of the active-candidate blocks (256), super-blocks (16384) and the
    chunks of a pair's sums (64): n times the sums of the list itself.  Sums of n equal terms:
    relative error below 2 n 2^-53 plus the bound of the sums, 1e-10 for the sizes here."""
    import abd_hip
    from abd_hip.ipc import IPCContactEnergy
    from test_gpu_parity import T, _gpu_scene, _stage_lists, contact_scene
    abd_hip.load()
    spec = contact_scene()
    cp = params(ground=spec.ground, psd=psd)
    m = _gpu_scene(spec)
    sc = O.OracleScene(spec)
    x = O.project(sc, spec.A, spec.p)
    m.x.copy_(T(x))
    m.xk.copy_(T(x))
    G = _stage_lists(m, cp)
    nij, nb = len(G["pairs"].ij), spec.n_bodies
    ipc = IPCContactEnergy(cp)
    vg = G["vg"][:0]

    def gh(pt, ee):
        g = torch.zeros((4 * nb, 3), dtype=torch.float64, device="cuda")
        blocks = torch.zeros(((nb + 2 * nij) * 16, 3, 3), dtype=torch.float64, device="cuda")
        hl, n = ipc.gh([pt.contiguous(), ee.contiguous(), vg, nij, m, g, blocks], return_active=True)
        return g.cpu().numpy(), blocks.cpu().numpy(), hl.cpu().numpy(), n

    # only the active candidates (found one at a time from their count), then n of each
    pt, ee = G["pt"], G["ee"]
    pt = pt[[k for k in range(len(pt)) if gh(pt[k:k + 1], ee[:0])[3]]]
    ee = ee[[k for k in range(len(ee)) if gh(pt[:0], ee[k:k + 1])[3]]]
    assert len(pt) + len(ee) > 2
    g1, b1, h1, n1 = gh(pt, ee)
    assert n1 == len(pt) + len(ee)
    k = -(-total // n1)
    gk, bk, hk, nk = gh(pt.repeat_interleave(k, 0), ee.repeat_interleave(k, 0))
    assert nk == k * n1 and np.array_equal(h1, hk)
    assert rel_err(gk, k * g1) <= 1e-10 and rel_err(bk, k * b1) <= 1e-10


def test_recording_leaves_other_threads_alone():
    """A driver records its iteration for replay while another thread synchronizes the device
    and allocates: neither is refused (a captured stream would make the runtime refuse both)."""
    import threading
    from abd_hip import scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    m = scenes.cube_mesh()
    specs = []
    for k in range(6):
        p = np.array([[0.0, 0.5005 + j * 1.001, 0.002 * j] for j in range(2 + k)])
        n = len(p)
        specs.append(scenes.build_scene([m] * n, np.stack([np.eye(3)] * n), p, np.zeros((n, 3, 3)),
                                        np.zeros((n, 3)), ground=0.0))
    done, errors, rounds = threading.Event(), [], [0]

    def other():
        try:
            while not done.is_set():
                torch.cuda.synchronize()
                t = torch.empty(1 << (12 + rounds[0] % 12), device="cuda")
                del t
                torch.cuda.empty_cache()
                rounds[0] += 1
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    th = threading.Thread(target=other)
    th.start()
    try:
        with torch.cuda.stream(torch.cuda.Stream()):
            for spec in specs:
                sim = AffineBodySimulator(spec, ContactParams(ground=0.0, psd=1, solver=3), native=True)
                for f in range(4):
                    sim.step(f)
    finally:
        done.set()
        th.join()
    assert not errors and rounds[0] > 0


@pytest.mark.parametrize("nb", [2, 3, 6])
@pytest.mark.parametrize("mesh", ["cube", "ico3"])
def test_culling_pass_edges(nb, mesh):
    """The collision set of overlapping bodies below one pass of the primitive filter (a cube's
    8, 18 and 12) and above it (642 points, 1920 edges, 1280 triangles; 1024 a pass), with
    fewer and more tasks than XCDs: the oracle's lists, exactly."""
    import abd_hip
    from abd_hip import scenes
    from test_gpu_parity import T, _gpu_scene, _stage_lists, oracle_lists
    abd_hip.load()
    m = scenes.cube_mesh() if mesh == "cube" else scenes.icosphere_mesh(3, 0.5)
    h = m[0][:, 1].max() - m[0][:, 1].min()
    rng = np.random.default_rng(nb)
    p = np.array([[0.02 * k, 0.45 * h + 0.97 * h * k, 0.01 * k] for k in range(nb)])
    A = np.stack([np.linalg.qr(np.eye(3) + 0.05 * rng.normal(size=(3, 3)))[0] for _ in range(nb)])
    spec = scenes.build_scene([m] * nb, A, p, np.zeros((nb, 3, 3)), np.zeros((nb, 3)), ground=0.0)
    cp = params(ground=0.0)
    g = _gpu_scene(spec)
    sc = O.OracleScene(spec)
    x = O.project(sc, spec.A, spec.p)
    g.x.copy_(T(x))
    g.xk.copy_(T(x))
    G = _stage_lists(g, cp)
    R = oracle_lists(sc, x, cp.dhat, cp.ground)
    assert len(R["ij"]) == nb - 1 and len(R["ee"]) and len(R["vg"])
    assert np.array_equal(G["pairs"].ij.cpu().numpy(), R["ij"])
    for k in ("pt", "ee", "vg"):
        assert np.array_equal(G[k].cpu().numpy(), R[k]), k


@pytest.mark.parametrize("block", [False, True])
@pytest.mark.parametrize("maxiter,check", [(1, 10), (7, 10), (10, 10), (11, 5), (40, 4)])
def test_large_cg_batches(block, maxiter, check):
    """CG over several workgroups (171 bodies) cut off and checked at the ends of its batches:
    the oracle's iterate and count.  Both run the same recurrence in double; after at most 40
    iterations of a system of condition below 3 they agree to 1e-9."""
    import abd_hip
    from abd_hip.sparse import BsrMatrix, SolveInfo, bsr_cg
    from test_gpu_ldlt import _structure, _system
    lib = abd_hip.load()
    m = 171
    rng = np.random.default_rng(8)
    ij = np.array(sorted({tuple(sorted(rng.choice(m, 2, replace=False).tolist())) for _ in range(200)}), np.int32)
    blocks, _ = _system(m, ij, rng)
    b = rng.normal(size=(4 * m, 3))
    x0 = 0.01 * rng.normal(size=(4 * m, 3))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = BsrMatrix(m, *_structure(lib, m, ij), d(blocks))
    x, info = d(x0), SolveInfo("cuda")
    tol = 1e-6
    bsr_cg(A, x, d(b), maxiter, tol, check, info, block_precond=block)
    ref, it, _ = (O.bsr_cg_block if block else O.bsr_cg)(m, ij, blocks, b, x0, tol, maxiter, check)
    assert int(info.iters[0]) == it
    assert rel_err(x.cpu().numpy(), ref) <= 1e-9
