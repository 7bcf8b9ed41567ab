"""A body with many neighbours (a plate under many cubes): the work of a long matrix row at the
edges of its splits, against the oracle."""
import numpy as np
import pytest
import torch

from helpers import oracle_lists, params, rel_err
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _plate(n, last):
    """A plate and n cubes on it, the plate the first or the last body: two thirds stand on it at
    0.2 to 0.9 of dhat, every third hangs beyond its rim, a pair without active contacts."""
    from abd_hip import scenes
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n)))
    V, F = scenes.cube_mesh()
    plate = (V * np.array([side + 1.0, 0.5, side + 1.0]), F)
    meshes, p, A = [plate], [[0.5 * side, 0.251, 0.5 * side]], [np.eye(3)]
    for k in range(n):
        if k % 3 == 2:
            h = min(0.05, 0.8 * (side + 0.5) / (n // 3))  # (they must not meet each other)
            meshes.append((h * V, F))
            p.append([side + 0.5008 + 0.5 * h, 0.5018 + 0.5 * h, 1.25 * h * (k // 3)])
            A.append(np.eye(3))
            continue
        a = rng.uniform(-0.3, 0.3)
        meshes.append((0.5 * V, F))
        p.append([k % side + 0.5, 0.501 + rng.uniform(0.2, 0.9) * 1e-3 + 0.25, k // side + 0.5])
        A.append([[np.cos(a), 0.0, np.sin(a)], [0.0, 1.0, 0.0], [-np.sin(a), 0.0, np.cos(a)]])
    order = list(range(1, n + 1)) + [0] if last else list(range(n + 1))
    z = np.zeros((n + 1, 3))
    return scenes.build_scene([meshes[k] for k in order], np.array(A)[order], np.array(p)[order],
                              np.zeros((n + 1, 3, 3)), z, ground=0.0)


@pytest.mark.parametrize("n,last", [(n, last) for n in (1, 63, 64, 72, 255, 256, 300) for last in (False, True)] +
                         [(4200, False)])
def test_gh_of_a_plate_under_cubes(n, last):
    """Gradient and Hessian on both sides of the bodies from which rows can be long (64), with
    a row's entries one more than those listed at once (256), its active pairs a multiple of
    those summed at once (72 has 48 of them, 8 at once) and not, and more pairs than workgroups
    for their off-diagonal blocks (4096).  1e-9 relative, the bound of
    every Hessian comparison with the oracle."""
    import abd_hip
    from abd_hip.ipc import IPCContactEnergy
    from test_gpu_parity import T, _gpu_scene, _stage_lists
    abd_hip.load()
    spec = _plate(n, last)
    cp = params(ground=0.0, psd=1)
    m = _gpu_scene(spec)
    sc = O.OracleScene(spec)
    x = O.project(sc, spec.A, spec.p)
    m.x.copy_(T(x))
    m.xk.copy_(T(x))
    G = _stage_lists(m, cp)
    R = oracle_lists(sc, x, cp.dhat, cp.ground)
    nij, nb = len(R["ij"]), n + 1
    assert nij == n
    rng = np.random.default_rng(1)
    g0, b0 = rng.normal(size=(4 * nb, 3)), rng.normal(size=((nb + 2 * nij) * 16, 3, 3))
    g, blocks = T(g0), T(b0)
    _, nact = IPCContactEnergy(cp).gh([G["pt"], G["ee"], G["vg"], G["pairs"], m, g, blocks], return_active=True)
    g_ref, b_ref, _ = O.contact_gh(sc, O.params(cp), x, R["pt"], R["ee"], R["vg"], nij, g0, b0)
    b = blocks.cpu().numpy().reshape(b_ref.shape)
    idle = [k for k, (i, j) in enumerate(R["ij"]) if (j if not last else i) % 3 == (0 if not last else 2)]
    assert nact >= 4 * (n - n // 3) and len(idle) == n // 3
    for k in idle:  # pairs without active contacts: their blocks are left alone
        for s in (nb + k, nb + nij + k):
            assert np.array_equal(b.reshape(-1, 16, 9)[s], b0.reshape(-1, 16, 9)[s])
    assert rel_err(g.cpu().numpy() - g0, g_ref - g0) <= 1e-9
    assert rel_err(b - b0.reshape(b.shape), b_ref - b0.reshape(b.shape)) <= 1e-9


def _cg_system(kind, m, rng):
    """Blocks of a system of m bodies: 50 on the diagonal, coupling blocks of normal entries times
    0.1, whose norm is below 10 for the kinds here (condition below 1.5)."""
    if kind == "dense":
        ij = np.stack(np.triu_indices(m, 1), 1)
    elif kind == "first":  # body 0 coupled to all
        ij = np.stack([np.zeros(m - 1, int), np.arange(1, m)], 1)
    elif kind == "last":
        ij = np.stack([np.arange(m - 1), np.full(m - 1, m - 1)], 1)
    else:  # "sparse": rows of 1 to about 10 entries
        ij = rng.integers(0, m, (2 * m, 2))
        ij = np.unique(np.sort(ij[ij[:, 0] != ij[:, 1]], axis=1), axis=0)
    n = len(ij)
    B = np.zeros((m + 2 * n, 12, 12))
    Q = rng.normal(size=(m, 12, 12))
    B[:m] = 50.0 * np.eye(12) + 0.02 * (Q + Q.transpose(0, 2, 1))
    B[m:m + n] = 0.1 * rng.normal(size=(n, 12, 12))
    B[m + n:] = B[m:m + n].transpose(0, 2, 1)
    blocks = B.reshape(-1, 4, 3, 4, 3).transpose(0, 3, 1, 2, 4).reshape(-1, 3, 3)
    return ij.astype(np.int32), np.ascontiguousarray(blocks)


@pytest.mark.parametrize("block", [False, True])
@pytest.mark.parametrize("kind,m", [("dense", 171), ("first", 172), ("last", 400), ("sparse", 513),
                                    ("sparse", 3100)])
def test_large_cg_long_rows(kind, m, block):
    """CG over several workgroups with rows of one entry to hundreds, up to more workgroups (194)
    than one has threads for their partial sums in the block form (192): stopped by its test and
    cut off, the oracle's iterate, count and residual.  Both run the same recurrence in double;
    after at most 40 iterations of a system of condition below 1.5 they agree to 1e-9.  The
    residual r.z is off by 2 |r0| / |r| roundings an iteration, below 1e-9 at the sizes of r
    here (the smallest is 1e-6 of r0): 1e-8."""
    import abd_hip
    from abd_hip.sparse import BsrMatrix, SolveInfo, bsr_cg
    from test_gpu_ldlt import _structure
    lib = abd_hip.load()
    rng = np.random.default_rng(m)
    ij, blocks = _cg_system(kind, m, rng)
    b, x0 = rng.normal(size=(4 * m, 3)), 0.01 * rng.normal(size=(4 * m, 3))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    A = BsrMatrix(m, *_structure(lib, m, ij), d(blocks))
    for tol, maxiter, check in ((1e-5, 40, 3), (0.0, 2, 4)):
        x, info = d(x0), SolveInfo("cuda")
        bsr_cg(A, x, d(b), maxiter, tol, check, info, block_precond=block)
        ref, it, err = (O.bsr_cg_block if block else O.bsr_cg)(m, ij, blocks, b, x0, tol, maxiter, check)
        assert int(info.iters[0]) == it and (it < 40)
        assert rel_err(x.cpu().numpy(), ref) <= 1e-9
        assert abs(float(info.resid[0]) - err) <= 1e-8 * abs(err)


@pytest.mark.parametrize("m", [3, 4, 5, 20, 33])
def test_ldlt_of_a_body_coupled_to_all(m):
    """The direct solve where one block is updated by all other bodies at once: by two (one
    thread takes a tile), three (a row each) and many.  The oracle's same sums, 1e-14 (the bound
    of the other comparisons of this solve)."""
    import abd_hip
    from abd_hip.sparse import BsrMatrix, SolveInfo, bsr_ldlt
    from test_gpu_ldlt import _structure, _system
    lib = abd_hip.load()
    rng = np.random.default_rng(m)
    ij = np.stack([np.arange(m - 1), np.full(m - 1, m - 1)], 1).astype(np.int32)
    blocks, dense = _system(m, ij, rng)
    b = rng.normal(size=(4 * m, 3))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    A = BsrMatrix(m, *_structure(lib, m, ij), d(blocks))
    x, info = d(np.zeros((4 * m, 3))), SolveInfo("cuda")
    bsr_ldlt(A, x, d(b), info=info)
    ref, st = O.bsr_ldlt(m, ij, blocks, b, np.zeros((4 * m, 3)))
    assert st == 1 and int(info.iters[0]) == 1
    assert rel_err(x.cpu().numpy(), ref) <= 1e-14
    assert rel_err(x.cpu().numpy().ravel(), np.linalg.solve(dense, b.ravel())) <= 1e-10
