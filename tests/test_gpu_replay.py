"""Newton iterations replayed from a recorded graph against the same iterations launched
kernel by kernel, for one scene and where the candidate superset changes between them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_replay_between_supersets():
    """A graph recorded for a superset of few edge pairs (below two a vertex) replayed after an
    iteration with many (above), in a step that leaves its ranges and is filtered anew: the
    swept set of that step (its size is in the statistics) and the states of the launches.

    Body 0 is a cube turned by 45 degrees.  A frame that carries it past body 1 sweeps many
    pairs.  In the next, stretched in its plane, it starts inside those ranges and leaves them
    at once along z; Newton then takes the stretch back from above, so that its second step
    leaves the second superset's ranges too.  In its first step the top edges pass the height
    of body 1's, in the second they lie above it."""
    from abd_hip import scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    c = np.sqrt(0.5)
    R = np.array([[c, -c, 0.0], [c, c, 0.0], [0.0, 0.0, 1.0]])
    nb, reach, corner, stretch = 5, 1.1, 0.75, np.diag([1.5, 1.5, 1.0])
    A = np.stack([R.T] + [np.eye(3)] * (nb - 1))
    p = np.zeros((nb, 3))
    p[1] = (-corner - 0.5, corner + 0.5, 0.15)
    p[2:, 2] = 20.0 * np.arange(1, nb - 1)  # far away: vertices without pairs
    spec = scenes.build_scene([scenes.cube_mesh()] * nb, A, p, np.zeros((nb, 3, 3)), np.zeros((nb, 3)), ground=-100.0)
    cp = ContactParams(ground=-100.0, psd=1, solver=3)
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731

    def run(graphs):
        sim = AffineBodySimulator(spec, cp, native=True)
        sim.set_graphs(graphs)
        st, out = sim.states, []
        for k in range(5):
            q = p + np.array([64.0 * k, 0.0, 0.0])
            mid = q[0].copy()
            q[0, :2] -= reach
            v = np.zeros((nb, 3))
            v[0, :2] = 2.0 * reach / cp.dt
            st.A0.copy_(T(A))
            st.p0.copy_(T(q))
            st.Adot.zero_()
            st.pdot.copy_(T(v))
            its = [sim.step()]
            st.A0[0].copy_(T((R @ stretch).T))
            st.p0[0].copy_(T(mid))
            st.Adot.zero_()
            st.pdot.zero_()
            st.pdot[0, 2] = 0.2 / cp.dt
            its.append(sim.step())
            out.append((its, dict(sim.stats), st.A0.clone(), st.p0.clone()))
        return out, sim.graph_counts()

    # (one after the other: buffers that grow anywhere in the process outdate recorded graphs)
    got, gc = run(True)
    ref, _ = run(False)
    assert gc["recorded"] >= 1 and gc["replayed"] >= 2, gc
    assert got[0][0][0] == 2  # the first frame of a pass ends before its superset is recorded
    for k, (a, b) in enumerate(zip(got, ref)):
        assert a[0] == b[0] and a[1] == b[1], (k, a[:2], b[:2])
        assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), k


@pytest.mark.parametrize("solver,psd", [(3, 1), (0, 0)])
def test_one_scene_replay_equals_launches(solver, psd):
    """One scene's iterations recorded and replayed while another thread synchronizes the device
    and allocates: taken, and the states, iterations and statistics of the same iterations
    launched kernel by kernel."""
    import threading
    from abd_hip import scenes
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    m = scenes.cube_mesh()
    n = 5
    p = np.array([[0.0, 0.5005 + k * 1.001, 0.002 * k] for k in range(n)])
    spec = scenes.build_scene([m] * n, np.stack([np.eye(3)] * n), p, np.zeros((n, 3, 3)), np.zeros((n, 3)),
                              ground=0.0)
    cp = ContactParams(ground=0.0, psd=psd, solver=solver)

    def run(graphs):
        sim, out = AffineBodySimulator(spec, cp, native=True), []
        sim.set_graphs(graphs)
        for f in range(6):
            it = sim.step(f)
            out.append((it, dict(sim.stats), sim.states.A0.clone(), sim.states.p0.clone()))
        return out, sim.graph_counts()

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
            got, gc = run(True)
    finally:
        done.set()
        th.join()
    assert not errors and rounds[0] > 0
    assert gc["recorded"] >= 1 and gc["replayed"] >= 5, gc
    ref, none = run(False)
    assert none["recorded"] == none["replayed"] == 0
    for f, (a, b) in enumerate(zip(got, ref)):
        assert a[0] == b[0] and a[1] == b[1], f
        assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), f
