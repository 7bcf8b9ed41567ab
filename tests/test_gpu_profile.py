"""The byte counts that a rate is quoted on."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu]

import helpers


def test_line_search_bytes_count_a_candidate_once_a_launch():
    """A cube half a d-hat above the ground on a planted step 0.3 d-hat down, against the
    barrier, which no halving makes acceptable: its four bottom vertices are near at all of
    the 11 lengths (1 to 2^-10), evaluated in two launches, one and ten.  A launch reads a candidate's tuple, index and rest vertex (32 bytes) and its
    apart_until (4) once, however many trials it evaluates, and one body state (96 bytes) a
    trial; the frame-start energy reads the four candidates (32 bytes)."""
    from abd_hip import _lib
    from abd_hip.abd import AffineBodySimulator
    from abd_hip.const_params import ContactParams
    dhat = ContactParams().dhat
    spec = helpers.one_cube([0.0, 0.5 + 0.5 * dhat, 0.0], [0.0, 0.0, 0.0], ground=0.0)
    cp = ContactParams(ground=0.0, solver=1, solver_tol=1e30, max_iter=1)
    dq = np.zeros((4, 3))
    dq[0, 1] = 0.3 * dhat  # the step is -alpha dq
    sim = AffineBodySimulator(spec, cp, "cuda", native=True)
    sim.dq.copy_(torch.as_tensor(dq, device="cuda"))
    print("planted step towards the ground", flush=True)
    _lib.profile_select(["energy"])
    _lib.profile_begin()
    try:
        sim.step(0)
        torch.cuda.synchronize()
    finally:
        _lib.profile_end()
        _lib.profile_select(None)
    _, launches, nbytes = _lib.profile_query()["energy"]
    np.testing.assert_allclose(sim.states.p.cpu().numpy(), spec.p - 2.0 ** -10 * dq[:1], rtol=0, atol=1e-12)
    n, trials, passes = 4, 11, 2
    assert launches == 1 + passes
    assert nbytes == 32 * n + passes * 36 * n + 96 * trials
