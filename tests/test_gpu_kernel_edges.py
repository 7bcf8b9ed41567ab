"""Kernels at the sizes where their work splits can go wrong (one item, remainders, one more
than a full grid), against the oracle."""
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
