"""The one-wave form of the end of an all-electron evaluate (up to 16 electrons)
against the oracle, FP64, at its edges: 1, 2, 3, 15, 16 electrons (17 take the
other form), 10, 16, 17 and 41 nuclei (16 a tile), Pade functions of one and of
two terms.  Tolerances as in test_gpu_finish: pair sums 1e-12 relative, what
carries an inverse 1e-8."""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from qmcbeaver_amd import Context
from tests.test_gpu_finish import system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_up,n_dn,terms,n_nuc", [
    (1, 0, 1, 10), (1, 1, 2, 17), (2, 1, 1, 16), (8, 7, 2, 41), (8, 8, 1, 10), (15, 1, 1, 17),
    (9, 8, 1, 17),
])
def test_small_evaluate_matches_oracle(n_up, n_dn, terms, n_nuc):
    print("case finish small", n_up, n_dn, terms, n_nuc, flush=True)
    p = system(n_up, n_dn, terms, n_nuc)
    N, W = n_up + n_dn, 5
    rng = np.random.default_rng(N)
    xyz = np.reshape(p["nuc_xyz"], (-1, 3))
    R = xyz[rng.integers(0, len(xyz), size=(W, N))] + rng.normal(scale=0.9, size=(W, N, 3))
    with Context(p, precision="fp64", max_walkers=W) as c:
        got = c.evaluate(range(W), R)
    want = Oracle(p).evaluate_all(R)
    for f, tol in (("jastrow_u", 1e-12), ("v_ee", 1e-12), ("v_ne", 1e-12), ("log_psi", 1e-8),
                   ("grad_lnpsi", 1e-8), ("lap_ratio", 1e-8), ("e_local", 1e-8)):
        a, b = got.a[f], want.a[f]
        assert np.isfinite(a).all(), f
        err = np.max(np.abs(a - b)) / max(1.0, np.max(np.abs(b)))
        assert err < tol, (f, err)
    np.testing.assert_array_equal(got.a["sign_psi"], want.a["sign_psi"])
