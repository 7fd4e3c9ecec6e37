"""The wave-a-matrix inverse (n <= 32 a spin) against the oracle, FP64, at the
edges of its tiles (16 and 32) and with both spins in one launch (same tile)
or two, batches that do not fill a workgroup of four matrices, and a singular
walker among regular ones (an electron so far away that its row is zero).

Tolerance 1e-8: FP64 rounding amplified by condition numbers of 10^3-10^5.
"""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from qmcbeaver_amd import Context, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_up,n_dn,W", [
    (1, 1, 5), (15, 2, 3), (16, 16, 9), (17, 16, 6), (31, 17, 1), (32, 32, 7), (32, 5, 4),
])
def test_small_inverse_matches_oracle(n_up, n_dn, W):
    print("case small inverse", n_up, n_dn, W, flush=True)
    p = dict(synth.make_system(1).pack())
    rng = np.random.default_rng(100 * n_up + n_dn)
    N = n_up + n_dn
    q, _ = np.linalg.qr(rng.normal(size=(p["n_basis"], N)))
    p["n_up"], p["n_dn"] = n_up, n_dn
    p["mo_up"] = np.ascontiguousarray(q[:, :n_up].T)
    p["mo_dn"] = np.ascontiguousarray(q[:, n_up:].T)
    xyz = np.reshape(p["nuc_xyz"], (-1, 3))
    R = xyz[rng.integers(0, len(xyz), size=(W, N))] + 0.8 * rng.normal(size=(W, N, 3))
    bad = W - 1 if W > 3 else -1
    want = Oracle(p).evaluate_all(R)
    if bad >= 0:
        R[bad, 0] = 1.0e4
    ids = np.arange(W)[::-1].copy()  # slots in another order than rows
    with Context(p, precision="fp64", max_walkers=W) as c:
        got = c.evaluate(ids, R)
    ok = np.arange(W) != bad
    np.testing.assert_array_equal(got.a["singular"].astype(bool), ~ok)
    np.testing.assert_array_equal(got.a["sign_psi"][ok], want.a["sign_psi"][ok])
    for f in ("log_psi", "grad_lnpsi", "lap_ratio", "e_local"):
        a, b = got.a[f][ok], want.a[f][ok]
        err = np.max(np.abs(a - b)) / max(1.0, np.max(np.abs(b)))
        assert err < 1e-8, (f, err)
