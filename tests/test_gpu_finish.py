"""The end of an all-electron evaluate (finish.hip: traces, Jastrow pair tiles,
assembly) against the oracle, FP64, at the edges of its tiles: 64 electrons a
tile (2, 64, 65, 128, 129 and 256 electrons, unequal spins) and 40 nuclei a
tile (10, 41), with Pade functions of one and of two terms.

Tolerances: pair sums (U, V_ee, V_ne) 1e-12 relative, at most 256^2 terms of
2^-53 each; everything that carries an inverse 1e-8, FP64 rounding amplified by
the condition numbers (10^3-10^5) of these random-orbital Slater matrices.
"""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from qmcbeaver_amd import Context, synth

pytestmark = pytest.mark.gpu


def system(n_up, n_dn, terms, n_nuc):
    p = dict(synth.make_system(1).pack())
    rng = np.random.default_rng(100 * n_up + n_dn + n_nuc)
    q, _ = np.linalg.qr(rng.normal(size=(p["n_basis"], n_up + n_dn)))
    p["n_up"], p["n_dn"] = n_up, n_dn
    p["mo_up"] = np.ascontiguousarray(q[:, :n_up].T)
    p["mo_dn"] = np.ascontiguousarray(q[:, n_up:].T)
    more = n_nuc - p["n_nuc"]
    if more:  # bare charges: nuclei without basis functions
        p["n_nuc"] = n_nuc
        p["nuc_xyz"] = np.concatenate([np.reshape(p["nuc_xyz"], (-1, 3)),
                                       rng.normal(scale=6.0, size=(more, 3))])
        p["nuc_z"] = np.concatenate([p["nuc_z"], np.ones(more)])
        for k in ("en_up", "en_dn"):
            p[k] = np.concatenate([p[k], np.repeat(p[k][:1], more, axis=0)])
    if terms > 1:  # u = (a r + c r^2) / (1 + b r + d r^2)
        for k in ("ee_updn", "ee_upup", "ee_dndn"):
            row = p[k].copy()
            row[0] = row[1] = 2
            row[3], row[3 + synth.PADE_MAX] = 0.05, 0.3
            p[k] = row
    return p


@pytest.mark.parametrize("n_up,n_dn,terms,n_nuc", [
    (1, 1, 1, 10), (32, 32, 1, 10), (33, 32, 2, 10), (64, 64, 1, 41), (80, 49, 1, 10),
    (128, 128, 2, 41),
])
def test_evaluate_matches_oracle(n_up, n_dn, terms, n_nuc):
    print("case finish", n_up, n_dn, terms, n_nuc, flush=True)
    p = system(n_up, n_dn, terms, n_nuc)
    N, W = n_up + n_dn, 3
    rng = np.random.default_rng(N)
    xyz = np.reshape(p["nuc_xyz"], (-1, 3))
    R = xyz[rng.integers(0, len(xyz), size=(W, N))] + rng.normal(scale=0.9, size=(W, N, 3))
    with Context(p, precision="fp64", max_walkers=W) as c:
        got = c.evaluate(range(W), R)
    want = Oracle(p).evaluate_all(R)
    for f, tol in (("jastrow_u", 1e-12), ("v_ee", 1e-12), ("v_ne", 1e-12), ("log_psi", 1e-8),
                   ("grad_lnpsi", 1e-8), ("lap_ratio", 1e-8), ("e_local", 1e-8)):
        a, b = got.a[f], want.a[f]
        ok = np.isfinite(b)  # the oracle's determinant is a plain product: one may underflow
        assert ok.sum() * 3 >= 2 * ok.size and np.isfinite(a).all(), f
        err = np.max(np.abs(a - b)[ok]) / max(1.0, np.max(np.abs(b[ok])))
        assert err < tol, (f, err)
    ok = np.isfinite(want.a["log_psi"])  # ... and has no sign
    np.testing.assert_array_equal(got.a["sign_psi"][ok], want.a["sign_psi"][ok])
