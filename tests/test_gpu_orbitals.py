"""The fused basis-and-contraction kernel (orbitals.hip) against the two
kernels it replaces, which a fixed contraction tile (QMCB_GEMM_TILE) selects:
the same functions summed in the same order, so every result of an
all-electron evaluate, a staged move and the accepted state must agree bit
for bit.

300 basis functions (the last chunk of 32 holds 12), orbital counts at the
edges of its tiles (1, 16, 17, 32 with unequal spins) and of its workgroups
(64, 65 and 128, 140 active), point counts at the edges of a 16-point tile and
either side of the rule that picks the kernel (256 workgroups: 4096 points of
up to 64 orbitals), and active orbitals beyond the occupied ones.
"""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth

pytestmark = pytest.mark.gpu

FIELDS = ("log_psi", "sign_psi", "grad_lnpsi", "mod_drift", "lap_ratio", "e_local", "det_ratio")


def system(n_up, n_dn, n_act=0):
    p = dict(synth.make_system(1).pack())
    rng = np.random.default_rng(1000 * n_up + n_dn)
    na, nb = n_act or n_up, n_act or n_dn
    q, _ = np.linalg.qr(rng.normal(size=(p["n_basis"], na + nb)))
    p["n_up"], p["n_dn"] = n_up, n_dn
    p["mo_up"] = np.ascontiguousarray(q[:, :na].T)
    p["mo_dn"] = np.ascontiguousarray(q[:, na:].T)
    if n_act:
        occ = np.stack([np.arange(n_up), np.r_[np.arange(n_up - 1), n_act - 1]])
        p["n_det"], p["ci_coef"] = 2, np.array([0.9, 0.3])
        p["n_act_up"] = p["n_act_dn"] = n_act
        p["occ_up"] = np.ascontiguousarray(occ, dtype=np.int32)
        p["occ_dn"] = np.ascontiguousarray(occ[:, :n_dn] % n_act, dtype=np.int32)
    return p


def run(p, R, precision, tile, monkeypatch):
    if tile:
        monkeypatch.setenv("QMCB_GEMM_TILE", tile)
    else:
        monkeypatch.delenv("QMCB_GEMM_TILE", raising=False)
    W, N = R.shape[:2]
    ids = np.arange(W)
    out = []
    with Context(p, precision=precision, max_walkers=W) as c:
        out.append(c.evaluate(ids, R))
        for m in (0, N - 1):
            X = R.copy()
            X[:, m] += 0.05
            out.append(c.evaluate(ids, X, m))
            c.accept(ids, ids % 2 == 0)
            R = np.where((ids % 2 == 0)[:, None, None], X, R)
        out.append(c.evaluate(ids, R, 0))
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32store", "bf16store"])
@pytest.mark.parametrize("n_up,n_dn,n_act,W", [
    (1, 1, 0, 33), (17, 16, 0, 5), (32, 15, 0, 257), (64, 1, 0, 127), (64, 1, 0, 129),
    (65, 64, 0, 16), (128, 128, 0, 3), (1, 1, 0, 4096), (2, 1, 0, 4097), (5, 5, 9, 40),
    (3, 3, 140, 40),
])
def test_fused_equals_separate(precision, n_up, n_dn, n_act, W, monkeypatch):
    print("case orbitals", precision, n_up, n_dn, n_act, W, flush=True)
    p = system(n_up, n_dn, n_act)
    rng = np.random.default_rng(W)
    xyz = np.asarray(p["nuc_xyz"]).reshape(-1, 3)
    N = n_up + n_dn
    R = xyz[rng.integers(0, len(xyz), size=(W, N))] + rng.normal(scale=0.8, size=(W, N, 3))
    a = run(p, R, precision, None, monkeypatch)
    b = run(p, R, precision, "4,1", monkeypatch)
    for i, (x, y) in enumerate(zip(a, b)):
        for f in FIELDS:
            np.testing.assert_array_equal(x.a[f], y.a[f], err_msg=f"call {i} {f}")
