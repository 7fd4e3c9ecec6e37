"""Runs of single-electron steps in one launch (walk.hip) at the edges of its
column tiles (16, 32, 64, 96, 128 electrons a spin), with unequal spins, each
operand type, cusp replacement and a Pade function of more than one term.

* The resident state after a walk is that of a fresh all-electron evaluate of
  the same positions: the same zero-length move of the last electron from
  either gives the same results (not asked of FP32 storage under an FP64 GEMM,
  where a moved electron's row enters its own traces unrounded and is stored
  rounded, so a walk's gradients differ from a fresh evaluate's by 2^-24 times
  the condition number, in the step-by-step kernels too).  Tolerances: FP64 rounding of n^2-term sums amplified by
  the Slater condition numbers of these random-orbital molecules (10^3-10^5 x
  10^-16 x the steps' accumulation): 1e-8; with FP32 operands the same, since
  the resident and the fresh state hold the same rounded rows.
* One call of K steps and K calls of one step draw the same numbers and follow
  the same walk: bit for bit where every sum is formed afresh at each move
  (FP32 operands, or FP64 ones up to 32 electrons a spin), to rounding (1e-9
  relative to the largest coordinate) where T1 and T2 are carried through a
  block.
* FP32 operands, 33-64 electrons: the batch sizes either side of the rule that
  picks this kernel give a walker the same bits.
"""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth

pytestmark = pytest.mark.gpu


def system(n_up, n_dn, terms=1):
    p = dict(synth.make_system(1).pack())
    rng = np.random.default_rng(100 * n_up + n_dn)
    q, _ = np.linalg.qr(rng.normal(size=(p["n_basis"], n_up + n_dn)))
    p["n_up"], p["n_dn"] = n_up, n_dn
    p["mo_up"] = np.ascontiguousarray(q[:, :n_up].T)
    p["mo_dn"] = np.ascontiguousarray(q[:, n_up:].T)
    if terms > 1:  # u = (a r + c r^2) / (1 + b r + d r^2)
        for k in ("ee_updn", "ee_upup", "ee_dndn"):
            row = p[k].copy()
            row[0] = row[1] = 2
            row[3], row[3 + synth.PADE_MAX] = 0.05, 0.3
            p[k] = row
    return p


def walkers(p, W, seed):
    N = p["n_up"] + p["n_dn"]
    rng = np.random.default_rng(seed)
    return p["nuc_xyz"][rng.integers(0, p["n_nuc"], size=(W, N))] + 0.8 * rng.normal(size=(W, N, 3))


def rel(a, b):
    return float(np.max(np.abs(a - b) / np.maximum(1.0, np.abs(b))))


CASES = [(1, 0, "fp64"), (1, 1, "fp32"), (16, 16, "fp32"), (17, 3, "fp32"), (17, 17, "fp64"),
         (32, 32, "fp32store"), (32, 31, "bf16store"), (33, 33, "fp32"), (33, 20, "fp64"),
         (64, 64, "fp32"), (64, 64, "fp64"), (65, 9, "fp64"), (96, 96, "fp32store"),
         (97, 97, "fp64"), (128, 128, "fp64")]


@pytest.mark.parametrize("n_up,n_dn,precision", CASES)
@pytest.mark.parametrize("drift", [0, 1])
def test_walk_state_and_call_splits(n_up, n_dn, precision, drift):
    p = system(n_up, n_dn, terms=2 if n_up in (17, 65) else 1)
    N, W = n_up + n_dn, 12
    steps = min(N, 40) + 5
    print("case walk", n_up, n_dn, precision, "drift", drift, flush=True)
    R0, ids = walkers(p, W, 3), np.arange(W)
    kw = dict(precision=precision, max_walkers=W, seed=11, drift_mod=drift,
              refresh_interval=7 if precision == "fp32" else 0)
    first = max(0, n_up - 20)  # cross from one spin to the other
    out = []
    for calls in (1, steps):
        with Context(p, **kw) as c:
            c.evaluate(ids, R0)
            for k in range(calls):
                c.vmc_steps(W, first + k, steps // calls, 0.02)
            R = c.positions(W)
            res = c.evaluate(ids, R, whichE=N - 1)  # zero-length move
            out.append((R, res.a["e_local"].copy(), res.a["log_psi"].copy(),
                        res.a["grad_lnpsi"].copy()))
    if precision in ("fp32", "bf16store") or n_up <= 32:
        np.testing.assert_array_equal(out[0][0], out[1][0])
    else:
        np.testing.assert_allclose(out[0][0], out[1][0], rtol=0, atol=1e-9 * np.abs(R0).max())
    assert np.any(out[0][0] != R0)
    if precision == "fp32store":
        return
    with Context(p, precision=precision, max_walkers=W, drift_mod=drift) as fresh:
        ok = fresh.evaluate(ids, out[0][0])["singular"] == 0
        ref = fresh.evaluate(ids, out[0][0], whichE=N - 1)
    assert ok.sum() >= W - 2
    for i, k in ((1, "e_local"), (2, "log_psi"), (3, "grad_lnpsi")):
        assert rel(out[0][i][ok], ref.a[k][ok]) < 1e-8, k


def test_walk_cusps_dmc_state():
    """Cusp replacement inside the run, and DMC weights: the walk of a branching
    population stays consistent with a fresh evaluate."""
    s = synth.make_system(-1, seed=5, n_elec=38)
    W = 32
    print("case walk cusps dmc 38", flush=True)
    R0, ids = synth.initial_walkers(s, W, 4), np.arange(W)
    with Context(s.pack(), precision="fp64", max_walkers=2 * W, seed=2, drift_mod=1,
                 replace_cusps=True) as c:
        e = c.evaluate(ids, R0)["e_local"]
        c.dmc_init(W)
        c.dmc_steps(0, 3 * 38 + 5, 0.01, float(np.median(e)), target=W, reweight_after=30,
                    energy_modification=True)
        slots, _ = c.dmc_population()
        R = c.positions(2 * W)[slots]
        res = c.evaluate(slots, R, whichE=0).a["e_local"]
    with Context(s.pack(), precision="fp64", max_walkers=2 * W, drift_mod=1,
                 replace_cusps=True) as fresh:
        ref = fresh.evaluate(np.arange(len(slots)), R)
    ok = ref["singular"] == 0
    assert rel(res[ok], ref["e_local"][ok]) < 1e-8


def test_walk_same_bits_either_side_of_the_batch_rule():
    """120 electrons, FP32 operands: walkers of a batch of 1024 (one launch per
    run) and the same ones among 1040 (step by step)."""
    s = synth.make_system(-1, seed=5, n_elec=120)
    R0 = synth.initial_walkers(s, 1040, 8)
    print("case walk batch rule 120", flush=True)
    out = []
    for W in (1024, 1040):
        with Context(s.pack(), precision="fp32", max_walkers=W, seed=4, drift_mod=1,
                     refresh_interval=16) as c:
            c.evaluate(np.arange(W), R0[:W])
            c.vmc_steps(W, 50, 24, 0.02)
            out.append(c.positions(W)[:1024])
    np.testing.assert_array_equal(out[0], out[1])
