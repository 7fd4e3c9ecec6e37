"""The step-by-step device walk: what the environment's switches select, and what
walks that walk_kernel does not take run (FP32 operands beyond 64 electrons a
spin, larger batches beyond 32).

* QMCB_GEMM_TILE and QMCB_SEPARATE_PROPOSE reach the kernels they name.
* Walker groups and the draw of the next proposal change no bit, in VMC and DMC.
* The FP64 walk's resident state is that of a fresh evaluate (1e-8, the rounding
  of n^2-term sums by the condition number of the Slater matrices).
* walk_kernel against the steps: FP64 operands with FP64 storage to rounding
  (1e-9 of the largest coordinate, 1e-8 of weights); with FP32 storage a
  last-bit difference can flip the rounding of a stored derivative, 2^-24 of a
  term of a drift of up to 10^3 times tau 0.02: 1e-5.
"""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth
from tests.test_gpu_walk import rel, system, walkers

pytestmark = pytest.mark.gpu


def launches(c, call):
    c.enable_timing(True)
    call()
    k = {n: v["launches"] for n, v in c.kernel_times().items()}
    c.enable_timing(False)
    return k


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32store"])
def test_switches_reach_the_kernels_they_name(precision, monkeypatch):
    p = system(32, 32)
    W, steps = 64, 6
    R0, ids = walkers(p, W, 1), np.arange(W)
    print("case walk switches", precision, flush=True)
    seen = {}
    for var, value in (("QMCB_GEMM_TILE", "4,2"), ("QMCB_SEPARATE_PROPOSE", "0"),
                       ("QMCB_SEPARATE_PROPOSE", "1")):
        with monkeypatch.context() as m:
            m.setenv(var, value)
            with Context(p, precision=precision, max_walkers=W, seed=1) as c:
                c.evaluate(ids, R0)
                seen[var, value] = launches(c, lambda: c.vmc_steps(W, 0, steps, 0.02))
    assert seen["QMCB_GEMM_TILE", "4,2"]["basis"] == steps
    assert seen["QMCB_GEMM_TILE", "4,2"]["orbital_gemm"] == steps
    assert seen["QMCB_SEPARATE_PROPOSE", "0"]["propose"] == 1
    assert seen["QMCB_SEPARATE_PROPOSE", "1"]["propose"] == steps


CASES = [(32, 32, "fp64", 800, "0"), (32, 20, "fp32", 800, "0"), (40, 9, "fp32", 1040, None),
         (75, 75, "fp32", 800, None), (66, 10, "bf16store", 800, None)]


@pytest.mark.parametrize("n_up,n_dn,precision,W,switch", CASES)
def test_groups_and_proposals_change_no_bit(n_up, n_dn, precision, W, switch, monkeypatch):
    p = system(n_up, n_dn)
    N = n_up + n_dn
    R0, ids = walkers(p, W, 2), np.arange(W)
    print("case step groups", n_up, n_dn, precision, flush=True)
    out = []
    for groups, env in ((1, switch), (2, switch), (3, switch), (-1, switch), (1, "1"), (3, "1")):
        with monkeypatch.context() as m:
            if env is not None:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(p, precision=precision, max_walkers=W, seed=6, drift_mod=1,
                         refresh_interval=20, walker_groups=groups) as c:
                c.evaluate(ids, R0)
                st = c.vmc_steps(W, n_up - 5, 70, 0.02)
                st2 = c.vmc_steps(W, n_up + 65, 90, 0.02)
                out.append((c.positions(W), c.sample_series(),
                            np.array([st.sum_e_local, st.sum_accept, st2.sum_e_local,
                                      st2.sum_accept])))
    assert np.any(out[0][0] != R0)
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("precision,switch", [("fp64", "0"), ("fp32", None)])
def test_dmc_groups_change_no_bit(precision, switch, monkeypatch):
    n = 33 if precision == "fp64" else 66
    p = system(n, 10)
    N, W = n + 10, 600
    R0, ids = walkers(p, W, 3), np.arange(W)
    print("case step dmc groups", precision, flush=True)
    out = []
    for groups in (1, 2, 3):
        with monkeypatch.context() as m:
            if switch is not None:
                m.setenv("QMCB_SEPARATE_PROPOSE", switch)
            with Context(p, precision=precision, max_walkers=2 * W, seed=6, drift_mod=1,
                         refresh_interval=16, walker_groups=groups) as c:
                e = c.evaluate(ids, R0)["e_local"]
                c.dmc_init(W)
                c.dmc_steps(0, 2 * N + 5, 0.001, float(np.median(e)), target=W, reweight_after=0,
                            energy_modification=True)
                slots, wts = c.dmc_population()
                out.append((np.asarray(slots), np.asarray(wts), c.positions(2 * W)[slots],
                            c.sample_series()))
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n_up,n_dn,precision", [(16, 7, "fp64"), (50, 50, "fp64"),
                                                 (90, 30, "fp64"), (128, 100, "fp64"),
                                                 (32, 32, "fp32store"), (100, 70, "fp32store")])
def test_walk_kernel_and_steps_agree(n_up, n_dn, precision, monkeypatch):
    p = system(n_up, n_dn)
    N, W, steps = n_up + n_dn, 12, 40
    R0, ids = walkers(p, W, 4), np.arange(W)
    print("case walk against steps", n_up, n_dn, precision, flush=True)
    out = []
    for env in (None, "0"):
        with monkeypatch.context() as m:
            if env:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(p, precision=precision, max_walkers=W, seed=8, drift_mod=1,
                         refresh_interval=15) as c:
                ok = c.evaluate(ids, R0)["singular"] == 0
                st = c.vmc_steps(W, max(0, n_up - 20), steps, 0.02)
                R = c.positions(W)
                res = c.evaluate(ids, R, whichE=N - 1)
                out.append((R, res.a["e_local"].copy(), res.a["grad_lnpsi"].copy(),
                            st.sum_accept))
    tol = 1e-9 if precision == "fp64" else 1e-5
    assert out[0][3] == out[1][3] > 0 and ok.sum() >= W - 2
    np.testing.assert_allclose(out[1][0][ok], out[0][0][ok], rtol=0, atol=tol * np.abs(R0).max())
    if precision == "fp64":
        with Context(p, precision=precision, max_walkers=W, drift_mod=1) as fresh:
            ok &= fresh.evaluate(ids, out[1][0])["singular"] == 0
            ref = fresh.evaluate(ids, out[1][0], whichE=N - 1)
        assert rel(out[1][1][ok], ref.a["e_local"][ok]) < 1e-8
        assert rel(out[1][2][ok], ref.a["grad_lnpsi"][ok]) < 1e-8


def test_dmc_with_cusps_agrees_with_the_steps(monkeypatch):
    s = synth.make_system(-1, seed=5, n_elec=38)
    W = 32
    R0, ids = synth.initial_walkers(s, W, 4), np.arange(W)
    print("case dmc cusps against steps", flush=True)
    out = []
    for env in (None, "0"):
        with monkeypatch.context() as m:
            if env:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(s.pack(), precision="fp64", max_walkers=2 * W, seed=2, drift_mod=1,
                         replace_cusps=True) as c:
                e = c.evaluate(ids, R0)["e_local"]
                c.dmc_init(W)
                c.dmc_steps(0, 2 * 38 + 5, 0.01, float(np.median(e)), target=W, reweight_after=30,
                            energy_modification=True)
                slots, wts = c.dmc_population()
                out.append((np.asarray(slots), np.asarray(wts), c.positions(2 * W)[slots]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-8, atol=0)
    np.testing.assert_allclose(out[1][2], out[0][2], rtol=0, atol=1e-9 * np.abs(R0).max())


def test_kernel_timing_leaves_runs_whole():
    """With kernel timing a run of steps is still one launch, counted as its
    steps: one reduction of the samples a call, not one a sweep."""
    s = synth.make_system(0)
    W, steps = 64, 40
    R0, ids = synth.initial_walkers(s, W, 4), np.arange(W)
    print("case walk timing", flush=True)
    with Context(s.pack(), precision="fp64", max_walkers=W, seed=2) as c:
        c.evaluate(ids, R0)
        k = launches(c, lambda: c.vmc_steps(W, 0, steps, 0.1))
        rows = c.sample_series()
    assert k["sm_move"] == steps and k["series"] == 1
    assert len(rows) == steps // 2


@pytest.mark.parametrize("n_elec", [38, 76])
def test_old_walkers_and_weights_either_way(n_elec, monkeypatch):
    """FP32 operands: walk_kernel and the steps take walkers through the same
    bits also where ages boost acceptances and decide deletions
    (old_walker_acceptance 2); weights and samples, whose energies are summed in
    another order, agree to 1e-12, ln of the ratio of two such sums."""
    s = synth.make_system(-1, seed=5, n_elec=n_elec)
    W = 300
    R0, ids = synth.initial_walkers(s, W, 4), np.arange(W)
    print("case old walkers", n_elec, flush=True)
    out = []
    for env in (None, "0"):
        with monkeypatch.context() as m:
            if env:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(s.pack(), precision="fp32", max_walkers=2 * W, seed=2, drift_mod=1,
                         old_walker_acceptance=2) as c:
                c.evaluate(ids, R0)
                c.vmc_steps(W, 0, 4 * n_elec + 1, 0.2)
                rows, R = c.sample_series().copy(), c.positions(W)
                e = c.evaluate(ids, R)["e_local"]
                c.dmc_init(W)
                c.dmc_steps(0, 3 * n_elec + 1, 0.003, float(np.median(e)), target=W,
                            reweight_after=0, energy_modification=True)
                slots, wts = c.dmc_population()
                out.append((R, np.asarray(slots), c.positions(2 * W)[slots], rows,
                            np.asarray(wts), c.sample_series()))
    for i in range(3):
        np.testing.assert_array_equal(out[0][i], out[1][i])
    for i in range(3, 6):
        np.testing.assert_allclose(out[0][i], out[1][i], rtol=1e-12, atol=0)


@pytest.mark.parametrize("n_up,n_dn", [(40, 9), (64, 16), (40, 17), (33, 0)])
def test_same_bits_either_side_of_the_batch_rule(n_up, n_dn):
    """FP32 operands, 33 to 64 up electrons: walkers among 1000 and among 1040."""
    p = system(n_up, n_dn)
    R0 = walkers(p, 1040, 5)
    print("case batch rule", n_up, n_dn, flush=True)
    out = []
    for W in (1000, 1040):
        with Context(p, precision="fp32", max_walkers=W, seed=4, drift_mod=1) as c:
            c.evaluate(np.arange(W), R0[:W])
            c.vmc_steps(W, n_up - 10, 60, 0.02)
            out.append(c.positions(W)[:1000])
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("n", [40, 80, 110])
def test_later_moves_take_rows_as_stored(n, monkeypatch):
    """FP64 operands, FP32 storage, beyond 32 electrons a spin: walk_kernel's block
    uses the replaced electrons' derivatives as they are stored, so its gradients
    are those of the steps (1e-9; a walker in ten may have had a rounding flipped
    by a last bit).  With the rows as formed they differ by 2^-24 times the
    condition numbers, 10^-6."""
    p = system(n, n)
    N, W = 2 * n, 40
    R0, ids = walkers(p, W, 4), np.arange(W)
    print("case rows as stored", n, flush=True)
    out = []
    for env in (None, "0"):
        with monkeypatch.context() as m:
            if env:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(p, precision="fp32store", max_walkers=W, seed=3) as c:
                ok = c.evaluate(ids, R0)["singular"] == 0
                c.vmc_steps(W, 3, 20, 0.02)
                R = c.positions(W)
                out.append((R, c.evaluate(ids, R, whichE=N - 1).a["grad_lnpsi"].copy()))
    err = np.max(np.abs(out[0][1] - out[1][1]) / np.maximum(1.0, np.abs(out[1][1])), axis=(1, 2))
    assert ok.sum() >= W - 4
    assert np.mean(err[ok] < 1e-9) >= 0.9, np.sort(err[ok])
