"""The FP64 device walk beyond 32 electrons a spin carries sums through a block
of moves.  A walk has the same bits however it is cut into launches:

* one call, calls of 1 to 7 steps, and the same steps with kernel timing on;
* walker_groups 1, 2, 3 and -1 (whose timing windows are calls of their own),
  with re-inversions, which end a run for every walker and touch a few;
* DMC calls of one step and of a whole block, with branching.

Between calls the kept sums do not outlive the state they belong to: an accept,
a refresh or an evaluate between two calls gives what a fresh evaluate of the
same positions gives (1e-8, the rounding of n^2-term sums by the condition
number of the Slater matrices)."""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth
from tests.test_gpu_walk import rel, system, walkers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_up,n_dn,precision", [(33, 20, "fp64"), (64, 64, "fp64"),
                                                 (75, 9, "fp32store"), (96, 65, "fp64"),
                                                 (101, 100, "fp64"), (128, 128, "fp32store")])
def test_walk_bits_do_not_depend_on_the_cuts(n_up, n_dn, precision):
    p = system(n_up, n_dn)
    N, W = n_up + n_dn, 10
    first, steps = max(0, n_up - 13), 31  # into the other spin, not on a block's end
    R0, ids = walkers(p, W, 5), np.arange(W)
    print("case walk cuts", n_up, n_dn, precision, flush=True)
    out = []
    for cut in (steps, 1, 7, "timing"):
        with Context(p, precision=precision, max_walkers=W, seed=3, drift_mod=1,
                     refresh_interval=12) as c:
            c.evaluate(ids, R0)
            c.enable_timing(cut == "timing")
            size = steps if cut == "timing" else cut
            for k in range(0, steps, size):
                c.vmc_steps(W, first + k, min(size, steps - k), 0.02)
            c.enable_timing(False)
            R = c.positions(W)
            res = c.evaluate(ids, R, whichE=(first + steps) % N)  # zero-length move
            out.append((R, res.a["e_local"].copy(), res.a["grad_lnpsi"].copy()))
    assert np.any(out[0][0] != R0)
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


def test_walk_bits_do_not_depend_on_walker_groups():
    p = system(75, 75)
    N, W = 150, 800
    R0, ids = walkers(p, W, 6), np.arange(W)
    print("case walk groups 75", flush=True)
    out = []
    for groups in (1, 2, 3, -1):
        with Context(p, precision="fp64", max_walkers=W, seed=9, refresh_interval=30,
                     walker_groups=groups) as c:
            c.evaluate(ids, R0)
            st = c.vmc_steps(W, 3, N + 20, 0.02)
            out.append((c.positions(W), c.sample_series(), np.array([st.sum_e_local,
                                                                     st.sum_accept])))
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


def test_dmc_bits_do_not_depend_on_call_lengths():
    s = synth.make_system(-1, seed=5, n_elec=70)
    N, W = 70, 40
    R0, ids = synth.initial_walkers(s, W, 4), np.arange(W)
    print("case dmc cuts 70", flush=True)
    out = []
    for size in (2 * N + 9, 1, 11):
        with Context(s.pack(), precision="fp64", max_walkers=2 * W, seed=2, drift_mod=1) as c:
            e = float(np.median(c.evaluate(ids, R0)["e_local"]))
            c.vmc_steps(W, 0, 5, 0.01)  # leaves a block unfinished
            c.dmc_init(W)
            steps = 2 * N + 9
            for k in range(0, steps, size):
                c.dmc_steps(5 + k, min(size, steps - k), 0.01, e, target=W, reweight_after=0,
                            energy_modification=True)
            slots, wts = c.dmc_population()
            out.append((np.asarray(slots), np.asarray(wts), c.positions(2 * W)))
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("between", ["accept", "refresh", "evaluate"])
def test_kept_sums_end_with_the_state_they_belong_to(between):
    n = 50
    p = system(n, n)
    N, W = 2 * n, 10
    R0, ids = walkers(p, W, 7), np.arange(W)
    print("case walk kept sums", between, flush=True)
    with Context(p, precision="fp64", max_walkers=W, seed=3) as c, \
            Context(p, precision="fp64", max_walkers=W) as fresh:
        c.evaluate(ids, R0)
        c.vmc_steps(W, 0, 11, 0.02)  # the block of electrons 8-15 is open at 11
        if between == "accept":  # move electron 30 of every second walker
            R = c.positions(W)
            R[:, 30] += 0.2
            c.evaluate(ids, R, whichE=30)
            c.accept(ids, (ids % 2).astype(np.uint8))
        elif between == "refresh":
            c.refresh(ids)
        else:
            R = c.positions(W)
            R[:, 30] += 0.2
            c.evaluate(ids, R)
        c.vmc_steps(W, 11, 3, 0.02)
        R = c.positions(W)
        res = c.evaluate(ids, R, whichE=N - 1)
        ok = fresh.evaluate(ids, R)["singular"] == 0
        ref = fresh.evaluate(ids, R, whichE=N - 1)
    assert ok.sum() >= W - 2
    for k in ("e_local", "log_psi", "grad_lnpsi"):
        assert rel(res.a[k][ok], ref.a[k][ok]) < 1e-8, k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_plan_counts_the_kept_sums(precision):
    from qmcbeaver_amd.core import plan_device_bytes
    p = system(50, 40)
    print("case walk plan", precision, flush=True)
    with Context(p, precision=precision, max_walkers=77) as c:
        assert c.device_bytes() == plan_device_bytes(p, precision=precision, max_walkers=77)


def test_all_electron_contexts_hold_no_kept_sums():
    p = system(50, 40)
    W, held = 1000, []
    print("case walk memory, all-electron moves", flush=True)
    for every in (False, True):
        with Context(p, precision="fp64", max_walkers=W, all_electron_moves=every) as c:
            held.append(c.device_bytes())
            c.evaluate(np.arange(8), walkers(p, 8, 3))
            assert np.isfinite(c.vmc_steps(8, 0, 3, 0.01).sum_e_local)
    # a block's sums, 8 x 8 x 50 numbers a walker, against a record of 3 x 90 + 4
    assert held[1] < held[0]
