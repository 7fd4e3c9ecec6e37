"""Large batches whose staggered re-inversion comes in short phases walk step by
step: which batches do, and that a walk that changes between the two ways with
its batch is that of the steps alone (FP32 operands with equal spins the same
positions; FP64 to 1e-9 of the largest coordinate, with FP32 storage 1e-5, for 99
of 100 walkers: the rest allows for matrices of a condition number beyond 10^6
and for moves that a last bit decides)."""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth
from tests.test_gpu_walk import system, walkers
from tests.test_gpu_walk_steps import launches

pytestmark = pytest.mark.gpu


# phases of S = ceil(1024 K / W) moves
CASES = [(17, "fp32", 4096, 8, True), (17, "fp32", 4095, 8, False), (32, "fp32", 4096, 12, False),
         (17, "fp32", 4096, 1, False), (32, "fp32", 8192, 32, True), (32, "fp32", 8192, 33, False),
         (17, "fp64", 6144, 6, True), (17, "fp64", 6143, 6, False), (17, "fp64", 6144, 7, False),
         (17, "fp64", 6144, 2, False), (1, "fp32", 32768, 32, True), (1, "fp64", 32767, 31, False),
         (16, "fp64", 32768, 2, True), (1, "fp64", 32768, 33, False), (1, "fp32", 32768, 0, False),
         (33, "fp64", 3940, 2, True), (33, "fp64", 3939, 4, False), (33, "fp64", 3940, 4, True),
         (64, "fp64", 1016, 1, True), (64, "fp64", 1015, 1, False), (65, "fp64", 1000, 1, True),
         (65, "fp64", 1500, 2, False), (65, "fp64", 1500, 0, False)]


@pytest.mark.parametrize("n,precision,W,K,steps", CASES)
def test_which_batches_walk_step_by_step(n, precision, W, K, steps):
    p = synth.make_system(0).pack() if n == 1 else system(n, n)
    R0 = np.tile(walkers(p, 32, 1), (-(-W // 32), 1, 1))[:W]
    print("case short phases", n, precision, W, K, flush=True)
    with Context(p, precision=precision, max_walkers=W, seed=2, refresh_interval=K) as c:
        c.evaluate(np.arange(W), R0)
        k = launches(c, lambda: c.vmc_steps(W, 0, 3, 0.02))
    assert k["sm_move"] == 3
    assert (k.get("propose", 0) > 0) == steps


@pytest.mark.parametrize("n,precision,W,K", [(17, "fp32", 4096, 4), (17, "fp64", 6144, 4),
                                             (17, "fp32store", 6144, 4), (40, "fp64", 2050, 2),
                                             (65, "fp64", 2050, 2)])
def test_changing_ways_with_the_batch(n, precision, W, K, monkeypatch):
    p = system(n, n)
    R0 = walkers(p, W, 3)
    print("case short phases change", n, precision, flush=True)
    out = []
    for env in (None, "0"):
        with monkeypatch.context() as m:
            if env:
                m.setenv("QMCB_SEPARATE_PROPOSE", env)
            with Context(p, precision=precision, max_walkers=W, seed=5, drift_mod=1,
                         refresh_interval=K) as c:
                ok = c.evaluate(np.arange(W), R0)["singular"] == 0
                at, rows = 10, []
                for num, k in ((700, 7), (W, 9), (700, 11), (W, 8), (W, 3), (700, 10)):
                    c.vmc_steps(num, at, k, 0.02)
                    at += k
                    rows.append(c.sample_series().copy())
                out.append((c.positions(W), rows))
    assert np.any(out[0][0] != R0) and ok.sum() >= W - 20
    if precision == "fp32":
        np.testing.assert_array_equal(out[0][0], out[1][0])
    else:
        tol = 1e-9 if precision == "fp64" else 1e-5
        d = np.abs(out[0][0] - out[1][0])[ok].max(axis=(1, 2))
        assert np.mean(d <= tol * np.abs(R0).max()) >= 0.99, np.sort(d)[-80:]
    assert [len(r) for r in out[0][1]] == [len(r) for r in out[1][1]]
