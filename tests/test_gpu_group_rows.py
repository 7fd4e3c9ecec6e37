"""Walker groups of a system whose spins are padded to different orbital counts:
the groups run on streams of their own, and one moves electrons of the other
spin while another still reads its rows.  Groups change no bit, across several
changes of spin, in VMC and DMC."""
import numpy as np
import pytest

from qmcbeaver_amd import Context
from tests.test_gpu_walk import system, walkers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_up,n_dn,precision,W", [(40, 9, "fp32", 1040), (66, 10, "fp32", 800),
                                                   (66, 10, "bf16store", 800),
                                                   (100, 40, "fp32", 800)])
def test_groups_of_unequal_spins(n_up, n_dn, precision, W):
    p = system(n_up, n_dn)
    N = n_up + n_dn
    R0, ids = walkers(p, W, 2), np.arange(W)
    print("case group rows", n_up, n_dn, precision, flush=True)
    out = []
    for groups in (1, 2, 3):
        with Context(p, precision=precision, max_walkers=2 * W, seed=6, drift_mod=1,
                     refresh_interval=20, walker_groups=groups) as c:
            e = c.evaluate(ids, R0)["e_local"]
            st = c.vmc_steps(W, n_up - 5, 2 * N + 20, 0.02)
            R = c.positions(W)
            c.dmc_init(W)
            c.dmc_steps(0, N + 15, 0.001, float(np.median(e)), target=W, reweight_after=0)
            slots, wts = c.dmc_population()
            out.append((R, np.array([st.sum_e_local, st.sum_accept]), np.asarray(slots),
                        np.asarray(wts), c.positions(2 * W)[slots]))
    assert np.any(out[0][0] != R0)
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)
