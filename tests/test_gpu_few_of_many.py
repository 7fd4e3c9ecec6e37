"""Calls for few walkers of a context that holds many: the sums and samples of a
VMC call are those of a context of just these walkers, either side of the size
at which the four sums are moved as one block (128 KB of slots between)."""
import numpy as np
import pytest

from qmcbeaver_amd import Context, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [50, 16384 + 50, 16384 + 96, 60000])
def test_sums_of_few_walkers(capacity):
    s = synth.make_system(0)
    W = 50
    R0, ids = synth.initial_walkers(s, W, 3), np.arange(W)
    out = []
    for cap in (W, capacity):
        print("case few of many", cap, flush=True)
        with Context(s.pack(), precision="fp64", max_walkers=cap, seed=4) as c:
            c.evaluate(ids, R0)
            c.vmc_steps(W, 0, 10, 0.1)
            st = c.vmc_steps(W, 10, 31, 0.1)
            out.append((np.array([st.sum_e_local, st.sum_e_local_sq, st.sum_accept,
                                  st.sum_prop_e_local]), c.sample_series(), c.positions(W)))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
