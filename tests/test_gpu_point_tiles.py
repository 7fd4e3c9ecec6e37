"""A wave of the orbital contraction takes one or two point tiles by the operand
type, orbitals and rows of a launch.  Either side of each rule a walker's
evaluate has the bits it has in a small batch (one tile a wave)."""
import numpy as np
import pytest

from qmcbeaver_amd import Context
from tests.test_gpu_walk import system, walkers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,rows", [
    (30, "fp64", (16300, 17000, 21000)), (40, "fp64", (17000,)),
    (30, "fp32", (17000, 21000)), (40, "fp32", (17000, 21000)), (70, "fp32", (17000, 34000)),
    (30, "bf16store", (17000, 21000)), (40, "bf16", (17000, 52000)), (70, "bf16", (17000, 52000)),
])
def test_point_tiles_give_the_same_bits(n, precision, rows):
    p = system(n, n)
    few = 70
    out = []
    for P in (few * n,) + rows:
        W = -(-P // n)
        print("case point tiles", n, precision, P, flush=True)
        R = np.tile(walkers(p, few, 3), (-(-W // few), 1, 1))[:W]
        with Context(p, precision=precision, max_walkers=W) as c:
            r = c.evaluate(np.arange(W), R)
            last = np.arange(W - few, W)  # the last tiles too
            out.append([r.a[k][:few] for k in ("log_psi", "e_local", "grad_lnpsi")])
            out.append([r.a[k][last[np.argsort(last % few)]]
                        for k in ("log_psi", "e_local", "grad_lnpsi")])
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)
