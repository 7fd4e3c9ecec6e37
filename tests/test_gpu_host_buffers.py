"""The host-buffer entry points either side of their staging: results, inputs
and positions travel through pinned host memory up to 4 MB and array by array
beyond.  Every output must be the same bit for bit, whatever the route.

64 electrons: a row's results are 3.2 kB, so 7 rows (staged), 1271 (just
under 4 MB), 1400 (beyond) and 1400 with energies alone (staged again).
"""
import ctypes as C

import numpy as np
import pytest

from qmcbeaver_amd import Context, lib, synth
from qmcbeaver_amd._abi import ResultArrays

pytestmark = pytest.mark.gpu

W = 1400


@pytest.fixture(scope="module")
def case():
    s = synth.make_system(1)
    R = synth.initial_walkers(s, W, 5)
    with Context(s.pack(), precision="fp64", max_walkers=W) as ctx:
        yield ctx, R


def chunks(ctx, R, size, which=-1):
    parts = [ctx.evaluate(range(a, min(a + size, W)), R[a:a + size], which)
             for a in range(0, W, size)]
    return {f: np.concatenate([p.a[f] for p in parts]) for f in ResultArrays.FIELDS}


@pytest.mark.parametrize("which", [-1, 63])
def test_batches_agree(case, which):
    ctx, R = case
    ctx.evaluate(range(W), R)
    X = R.copy()
    if which >= 0:
        X[:, which] += 0.1
    whole = chunks(ctx, X, W, which)
    for size in (7, 1271):
        got = chunks(ctx, X, size, which)
        for f in ResultArrays.FIELDS:
            assert np.array_equal(got[f], whole[f], equal_nan=True), (size, f)
    # energies alone: a copy that ends before the per-electron arrays
    res = ResultArrays(W, X.shape[1])
    none = C.c_void_p(None)
    for f in ("grad_lnpsi", "mod_drift"):
        setattr(res.struct, f, C.cast(none, C.POINTER(C.c_double)))
    ids = np.arange(W, dtype=np.int32)
    X = np.ascontiguousarray(X)
    st = lib().qmcb_evaluate(ctx._h, W, ids.ctypes.data_as(C.POINTER(C.c_int32)),
                             X.ctypes.data_as(C.POINTER(C.c_double)), which, C.byref(res.struct))
    assert st == 0
    for f in ResultArrays.FIELDS:
        if f not in ("grad_lnpsi", "mod_drift"):
            assert np.array_equal(res.a[f], whole[f], equal_nan=True), f


@pytest.mark.parametrize("num", [1, 9, W])
def test_staged_rows(case, num):
    ctx, R = case
    ctx.evaluate(range(W), R)
    rng = np.random.default_rng(num)
    ids = rng.permutation(W)[:num]
    X = R[ids].copy()
    X[:, 3] += rng.normal(scale=0.1, size=(num, 3))
    ctx.evaluate(ids, X, 3)
    order = rng.permutation(num)[:(num + 1) // 2]
    mask = rng.integers(0, 2, size=len(order)).astype(bool)
    ctx.accept(ids[order], mask)
    want = R.copy()
    want[ids[order[mask]]] = X[order[mask]]
    assert np.array_equal(ctx.positions(W), want)
    assert np.array_equal(ctx.positions(5), want[:5])
