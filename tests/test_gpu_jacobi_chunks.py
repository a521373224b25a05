"""Many-sweep Jacobi calls that take more than one launch, with the most
workgroups a launch has: the bits of the same sweeps issued one call at a
time.  (That no launch is left with one sweep is checked in
test_jacobi_plan.py: a result cannot show it reliably.)"""
import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from test_gpu_jacobi_grid import _dominant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,per_row,sweeps", [(2048, 520, 65), (2048, 300, 129), (1999, 260, 66), (600, 9, 193)])
def test_sweeps_equal_single_sweeps(m, per_row, sweeps):
    rng = np.random.default_rng(sweeps)
    dA = L.DeviceCSR.upload(_dominant(m, np.full(m, per_row), m))
    b, x = rng.standard_normal(m), rng.standard_normal(m)
    db, dw = L.DeviceArray.from_numpy(b), L.DeviceArray(m)
    got = []
    for calls, n in ((1, sweeps), (sweeps, 1)):
        dx = L.DeviceArray.from_numpy(x)
        for _ in range(calls):
            L.jacobi(dA, db, dx, dw, 0.6, n)
        got.append(dx.numpy())
    assert np.array_equal(*got)


@pytest.mark.parametrize("m,per_row,sweeps", [(2048, 520, 65), (513, 300, 4), (1200, 40, 50)])
def test_sweeps_whose_polls_give_up(m, per_row, sweeps, monkeypatch):
    # no loads allowed: every workgroup gives up at its first poll that is not
    # answered at once, and the last one to end runs the sweeps alone
    rng = np.random.default_rng(sweeps)
    dA = L.DeviceCSR.upload(_dominant(m, np.full(m, per_row), m))
    b, x = rng.standard_normal(m), rng.standard_normal(m)
    db, dw = L.DeviceArray.from_numpy(b), L.DeviceArray(m)
    got = []
    for spins in ("0", None):
        if spins:
            monkeypatch.setenv("SP3MM_GRID_SPINS", spins)
        else:
            monkeypatch.delenv("SP3MM_GRID_SPINS")
        dx = L.DeviceArray.from_numpy(x)
        L.jacobi(dA, db, dx, dw, 0.6, sweeps)
        L.sync()
        got.append(dx.numpy())
    assert np.array_equal(*got)
