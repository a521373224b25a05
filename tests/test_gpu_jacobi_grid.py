"""Many Jacobi sweeps of a medium system in one launch over several workgroups
(k_jacobi_grid): the bits of the same sweeps issued one call at a time (one
sweep is a launch of k_jacobi, which sums a row in the same order)."""
import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


def _dominant(m, lens, seed):
    rng = np.random.default_rng(seed)
    cols = [np.unique(np.append(rng.choice(m, min(int(k), m), replace=False), i)) for i, k in enumerate(lens)]
    irp = np.concatenate([[0], np.cumsum([c.size for c in cols])])
    ja = np.concatenate(cols)
    vals = rng.uniform(-1.0, 1.0, ja.size)
    rows = np.repeat(np.arange(m), np.diff(irp))
    vals[ja == rows] = np.bincount(rows, np.abs(vals), m) + 1.0
    return CSR(m, m, irp, ja, vals)


@pytest.mark.parametrize("m,per_row,sweeps", [(2048, 7, 5), (2047, 27, 64), (700, 100, 65), (513, 300, 4), (512, 300, 50),
                                              (800, 700, 130), (2048, 520, 7)])
def test_sweeps_equal_single_sweeps(m, per_row, sweeps):
    rng = np.random.default_rng(m)
    lens = np.full(m, per_row)
    lens[m // 2] = m  # a full row: more entries than its lanes keep in registers
    A = _dominant(m, lens, per_row)
    dA = L.DeviceCSR.upload(A)
    b, x = rng.standard_normal(m), rng.standard_normal(m)
    db, dx, dw = L.DeviceArray.from_numpy(b), L.DeviceArray.from_numpy(x), L.DeviceArray(m)
    L.jacobi(dA, db, dx, dw, 0.6, sweeps)
    many = dx.numpy()
    dx.free()
    dx = L.DeviceArray.from_numpy(x)
    for _ in range(sweeps):
        L.jacobi(dA, db, dx, dw, 0.6, 1)
    assert np.array_equal(many, dx.numpy())


def test_zero_diagonal_is_reported():
    A = _dominant(600, np.full(600, 40), 1)
    A.vals[(A.ja == A.row_ids()) & (A.ja == 311)] = 0.0
    dA = L.DeviceCSR.upload(A)
    v = [L.DeviceArray.from_numpy(np.ones(600)) for _ in range(3)]
    L.jacobi(dA, *v, 0.6, 10)
    with pytest.raises(RuntimeError, match="zero diagonal"):
        L.sync()
    L.sync()  # reported once
