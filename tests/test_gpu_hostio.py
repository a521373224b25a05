"""Large host arrays in and out (pinned staging filled by host threads): sizes
around the staging slots and the size rule, both index bases and value types,
and the same refusals as small arrays."""
import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu

SLOT = 1 << 18  # 32-bit columns per staging slot


def _matrix(M, nnz, N=1 << 20, seed=3):
    """nnz entries over M rows, rows of uneven length (some empty)."""
    rng = np.random.default_rng(seed)
    irp = np.sort(rng.integers(0, nnz + 1, M + 1))
    irp[0], irp[-1] = 0, nnz
    lens = np.diff(irp)
    start = rng.integers(0, N - int(lens.max(initial=0)), M)
    ja = np.arange(nnz) - np.repeat(irp[:-1], lens) + np.repeat(start, lens)
    return CSR(M, N, irp, ja, rng.uniform(-1.0, 1.0, nnz))


@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("vtype", [L.F64, L.F32])
@pytest.mark.parametrize("M,nnz", [
    (1, 1 << 18), (1000, SLOT - 1), (1000, SLOT), (999, SLOT + 1), (SLOT - 1, 3 * SLOT), (SLOT, 3 * SLOT + 17),
    (700001, 20 * SLOT + 5), (600000, 0), (100000, 262143),
])
def test_round_trip(M, nnz, vtype, base):
    print(f"M {M} nnz {nnz} vtype {vtype} base {base}", flush=True)
    m = _matrix(M, nnz)
    for _ in range(2):
        d = L.DeviceCSR.upload(m, vtype=vtype, base=base)
        got = d.download(base=base)
        assert np.array_equal(got.irp, m.irp) and np.array_equal(got.ja, m.ja)
        assert np.array_equal(got.vals, m.vals.astype(got.vals.dtype))
        d.free()


@pytest.mark.parametrize("fault", ["row", "rows", "low", "high", "huge", "order"])
def test_refusals(fault):
    m = _matrix(600000, 5 * SLOT)
    irp, ja = m.irp.copy(), m.ja.copy()
    rows = np.flatnonzero(np.diff(irp) > 1)
    want = "not valid sorted CSR"
    if fault in ("row", "rows"):
        at = [590001] if fault == "row" else [590001, 31]
        for r in at:
            irp[r + 1] = irp[r] - 1
        first = min(int(np.flatnonzero(np.diff(irp) < 0)[0]), min(at))
        want = f"decrease at row {first}$"
    elif fault == "low":
        ja[-1] = -1
    elif fault == "high":
        ja[4 * SLOT + 3] = m.N
    elif fault == "huge":
        ja[7] = (1 << 32) + ja[7]
    else:
        e = irp[rows[-1]]
        ja[e + 1] = ja[e]
    with pytest.raises(RuntimeError, match=want):
        L.DeviceCSR.upload(CSR(m.M, m.N, irp, ja, m.vals))
    d = L.DeviceCSR.upload(m)
    assert np.array_equal(d.download().ja, m.ja)
    d.free()
