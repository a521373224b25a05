"""One-pass SpGEMM whose short rows fold into the bin of the long ones: counts
around the folding limit, and a product with no rows."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


def _rows(rng, lens, n):
    ja = [np.sort(rng.choice(n, k, replace=False)) for k in lens]
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
    ja = np.concatenate(ja) if len(ja) and rp[-1] else np.zeros(0, np.int64)
    return CSR(len(lens), n, rp, ja, rng.uniform(0.5, 1.5, ja.size))


@pytest.mark.parametrize("short,long", [(0, 0), (0, 700), (1, 3000), (1023, 3000), (1024, 3000), (1025, 3000), (1024, 0)])
def test_folded_bins(short, long):
    rng = np.random.default_rng(short)
    lens = np.concatenate((np.full(short, 4), np.full(long, 40))).astype(np.int64)
    rng.shuffle(lens)
    A = _rows(rng, lens, 500)
    B = _rows(rng, np.full(500, 12), 900)
    dA, dB = L.DeviceCSR.upload(A), L.DeviceCSR.upload(B)
    out, _ = L.spgemm(dA, dB)
    got = out.download()
    one = CSR(900, 900, np.arange(901), np.arange(900), np.ones(900))
    want = O.sp3mm_pair(A, B, one) if short + long else CSR(0, 900, np.zeros(1, np.int64), np.zeros(0, np.int64), np.zeros(0))
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    if short + long:
        assert np.all(np.abs(got.vals - want.vals) <= O.error_bound(A, B, one, want))
    for m in (dA, dB, out):
        m.free()
