"""Small direct products whose rows all fit one bin (decided by one launch, the
offsets and the gather by one or two): row counts around the steps of both, and
products that the test sends to the binning after all."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


def _fixed(rng, m, n, length, empty=(), long=()):
    """Rows of `length` entries, but none in rows `empty` and 40 in rows `long`."""
    lens = np.full(m, length)
    lens[list(empty)] = 0
    lens[list(long)] = 40
    rp = np.concatenate(([0], np.cumsum(lens)))
    step = n // 64
    ja = np.arange(rp[-1]) - np.repeat(rp[:-1], lens)
    ja = ja * step + np.repeat(rng.integers(0, step, m), lens)
    return CSR(m, n, rp, ja, rng.uniform(-1.0, 1.0, rp[-1]))


@pytest.mark.parametrize("kind", ["uniform", "empty", "long"])
@pytest.mark.parametrize("la,lp", [(5, 2), (40, 3)])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 4095, 4096, 4097, 6144, 20000])
def test_one_bin(m, la, lp, kind):
    rng = np.random.default_rng(m + la)
    empty = {"empty": {0, m // 2, m - 1}}.get(kind, ())
    R = _fixed(rng, m, 640, 4, empty, (m // 3,) if kind == "long" else ())
    A = _fixed(rng, 640, 1280, la)
    P = _fixed(rng, 1280, 960, lp)
    print(f"m {m} {kind} la {la}", flush=True)
    want = O.sp3mm_pair(R, A, P)
    bound = O.error_bound(R, A, P, want)
    for _ in range(2):
        got, _ = L.rap_host(R, A, P, path=L.DIRECT)
        got.check()
        assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
        assert np.all(np.abs(got.vals - want.vals) <= bound)


@pytest.mark.parametrize("m", [524288, 524289, 700001])
def test_rows_around_the_joint_limit(m):
    """R selects one row of A per row, so the product is A*P's rows repeated."""
    rng = np.random.default_rng(3)
    sel = rng.integers(0, 640, m)
    R = CSR(m, 640, np.arange(m + 1), sel, np.ones(m))
    A, P = _fixed(rng, 640, 1280, 5), _fixed(rng, 1280, 960, 2)
    one = CSR(640, 640, np.arange(641), np.arange(640), np.ones(640))
    rows = O.sp3mm_pair(one, A, P)
    bound = O.error_bound(one, A, P, rows)
    got, _ = L.rap_host(R, A, P, path=L.DIRECT)
    lens = np.diff(rows.irp)[sel]
    assert np.array_equal(np.diff(got.irp), lens)
    at = np.repeat(rows.irp[sel], lens) + np.arange(lens.sum()) - np.repeat(got.irp[:-1], lens)
    assert np.array_equal(got.ja, rows.ja[at])
    assert np.all(np.abs(got.vals - rows.vals[at]) <= np.asarray(bound)[at])
