"""Long rows in LDS windows (k_window_direct): windows whose present entries are
listed, tested one by one, without room for the list, and with a list that
gives way to the second window; rows of A and P around the unrolled steps."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


def _rows(rng, lengths, universe):
    cols = [np.sort(rng.choice(universe, n, replace=False)) for n in lengths]
    rp = np.concatenate(([0], np.cumsum(lengths)))
    ja = np.concatenate(cols) if rp[-1] else np.zeros(0, np.int64)
    return rp, ja, rng.uniform(0.5, 1.5, ja.size)


def _problem(m, span1, present, span2):
    """Rows of R*A over `present` of `span1` columns, five products to a
    column; rows of P of 0 to 17 entries within `span2` columns."""
    rng = np.random.default_rng(span1 + m)
    uni = np.sort(rng.choice(span1, present, replace=False))
    na = 700
    A = CSR(na, span1, *_rows(rng, np.resize([0, 1, 63, 64, 65, 127, 129], na), uni))
    nr = 5 * present * na // int(A.irp[-1])
    R = CSR(m, na, *_rows(rng, np.full(m, min(nr, na)), np.arange(na)))
    P = CSR(span1, span2, *_rows(rng, np.resize([0, 1, 7, 8, 9, 15, 16, 17], span1), np.arange(span2)))
    return R, A, P


@pytest.mark.parametrize("m", [9, 264])
@pytest.mark.parametrize("span1,present,span2", [
    (6000, 2500, 3000),    # listed
    (6000, 5400, 3000),    # nearly full: tested one by one
    (18000, 11000, 1000),  # no room behind the values of the first window
    (12000, 5000, 7500),   # the list gives way to the second window
    (12000, 5000, 6016),   # both fit
])
def test_windows(m, span1, present, span2):
    R, A, P = _problem(m, span1, present, span2)
    print(f"m {m} window {present}/{span1} -> {span2}", flush=True)
    want = O.sp3mm_pair(R, A, P)
    got, st = L.rap_host(R, A, P, path=L.DIRECT)
    assert st["guarded_entries"] > 0 and st["spilled_rows"] == 0
    got.check()
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    assert np.all(np.abs(got.vals - want.vals) <= O.error_bound(R, A, P, want))
