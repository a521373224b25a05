"""Rows of a transpose put in order: by a bitmap of their columns (long rows of
narrow span) and by comparing pairs (short rows, wide spans)."""
import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [2100, 16384, 16385, 70000])
@pytest.mark.parametrize("n", [1, 47, 48, 49, 64, 65, 1023, 1024, 1025, 2100])
def test_rows_of_every_length(n, span):
    """Column c of A has n entries over rows lo .. lo + span - 1 (both ends taken
    for n > 1), columns with other lengths between them."""
    rng = np.random.default_rng(n + span)
    rows, cols = [], []
    for c in range(24):
        k = n if c % 3 else int(rng.integers(1, 40))
        lo = int(rng.integers(0, 500))
        ids = np.sort(rng.choice(span, k, replace=False))
        if k > 1:
            ids[0], ids[-1] = 0, span - 1
        rows.append(lo + ids)
        cols.append(np.full(k, c))
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    m = span + 500
    vals = rng.uniform(-1.0, 1.0, rows.size)
    A = CSR(m, 24, np.searchsorted(rows, np.arange(m + 1)), cols, vals)
    d = L.DeviceCSR.upload(A)
    got = L.transpose(d).download()
    back = np.lexsort((rows, cols))
    assert np.array_equal(got.irp, np.searchsorted(cols[back], np.arange(25)))
    assert np.array_equal(got.ja, rows[back]) and np.array_equal(got.vals, vals[back])
    d.free()
