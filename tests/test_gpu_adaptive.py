"""Products under the adaptive schedule (no schedule set): table sizes, groups and
hash multipliers come from a sample of R's rows.  Checked against the oracle
where the sample decides wrongly (rows it did not see have more distinct keys
than the sampled tables hold) and on both sides of its size rule."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd import problems
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu

LEN = 12  # entries per row of R and of A: a bound of 144 per row


def _clustered(m, spread_rows, ncol=4096, nout=8):
    """Every row of R selects LEN rows of A of LEN entries each.
    The rows of A that ordinary rows of R select hold the same LEN columns
    (LEN distinct stage-1 keys), those of the rows in `spread_rows` LEN * LEN
    different ones.  P maps every column to column % nout."""
    rng = np.random.default_rng(m)
    spread = np.zeros(m, bool)
    spread[list(spread_rows)] = True
    # 64 clusters of LEN rows of A with common columns, 64 clusters without
    kinds = 64
    acols = np.empty((2 * kinds * LEN, LEN), np.int64)
    for k in range(kinds):
        acols[k * LEN:(k + 1) * LEN] = np.sort(rng.choice(ncol, LEN, replace=False))
        d = rng.choice(ncol, LEN * LEN, replace=False).reshape(LEN, LEN)
        acols[(kinds + k) * LEN:(kinds + k + 1) * LEN] = np.sort(d, axis=1)
    na = acols.shape[0]
    A = CSR(na, ncol, np.arange(na + 1) * LEN, acols.ravel(), rng.uniform(0.5, 1.5, acols.size))
    cl = np.arange(m) % kinds + np.where(spread, kinds, 0)
    rcols = (cl[:, None] * LEN + np.arange(LEN)).ravel()
    R = CSR(m, na, np.arange(m + 1) * LEN, rcols, rng.uniform(0.5, 1.5, rcols.size))
    P = CSR(ncol, nout, np.arange(ncol + 1), np.arange(ncol) % nout, rng.uniform(0.5, 1.5, ncol))
    return R, A, P


def _check(got, want):
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    # positive terms only: any order of at most 144 + 144 additions stays far below 1e-12 relative
    assert np.max(np.abs(got.vals - want.vals) / np.abs(want.vals)) < 1e-12


@pytest.mark.parametrize("m,outliers", [(60_000, 0), (60_000, 37), (60_000, 30_000), (2_000, 5)])
def test_rows_the_sample_missed(m, outliers):
    """60,000 rows are sampled (8.6e6 multiply-adds), 2,000 are not; rows with
    144 distinct keys among rows with 12 fill the sampled tables and are
    redone by the long-row kernels."""
    L.set_tuning(None)
    rows = np.random.default_rng(3).choice(m, outliers, replace=False)
    R, A, P = _clustered(m, rows)
    got, _ = L.rap_host(R, A, P)
    _check(got, O.sp3mm_merged(R, A, P))


@pytest.mark.parametrize("graph", [False, True])
def test_batch_with_a_pattern_of_the_same_sizes(graph):
    """repack() with a pattern of the same sizes whose rows have more distinct
    keys than the tables sampled at creation hold: computed, not refused."""
    L.set_tuning(None)
    m = 300
    R1, A, P = _clustered(m, range(m))   # every row spread
    R0, _, _ = _clustered(m, [])         # no row spread; the same A and P
    full = lambda Q: CSR(Q.M, 4, np.arange(Q.M + 1) * 4, np.tile(np.arange(4), Q.M),
                         np.random.default_rng(1).uniform(0.5, 1.5, 4 * Q.M))
    P = full(P)                          # 4 nonzeros per output row either way
    dev = [L.DeviceCSR.upload(x) for x in (R0, A, P)]
    b = L.Batch([dev[0]], [dev[1]], [dev[2]], graph=graph)
    try:
        b.run(graph=graph)
        _check(b.result(0).download(), O.sp3mm_merged(R0, A, P))
        dR = L.DeviceCSR.upload(R1)
        b.repack(Rs=[dR])
        for _ in range(3):
            b.run(graph=graph)
            _check(b.result(0).download(), O.sp3mm_merged(R1, A, P))
        b.repack(Rs=[dev[0]])
        b.run(graph=graph)
        _check(b.result(0).download(), O.sp3mm_merged(R0, A, P))
    finally:
        b.free()


@pytest.mark.parametrize("n,path", [(57, "7pt"), (64, "7pt"), (33, "27pt"), (40, "27pt")])
def test_both_sides_of_the_size_rule(n, path):
    L.set_tuning(None)
    p = problems.poisson3d_sa(n) if path == "7pt" else problems.stencil27_sa(n, 3)
    R, A, P = p["R"], p["A"], p["P"]
    got, _ = L.rap_host(R, A, P)
    want = O.sp3mm_merged(R, A, P)
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    assert O.rel_errors(got, want, O.abs_product(R, A, P)).max() < 1e-12


def _random(rng, m, n, lens):
    """m x n with the given row lengths, columns uniform, values in [-1, 1)."""
    irp = np.concatenate([[0], np.cumsum(lens)])
    cols = np.concatenate([np.sort(rng.choice(n, int(k), replace=False)) for k in lens])
    return CSR(m, n, irp, cols, rng.uniform(-1.0, 1.0, cols.size))


@pytest.mark.parametrize("ncol,f32", [(30, False), (64, False), (1000, False), (1000, True), (7521, False),
                                      (17696, False), (17697, False)])
def test_unmerged_forwarding(ncol, f32):
    """Unstructured rows of thousands of products (k_scatter_direct): R rows
    around the 512 entries staged at once, empty and 2,000-entry rows of A and
    P, output widths up to the widest the LDS accumulators take and past it."""
    L.set_tuning(None)
    rng = np.random.default_rng(ncol)
    k, j, m = 3000, 21000, 260
    lr = rng.integers(400, 700, m)
    lr[:4] = 511, 512, 513, 1024
    la = rng.integers(0, 50, k)
    la[::500] = 2000
    lp = np.minimum(rng.integers(0, 24, j), ncol)
    lp[::3000] = min(2000, ncol)
    R, A, P = _random(rng, m, k, lr), _random(rng, k, j, la), _random(rng, j, ncol, lp)
    if f32:
        R, A, P = (x.with_vals(x.vals.astype(np.float32).astype(np.float64)) for x in (R, A, P))
        got, st, _ = L.rap_mixed_host(R, A, P, precision=L.MIXED64)
    else:
        got, st = L.rap_host(R, A, P)
    assert st["guarded_entries"] == m  # no row on the hash tables
    want = O.sp3mm_pair(R, A, P)
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    assert np.all(np.abs(got.vals - want.vals) <= O.error_bound(R, A, P, want))
