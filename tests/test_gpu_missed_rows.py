"""Adapted products with a few rows that the sampled tables do not hold: such a
row runs in tables of its bound, and on the long-row kernels only if it fills
those as well.  st["guarded_entries"] counts the rows on the long-row
kernels."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR
from test_gpu_adaptive import _check, _clustered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("nout,per_row,outliers,left", [
    (8, 1, 37, 0),        # 144 stage-1 keys fill the sampled table, not one of 256
    (8, 1, 1, 0),
    (4096, 1, 37, 0),     # 144 output columns, too
    (4096, 3, 37, 37),    # 432 output columns fill tables of 256 slots
])
def test_one_off_product(nout, per_row, outliers, left, f32):
    L.set_tuning(None)
    rows = np.random.default_rng(3).choice(60_000, outliers, replace=False)
    R, A, P = _clustered(60_000, rows, nout=nout)
    if per_row > 1:  # different columns for different rows
        n = P.M
        ja = (np.arange(n)[:, None] * per_row + np.arange(per_row)).ravel()
        P = CSR(n, n * per_row, np.arange(n + 1) * per_row, ja, np.repeat(P.vals, per_row))
    ops = [R, A, P]
    if f32:
        ops = [m.with_vals(m.vals.astype(np.float32).astype(np.float64)) for m in ops]
    d = [L.DeviceCSR.upload(m, vtype=L.F32 if f32 else L.F64) for m in ops]
    out, st = L.rap(*d, precision=L.MIXED64 if f32 else L.FP64)
    _check(out.download(), O.sp3mm_merged(*ops))
    assert st["guarded_entries"] == left


def _sampled_rows(m):
    """The rows of R that the library samples: one per 64th, at a pseudo-random place in it."""
    u = (1 << 64) - 1
    rows = []
    for p in range(64):
        z = 0x9E3779B97F4A7C15 * (p + 2) & u
        z = (z ^ z >> 30) * 0xBF58476D1CE4E5B9 & u
        z = (z ^ z >> 27) * 0x94D049BB133111EB & u
        lo, hi = p * m // 64, (p + 1) * m // 64
        rows.append(min(lo + ((z >> 32 | 1) * max(1, hi - lo) >> 32), m - 1))
    return rows


@pytest.mark.parametrize("graph", [None, False, True])
def test_every_row_but_the_sampled_ones(graph):
    L.set_tuning(None)
    m = 60_000
    ops = _clustered(m, np.setdiff1d(np.arange(m), _sampled_rows(m)))
    want = O.sp3mm_merged(*ops)
    d = [L.DeviceCSR.upload(x) for x in ops]
    if graph is None:
        out, st = L.rap(*d)
        print(f"{st['ms_total']:.3f} ms, {st['guarded_entries']} rows on the long-row kernels")
        _check(out.download(), want)
        assert st["guarded_entries"] == 0
        return
    b = L.Batch(*([x] for x in d), graph=graph)
    try:
        for _ in range(2):
            print(f"{b.run(graph=graph):.3f} ms")
            _check(b.result(0).download(), want)
    finally:
        b.free()


def test_rows_of_several_bins():
    """Short rows (a bound of 24) beside the clustered ones: the missed rows of
    both bins run in the larger bin's tables."""
    L.set_tuning(None)
    rng = np.random.default_rng(4)
    rows = rng.choice(60_000, 25, replace=False)
    R, A, P = _clustered(60_000, rows)
    short = rng.random(60_000) < 0.4
    short[rows] = False
    keep = ~np.repeat(short, 12) | (np.arange(R.ja.size) % 12 < 2)
    irp = np.concatenate(([0], np.cumsum(np.where(short, 2, 12))))
    ops = (CSR(R.M, R.N, irp, R.ja[keep], R.vals[keep]), A, P)
    got, st = L.rap_host(*ops)
    _check(got, O.sp3mm_merged(*ops))
    assert st["guarded_entries"] == 0


@pytest.mark.parametrize("graph", [False, True])
def test_batch_replays(graph):
    """A batch whose sample missed rows is built under the schedule's own
    tables: runs give the product, and go on after a repack with new values."""
    L.set_tuning(None)
    ops = _clustered(60_000, np.random.default_rng(6).choice(60_000, 9, replace=False))
    d = [L.DeviceCSR.upload(m) for m in ops]
    b = L.Batch(*([m] for m in d), graph=graph)
    try:
        for k in range(3):
            new = [m.with_vals(m.vals * (1.0 + 0.25 * k)) for m in ops]
            e = [L.DeviceCSR.upload(m) for m in new]
            b.repack(*([m] for m in e))
            b.run(graph=graph)
            _check(b.result(0).download(), O.sp3mm_merged(*new))
    finally:
        b.free()
