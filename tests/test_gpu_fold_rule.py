"""Direct products whose short rows fold into the bin of longer ones: counts and
bounds on both sides of the rule, and a product that the allocation-free entry
point's scratch holds only if its short rows keep slots of their own size."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu

N, NC = 20_000, 6_000


def _operands(short, short_len, long, long_len):
    """R of `short` rows of short_len entries among `long` rows of long_len,
    local in a band; A of 7 entries per row; P one entry per row."""
    rng = np.random.default_rng(short + long)
    lens = np.concatenate((np.full(short, short_len), np.full(long, long_len)))
    rng.shuffle(lens)
    first = np.linspace(0, N - 1500, lens.size).astype(np.int64)
    ja = np.concatenate([f + np.sort(rng.choice(1500, k, replace=False)) for f, k in zip(first, lens)])
    R = CSR(lens.size, N, np.concatenate(([0], np.cumsum(lens))), ja, rng.uniform(0.5, 1.5, ja.size))
    cols = np.arange(N)[:, None] + np.arange(-3, 4)
    ok = (cols >= 0) & (cols < N)
    A = CSR(N, N, np.concatenate(([0], np.cumsum(ok.sum(1)))), cols[ok], rng.uniform(0.5, 1.5, int(ok.sum())))
    P = CSR(N, NC, np.arange(N + 1), np.arange(N) * NC // N, rng.uniform(0.5, 1.5, N))
    return R, A, P


def _check(got, ops):
    want = O.sp3mm_merged(*ops)
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    # positive terms: some thousand additions in any order
    assert np.max(np.abs(got.vals - want.vals) / want.vals) < 1e-12


@pytest.mark.parametrize("short,short_len,long,long_len", [
    (1024, 1, 40, 500), (1025, 1, 40, 500), (6000, 1, 50, 500),        # 64 under 4096
    (8192, 8, 900, 30), (8193, 8, 900, 30), (1025, 8, 9000, 16),       # 64 under 256, under 128
    (3000, 30, 2000, 120),                                             # 256 under 1024
])
def test_products_around_the_rule(short, short_len, long, long_len):
    L.set_tuning(None)
    ops = _operands(short, short_len, long, long_len)
    _check(L.rap_host(*ops)[0], ops)


def test_allocation_free_product_keeps_small_slots():
    """8,000 rows of 7 products and 3,100 of 4,900: in slots of the long rows'
    size they need more than the 256 MB of fixed scratch."""
    L.set_tuning(None)
    ops = _operands(8000, 1, 3100, 700)
    d = [L.DeviceCSR.upload(m) for m in ops]
    ref, _ = L.rap(*d)
    want = ref.download()
    rp, col = L.DeviceArray(ops[0].M + 1, np.int64), L.DeviceArray(want.nnz, np.int32)
    val = L.DeviceArray(want.nnz)
    nnz, _ = L.rap_noalloc(*d, rp, col, val, want.nnz)
    _check(CSR(want.M, want.N, rp.numpy(), col.numpy().astype(np.int64), val.numpy()), ops)
    assert nnz == want.nnz
