"""Results of a batch: none after a run that failed, and each batch's own when
runs of several batches alternate."""
import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd import problems
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu


def _check(got, ops):
    want = O.sp3mm_merged(*ops)
    assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
    assert O.rel_errors(got, want, O.abs_product(*ops)).max() < 1e-12


@pytest.mark.parametrize("graph", [False, True])
def test_no_result_of_a_failed_run(graph):
    """A run whose product outgrew the batch: its offsets may end beyond the
    output, so nothing is copied out by them until a run has succeeded."""
    L.set_tuning(None)
    p = problems.poisson2d_sa(64)
    R, A, P = ops = [p[k] for k in "RAP"]
    ja = A.ja.copy()
    assert ja[A.irp[66] - 1] == 129
    ja[A.irp[66] - 1] = 4000  # the product gains entries
    d = [L.DeviceCSR.upload(m) for m in ops]
    moved = L.DeviceCSR.upload(CSR(A.M, A.N, A.irp, ja, A.vals))
    b = L.Batch(*([m] for m in d), graph=graph)
    try:
        for _ in range(2):
            b.run(graph=graph)
            _check(b.result(0).download(), ops)
            b.repack(As=[moved])
            with pytest.raises(RuntimeError, match="replayed product"):
                b.run(graph=graph)
            with pytest.raises(RuntimeError, match="there are no results"):
                b.result(0)
            b.repack(As=[d[1]])
    finally:
        b.free()


@pytest.mark.parametrize("counts", [(3, 2), (255, 1), (256, 254)])
def test_alternating_batches(counts):
    """Up to 255 products' entry ranges pass through memory that all batches
    share, more through a batch's own."""
    L.set_tuning(None)
    rng = np.random.default_rng(2)
    kinds = [[problems.poisson2d_sa(n)[k] for k in "RAP"] for n in (8, 11, 16)]
    probs = [[kinds[i] for i in rng.integers(0, 3, n)] for n in counts]
    dev = {id(k): [L.DeviceCSR.upload(m) for m in k] for k in kinds}
    bs = [L.Batch(*([dev[id(k)][j] for k in ps] for j in range(3)), graph=i == 0) for i, ps in enumerate(probs)]
    try:
        for order in ((0, 1), (1, 0), (0, 0)):
            for i in order:
                bs[i].run(graph=i == 0)
            for i in (0, 1):
                for k in sorted({0, len(probs[i]) // 2, len(probs[i]) - 1}):
                    _check(bs[i].result(k).download(), probs[i][k])
    finally:
        for b in bs:
            b.free()
