"""Replays of a hierarchy on its fixed pattern: values straight into the output
(several bins, long rows in LDS windows), and the full replay that plans with
retried rows keep.  Each replay against a hierarchy built call by call from the
same values."""
import ctypes as C

import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tuning", [None, {"h1_shift": 2, "h2_div": 8}])
@pytest.mark.parametrize("dims,levels", [((5, 4, 3), 1), ((17, 13, 11), 2), ((36, 33, 31), 3)])
def test_replays_match_fresh_builds(dims, levels, tuning):
    L.init(0)
    L.set_tuning(tuning)
    try:
        A = problems.poisson_operator(dims)
        aggs = []
        d = dims
        for _ in range(levels):
            agg, d = problems.structured_aggregation(d, (2, 2, 2))
            aggs.append((agg, int(np.prod(d))))
        dA = L.DeviceCSR.upload(A)
        H = L.Hierarchy(dA, aggs, graph=True)
        rng = np.random.default_rng(5)
        for rep in range(3):
            vals = np.ascontiguousarray(A.vals * (1.0 + 0.2 * rng.random(A.vals.size)))
            print(f"{dims} tuning {tuning} replay {rep}", flush=True)
            assert L.lib().sp3mm_copy_to_device(dA.d.val, vals.ctypes.data, vals.nbytes) == 0
            H.update(graph=rep != 1)
            fresh, coarse = L.hierarchy_device(dA, aggs)
            built = [lev[1] for lev in fresh[1:]] + [coarse]
            for lvl in range(levels):
                got, want = H.level(lvl)[2].download(), built[lvl].download()
                got.check()
                assert np.array_equal(got.irp, want.irp) and np.array_equal(got.ja, want.ja)
                assert np.max(np.abs(got.vals - want.vals)) <= 1e-12 * np.max(np.abs(want.vals))
            for dR, _, dP in fresh:
                dR.free()
                dP.free()
            for m in built:
                m.free()
        H.free()
        dA.free()
    finally:
        L.set_tuning(None)


@pytest.mark.parametrize("dims", [(4, 3, 2), (16, 16, 4), (64, 61, 59)])
def test_fingerprint_sees_the_last_row(dims):
    """Patterns of one workgroup's work up to many steps of its loop: a column
    of the last row moved by one is refused, and moved back accepted."""
    L.init(0)
    A = problems.poisson_operator(dims)
    agg, d = problems.structured_aggregation(dims, (2, 2, 2))
    dA = L.DeviceCSR.upload(A)
    H = L.Hierarchy(dA, [(agg, int(np.prod(d)))], graph=True)
    at = int(A.irp[-2])
    addr = C.cast(dA.d.col, C.c_void_p).value + 4 * at
    for shift, ok in ((1, False), (0, True)):
        col = np.array([A.ja[at] - shift], np.int32)
        assert L.lib().sp3mm_copy_to_device(addr, col.ctypes.data, 4) == 0
        if ok:
            H.update()
        else:
            with pytest.raises(RuntimeError, match="pattern"):
                H.update()
    H.free()
    dA.free()
