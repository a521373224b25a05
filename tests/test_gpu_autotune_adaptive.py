"""The autotuner against the adaptive default schedule: it is the start that a
candidate has to beat, and it stays where none does."""
import numpy as np
import pytest

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd import problems

pytestmark = pytest.mark.gpu

# The medians below are of the same products; before the start was timed as it
# runs they differed by 1.6 (left by the tuner) and 4 (reported as the default).
SLACK = 1.25


def _median_ms(ops, n=11):
    v = []
    for _ in range(n):
        out, st = L.rap(*ops)
        out.free()
        v.append(st["ms_total"])
    return float(np.median(v))


def test_tuning_leaves_no_slower_products():
    """A lognormal operator, whose products the default schedule forwards
    unmerged (no candidate schedule does)."""
    L.set_tuning(None)
    p = problems.irregular_sa(10_000)
    ops = [L.DeviceCSR.upload(p[k]) for k in "RAP"]
    before = _median_ms(ops)
    try:
        default = L.get_tuning()
        best, ms_best, ms_default = L.autotune(*ops, reps=1)
        after = _median_ms(ops)
        print(f"before {before:.3f}, default {ms_default:.3f}, best {ms_best:.3f}, after {after:.3f} ms")
        assert best == default == L.get_tuning()
        assert ms_best <= ms_default < SLACK * before
        assert after < SLACK * before
    finally:
        L.set_tuning(None)


def test_a_faster_schedule_is_installed():
    """A schedule that was set is the start as it stands, and one that the
    tuner finds faster is used as it is afterwards."""
    p = problems.poisson3d_sa(64)
    ops = [L.DeviceCSR.upload(p[k]) for k in "RAP"]
    try:
        L.set_tuning({"h1_shift": -1, "h2_div": 1, "u1": 2})  # tables of eight times the slots needed
        slow = _median_ms(ops)
        best, ms_best, ms_default = L.autotune(*ops, reps=2)
        print(f"start {slow:.3f} ({ms_default:.3f}), best {ms_best:.3f}: {best}")
        assert L.get_tuning() == best and ms_best < ms_default < SLACK * slow
    finally:
        L.set_tuning(None)


def test_batch_reports_its_runs():
    p = problems.irregular_sa(3_000)
    ops = [L.DeviceCSR.upload(p[k]) for k in "RAP"]
    L.set_tuning(None)
    b = L.Batch(*([m] for m in ops), graph=True)
    try:
        before = float(np.median([b.run() for _ in range(11)]))
        best, ms_best, ms_default = b.autotune(reps=1)
        after = float(np.median([b.run() for _ in range(11)]))
        print(f"before {before:.3f}, default {ms_default:.3f}, best {ms_best:.3f}, after {after:.3f} ms: {best}")
        assert best == L.get_tuning()
        assert ms_best <= ms_default < SLACK * before and after < SLACK * before
    finally:
        b.free()
        L.set_tuning(None)
