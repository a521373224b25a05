"""The wait behind short work: sp3mm_sync against a blocking copy of a few bytes
out of pageable memory, which is how it once read the consumers' state."""
import time

import numpy as np
import pytest
import torch

from sp3mm4amg_amd import lib as L

pytestmark = pytest.mark.gpu


def _median_us(f, n=301):
    for _ in range(20):
        f()
    v = []
    for _ in range(n):
        t0 = time.perf_counter()
        f()
        v.append(time.perf_counter() - t0)
    return float(np.median(v)) * 1e6


def test_waiting_costs_less_than_a_copy():
    x = L.DeviceArray.from_numpy(np.ones(64))
    assert L.dot(x, x) == 64.0  # the consumers' state exists from here on
    src = torch.zeros(2, dtype=torch.float64, device="cuda")
    dst = torch.zeros(2, dtype=torch.float64)
    copy = sync = 1e9
    for _ in range(3):
        copy = min(copy, _median_us(lambda: dst.copy_(src)))
        sync = min(sync, _median_us(L.sync))
    print(f"copy {copy:.1f} us, sync {sync:.1f} us")
    assert sync < copy
