"""sp3mm_trim gives back the pool's free blocks and the pinned staging of large
host copies, and calls go on as before."""
import numpy as np
import pytest
import torch

from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd import problems

pytestmark = pytest.mark.gpu


def _mapped():
    """Bytes mapped into the process: pinned memory and device blocks among them."""
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) for line in f if line.startswith("VmSize")) << 10


def test_trim_between_copies():
    A = problems.poisson_operator((64, 64, 64))
    L.sync()
    for k in range(3):
        d = L.DeviceCSR.upload(A)  # 31 MB: staged
        got = d.download()
        assert np.array_equal(got.irp, A.irp) and np.array_equal(got.ja, A.ja) and np.array_equal(got.vals, A.vals)
        live = d.nnz * 12
        d.free()
        before, mapped = torch.cuda.mem_get_info()[0], _mapped()
        L.trim()
        freed, unmapped = torch.cuda.mem_get_info()[0] - before, mapped - _mapped()
        print(f"device {freed >> 20} MB given back, {unmapped >> 20} MB unmapped")
        assert freed >= live
        assert unmapped >= freed + (12 << 20)  # and most of the 16 MB
        L.trim()  # nothing left to give
