"""Products that are forwarded unmerged when there is memory for whole dense
rows, with less: the library's pool limited to less than those rows take
(SP3MM_POOL_LIMIT, read when the device is initialised, so in a child)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import oracle as O
from sp3mm4amg_amd.csr import CSR

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
import numpy as np
from sp3mm4amg_amd import lib as L
from sp3mm4amg_amd.csr import CSR
z = np.load(sys.argv[1])
ops = [CSR(*z[k + "_shape"], z[k + "_irp"], z[k + "_ja"], z[k + "_vals"]) for k in "RAP"]
got, st = L.rap_host(*ops)
assert L.last_error() == "", L.last_error()
np.savez(sys.argv[2], irp=got.irp, ja=got.ja, vals=got.vals, ms=st["ms_total"])
"""


def _random(rng, m, n, k):
    ja = np.sort(np.stack([rng.choice(n, k, replace=False) for _ in range(m)]), axis=1)
    return CSR(m, n, np.arange(m + 1) * k, ja.ravel(), rng.uniform(0.5, 1.5, m * k))


def test_unmerged_rows_that_do_not_fit(tmp_path):
    # 1,900 dense rows of 17,024 columns: 388 MB; the result is about 125 MB
    rng = np.random.default_rng(8)
    ops = dict(R=_random(rng, 1900, 20_000, 300), A=_random(rng, 20_000, 20_000, 12), P=_random(rng, 20_000, 17_000, 2))
    want = O.sp3mm_merged(*ops.values())
    np.savez(tmp_path / "ops.npz", **{k + "_" + f: v for k, m in ops.items() for f, v in
                                      dict(shape=[m.M, m.N], irp=m.irp, ja=m.ja, vals=m.vals).items()})
    for limit in (0, 300 << 20):
        env = dict(os.environ, PYTHONPATH=ROOT, SP3MM_POOL_LIMIT=str(limit), SP3MM_DENSE_BLOCKS="32")
        r = subprocess.run([sys.executable, "-c", CHILD, str(tmp_path / "ops.npz"), str(tmp_path / "out.npz")], env=env,
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-800:]
        got = np.load(tmp_path / "out.npz")
        print(f"limit {limit >> 20} MB: {float(got['ms']):.2f} ms", flush=True)
        assert np.array_equal(got["irp"], want.irp) and np.array_equal(got["ja"], want.ja)
        # positive terms: at most some thousand additions in any order
        assert np.max(np.abs(got["vals"] - want.vals) / want.vals) < 1e-12
