"""Host rules of the many-sweep Jacobi launches (csrc/jacobi_plan.hpp), compiled
and run on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="g++ is missing")


def _run(tmp_path, body):
    src = tmp_path / "plan.cpp"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "jacobi_plan.hpp"\nusing namespace sp3mm;\n'
                   "int main() {\n" + body + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "sp3mm4amg_amd", "csrc"), str(src),
                    "-o", str(tmp_path / "plan")], check=True, capture_output=True, text=True, timeout=120)
    return subprocess.run([str(tmp_path / "plan")], check=True, capture_output=True, text=True, timeout=60).stdout


def test_no_launch_of_one_sweep(tmp_path):
    # a launch of one sweep would overwrite x while other workgroups still read it
    out = _run(tmp_path, "for (int s = 4; s <= 400; s++) { std::printf(\"%d\", s);\n"
                         "for (int k = 0; k < s;) { const int n = jacobi_chunk(s - k); std::printf(\" %d\", n); k += n;\n"
                         "if (n < 1) std::abort(); } std::printf(\"\\n\"); }")
    rows = [[int(v) for v in line.split()] for line in out.splitlines()]
    assert [r[0] for r in rows] == list(range(4, 401))
    for s, *chunks in rows:
        assert sum(chunks) == s and all(2 <= n <= 64 for n in chunks), (s, chunks)


def test_launch_needs_all_its_workgroups_on_the_chip(tmp_path):
    # 64 lanes per row: 8 rows per workgroup; 256 workgroups do not fit 32 CUs of 4
    out = _run(tmp_path, "const int q[][4] = {{2048, 64, 4, 256}, {2048, 64, 4, 64}, {2048, 64, 4, 63}, {2048, 64, 4, 32},"
                         "{513, 64, 1, 64}, {513, 64, 1, 65}, {2048, 1, 4, 1}, {2048, 64, 0, 256}};\n"
                         "for (auto &v : q) std::printf(\"%d %d\\n\", jacobi_groups(v[0], v[1]),"
                         " (int)jacobi_grid_resident(v[0], v[1], v[2], v[3]));")
    got = [tuple(int(v) for v in line.split()) for line in out.splitlines()]
    assert got == [(256, 1), (256, 1), (256, 0), (256, 0), (65, 0), (65, 1), (4, 1), (256, 0)]
