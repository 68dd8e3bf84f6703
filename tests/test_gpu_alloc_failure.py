"""A first solve one of whose device allocations fails reports that, and the solve
that follows works and leaves the handle with the memory of one that never
failed."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failed_first_solves_leave_nothing_behind(pkg, tmp_path):
    exe, here = str(tmp_path / "alloc_failure_check"), os.path.join(ROOT, "opm-porsol_amd")
    cmd = ["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "alloc_failure_check.cpp"), "-o", exe, "-L", here, "-lmhs", f"-Wl,-rpath,{here}",
           "-ldl"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    res = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    lines = [tuple(map(int, l.split())) for l in res.stdout.splitlines()]
    made, clean = lines[0]
    assert made > 10 and clean > 0 and len(lines) == made + 1
    assert [l for l in lines[1:] if l[1] != clean] == [], res.stderr
