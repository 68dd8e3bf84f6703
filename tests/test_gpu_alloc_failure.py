"""Device memory of a handle: a first solve one of whose allocations fails reports
that, and the solve that follows works and leaves the handle with the memory of
one that never failed; and the first solves of a handle do not depend on what its
memory held before."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build(name, tmp_path):
    exe, here = str(tmp_path / name), os.path.join(ROOT, "opm-porsol_amd")
    cmd = ["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", name + ".cpp"), "-o", exe, "-L", here, "-lmhs", f"-Wl,-rpath,{here}", "-ldl"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    return exe


def _run(*cmd):
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    return [tuple(map(int, l.split())) for l in res.stdout.splitlines()], res.stderr


def test_failed_first_solves_leave_nothing_behind(pkg, tmp_path):
    lines, err = _run(_build("alloc_failure_check", tmp_path))
    made, clean = lines[0]
    assert made > 10 and clean > 0 and len(lines) == made + 1
    assert [l for l in lines[1:] if l[1] != clean] == [], err


def test_first_solves_on_used_memory(pkg, tmp_path):
    exe = _build("used_memory_check", tmp_path)
    (clean, err0), (used, err) = _run(exe, "0"), _run(exe, "1")
    assert len(clean) == len(used) == 16, err0 + err
    # the same few steps whichever operator the tuner chose
    steps = max(l[1] for l in clean)
    assert all(l[0] == 0 and l[2] == 1 for l in clean) and steps < 20, clean
    assert all(l[0] == 0 and l[2] == 1 and l[1] <= steps for l in used), (used, err)
