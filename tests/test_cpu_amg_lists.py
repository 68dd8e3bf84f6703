"""Host-side gather lists of the multigrid set-up: what their 32-bit ends can
hold is checked on the lists themselves (a face between two blocks is in both
blocks' lists, so they are longer than the face matrix), they are the same on
one host thread as on several, and the autotuner times each tail that they
allow once; and the LDS limit of the one-workgroup tail, which every handle
sets on its own device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIP = ["-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include")]
HIP_LIBS = ["-L", os.path.join(ROCM, "lib"), "-lamdhip64", f"-Wl,-rpath,{os.path.join(ROCM, 'lib')}"]
STRENGTHS = [("1", "1", "1"), ("1", "1", "0.1"), ("0.1", "0.1", "1")]   # blocks 2x2x2, 2x2x1, 1x1x2


@pytest.fixture(scope="module")
def lists(pkg, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("amg") / "amg_lists_check")
    here = os.path.join(ROOT, "opm-porsol_amd")
    cmd = ["g++", "-O1", "-std=c++17", "-Wall", "-pthread", *HIP, "-I", os.path.join(here, "csrc"), "-I",
           os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "amg_lists_check.cpp"), "-o", exe, "-L", here,
           "-lmhs", f"-Wl,-rpath,{here}", *HIP_LIBS]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr

    def run(strength, dims, limit=0, element_limit=0, threads=2):
        cmd = [exe, str(threads), *strength, str(limit), str(element_limit), *map(str, dims)]
        res = subprocess.run(cmd, capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stdout + res.stderr
        return dict(line.split(" ", 1) for line in res.stdout.splitlines())

    return run


@pytest.mark.parametrize("strength", STRENGTHS)
@pytest.mark.parametrize("dims", [(12, 11, 9), (8, 8, 8, 5, 4, 7)])
def test_lists_past_the_limit_are_refused(lists, strength, dims):
    ok = lists(strength, dims)
    assert ok["amg"] == ok["element"] == "ok"
    # longer than the face matrix that used to bound them, by less than the ends' extra bit
    assert int(ok["matrix"]) < int(ok["ap"]) <= 2 * int(ok["matrix"])
    assert int(ok["longest"]) <= 2 * int(ok["matrix"])
    n, m = int(ok["longest"]), int(ok["element_list"])
    assert lists(strength, dims, limit=n)["hash"] == ok["hash"]
    assert "too large" in lists(strength, dims, limit=n - 1)["amg"]
    assert lists(strength, dims, element_limit=m)["hash"] == ok["hash"]
    assert "too many entries" in lists(strength, dims, element_limit=m - 1)["element"]


@pytest.mark.parametrize("strength", STRENGTHS)
@pytest.mark.parametrize("dims", [(40, 36, 30), (30, 20, 25, 41, 19, 22)])
def test_one_host_thread_and_several_build_the_same_lists(lists, strength, dims):
    one, many = lists(strength, dims, threads=1), lists(strength, dims, threads=8)
    assert int(one["asked"]) > 0 and int(many["asked"]) > 0   # the program's answer was the one used
    assert one["hash"] == many["hash"]


@pytest.mark.parametrize("dims", [(1, 1, 1), (9, 9, 9), (20, 20, 10), (40, 36, 30), (8, 8, 8, 26, 25, 24)])
def test_autotuner_times_every_tail_once(lists, dims):
    out = lists(STRENGTHS[0], dims)
    for vsize in (4, 8):
        for nrhs in (1, 3):
            levels, last = out[f"tail_{vsize}_{nrhs}"].split("|")
            levels = list(map(int, levels.split()))
            assert levels == sorted(set(levels), reverse=True) and levels[-1] == int(last)


def test_tail_lds_limit_is_set_for_every_handle(pkg, tmp_path):
    exe, here = str(tmp_path / "tail_limit_check"), os.path.join(ROOT, "opm-porsol_amd")
    cmd = ["g++", "-O1", "-std=c++17", *HIP, "-I", os.path.join(here, "csrc"), "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "tail_limit_check.cpp"), "-o", exe, "-L", here, "-lmhs", f"-Wl,-rpath,{here}",
           *HIP_LIBS]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    out = [subprocess.run([exe, *a], capture_output=True, text=True, timeout=60) for a in ([], ["refuse"])]
    assert [o.returncode for o in out] == [0, 0], out
    lines = [[tuple(map(int, l.split())) for l in o.stdout.splitlines()] for o in out]
    # two precisions, one to four right-hand sides, for each of the two handles
    assert lines[0] == [(152 * 1024, 8, 8)] * 2
    # refused: what a launch may take without asking
    assert [l[0] for l in lines[1]] == [64 * 1024] * 2
