"""Which forwards are launched in pieces, and in which (no GPU needed):
tests/fwd_pieces_check.cpp on the rule of simple-vsa_amd/csrc/fwd_pieces.h.  The
sizes that test_gpu_fwd_pieces.py runs do split, their neighbours below each
line do not; and what the rule takes for resident is what the compiler's
registers and LDS allow."""

import os
import re
import shutil
import subprocess

import pytest

from test_kernel_resources import HIPCC, _remarks

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("pieces") / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror",
                    "-I" + os.path.join(os.path.dirname(HERE), "simple-vsa_amd", "csrc"),
                    os.path.join(HERE, "fwd_pieces_check.cpp"), "-o", exe], check=True)

    def run(*args):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True)
        return [int(x) for x in out.stdout.split()]
    return run


# head dim, workgroups a CU holds, key blocks, topk, the caller's block volume
GPU_CASES = [(128, 4, 384, 48, 64), (64, 8, 1280, 160, 64), (128, 4, 400, 50, 33)]


@pytest.mark.parametrize("d,per_cu,kb,tk,be", GPU_CASES)
@pytest.mark.parametrize("pieces,off", [(10, -1), (10, 0), (10, 1), (11, -3), (12, 5)])
def test_the_gpu_tests_sizes_split(check, d, per_cu, kb, tk, be, pieces, off):
    held = CUS * per_cu
    tiles = 4 * (pieces * held // 4 + off)
    got = check(d, 64, be, tiles, 64 * kb, tk, 2, CUS)
    assert len(got) == (tiles + 7) // 8 * 8 // held >= 10
    assert got[:-1] == [held] * (len(got) - 1) and held <= got[-1] < 2 * held
    assert sum(got) == (tiles + 7) // 8 * 8
    # what they are compared with is one launch
    assert len(check(d, 64, be, 4 * held, 64 * kb, tk, 2, CUS)) == 1


@pytest.mark.parametrize("d,per_cu,kb,tk", [(128, 4, 384, 48), (64, 8, 1280, 160)])
def test_one_launch_below_each_line(check, d, per_cu, kb, tk):
    tiles = 10 * CUS * per_cu
    full = (d, 64, 64, tiles, 64 * kb, tk, 2, CUS)
    assert len(check(*full)) == 10

    def changed(i, value):
        return len(check(*full[:i], value, *full[i + 1:]))
    assert changed(1, 128) == 1                  # block volume
    assert changed(2, 32) == 1                   # the second 32 rows do not exist
    assert changed(3, tiles - 8) == 1            # workgroups
    assert changed(4, 64 * (kb - 1)) == 1        # K / V against the L2
    assert changed(5, tk - 1) == 1               # route length
    assert len(check(256, 64, 64, tiles, 64 * kb, tk, 2, CUS)) == 1


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_resident_workgroups_are_what_the_compiler_gives(check, tmp_path):
    found = {}
    for part in _remarks("fine_fwd", str(tmp_path)).split("Function Name: ")[1:]:
        m = re.match(r"\S*sparse_fwd_kernelI(?:DF16b|DF16_)Li(64|128)ELi64E", part)
        if m:
            waves = int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", part).group(1))
            lds = int(re.search(r"LDS Size \[bytes/block\]: (\d+)", part).group(1))
            found.setdefault(int(m.group(1)), set()).add(min(4 * waves // 2, 160 * 1024 // lds))
    assert found == {d: set(check(d)) for d in (64, 128)}
