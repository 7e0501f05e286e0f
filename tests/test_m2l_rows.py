"""LDS accesses of the target-stationary M2L (csrc/hip/rcr_ts_rows.h) on the CPU:
ts_rows_check.cpp runs the 64 lanes of a wavefront over two batches of every
order from 1 to 16, with targets met by one and by many vectors of a batch, and
checks each access."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("what", ["range", "order"])
def test_accesses(what, tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas",
                    "-I" + os.path.join(ROOT, "fmbem_gpu_c_amd", "csrc", "hip"),
                    os.path.join(ROOT, "tests", "ts_rows_check.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe, what], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout
