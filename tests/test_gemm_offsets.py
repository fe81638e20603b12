"""CPU enumeration check of the many-row and several-row GEMMs' buffer offsets.

tests/cpu/gemm_offsets_check.cpp includes axiomlm_amd/csrc/gemm_offsets.h -- the functions the
kernels themselves call -- and walks whole launches at ragged row counts, odd matrix heights and
half stages of K: no load may leave its buffer, whichever of a buffer load's two offsets its
range check covers."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "cpu", "gemm_offsets_check.cpp")
INC = os.path.join(ROOT, "axiomlm_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gemm_offsets_stay_in_their_buffers(tmp_path):
    exe = str(tmp_path / "gemm_offsets_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-fno-sanitize-recover=all", f"-I{INC}",
                    SRC, "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("ok ") == 3, res.stdout
