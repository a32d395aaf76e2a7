"""Host check of the row and column of a chunk in the row-strided SwiGLU form
(kernelproblems_amd/csrc/kp_row_chunks.hpp): the constexpr definition the
kernels compile, built here with g++ and run up to the largest rows that a
launch takes, whose columns do not fit 32 bits."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_columns_past_32_bits(tmp_path):
    exe = tmp_path / "row_chunks_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'kernelproblems_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "row_chunks_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip().endswith(" 0 bad"), res.stdout + res.stderr
