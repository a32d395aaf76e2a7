"""Host check of the row shapes of the RMSNorm kernels for any width
(kernelproblems_amd/csrc/kp_rms_shapes.hpp): the constexpr rules the kernels
compile, built here with g++ and run over every width they take."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_column_is_owned_once(tmp_path):
    exe = tmp_path / "rms_shapes_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'kernelproblems_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "rms_shapes_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "0 bad widths", res.stdout + res.stderr
