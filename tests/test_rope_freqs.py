"""Host check of rotary embedding's inverse frequencies
(kernelproblems_amd/csrc/kp_rope_freqs.hpp), built here with g++: every head
width and several thetas against long double powers rounded once to fp32."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_rounded_once(tmp_path):
    exe = tmp_path / "rope_freqs_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'kernelproblems_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "rope_freqs_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip().endswith(" 0 bad"), res.stdout + res.stderr
