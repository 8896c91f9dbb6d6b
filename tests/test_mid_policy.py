"""CPU check of the rules by which projection launches go to the mid kernels
(heliopause_amd/csrc/hp_mid_policy.h), compiled with g++ (tests/mid_policy.cpp);
no GPU is involved."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_mid_policy(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "mid_policy"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{ROOT / 'heliopause_amd' / 'csrc'}",
                    str(ROOT / "tests" / "mid_policy.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mid policy ok" in r.stdout
