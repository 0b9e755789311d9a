"""Offsets of direct loads near the end of their operands (laya-cuda_amd/csrc/ranges.hpp, shared with the
kernels) walked on the CPU by tests/load_ranges.cpp (no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "laya-cuda_amd" / "csrc"


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not installed")
def test_scalar_offsets_stay_inside_their_resources(tmp_path):
    exe = tmp_path / "load_ranges"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(ROOT / "tests" / "load_ranges.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stderr
    assert int(run.stdout.split()[1]) > 100000
