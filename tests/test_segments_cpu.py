"""z segments of the FP32-flux stage's columns (host code, no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_segment_length_equals_the_shortest_list_schedule(tmp_path):
    exe = tmp_path / "check_segments"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(ROOT / "flash-x_amd" / "csrc"),
                    str(ROOT / "tests" / "cpp" / "check_segments.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout.strip())
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
