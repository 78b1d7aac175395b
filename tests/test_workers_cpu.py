"""Helper threads of the transfers (host code, no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_a_thread_that_cannot_start_leaves_its_share_to_the_others(tmp_path):
    exe = tmp_path / "check_workers"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", str(ROOT / "flash-x_amd" / "csrc"),
                    str(ROOT / "tests" / "cpp" / "check_workers.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout.strip(), r.stderr.strip())
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
