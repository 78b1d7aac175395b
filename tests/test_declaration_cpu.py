"""A hierarchy that could not be declared for want of memory (host code, no
GPU: the C API over stand-ins of the HIP runtime)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")


@pytest.mark.skipif(HIPCC is None or shutil.which("g++") is None, reason="no hipcc or host C++ compiler")
def test_failed_declaration_leaves_a_batch_without_a_hierarchy(tmp_path):
    obj, exe = tmp_path / "check.o", tmp_path / "check"
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-c",
                    str(ROOT / "tests" / "cpp" / "check_declaration.cpp"), "-o", str(obj)], check=True)
    subprocess.run(["g++", "-no-pie", str(obj), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout.strip())
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
