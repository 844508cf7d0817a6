"""Exchanges through LDS in the FP64 state-reading stage bodies, on the CPU: the
bodies compiled for the host, one fiber per lane, give the same results whether
a lane's writes reach the others at once or at the next barrier only
(tests/cpu/wave_check.cpp, tests/cpu/wave/hip/hip_runtime.h)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_exchange_has_its_barrier(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cxx = shutil.which("clang++", path=os.path.join(rocm, "llvm", "bin")) or shutil.which("clang++")
    if cxx is None:
        pytest.skip("needs clang++ (vector types of the kernel headers)")
    exe = str(tmp_path / "wave_check")
    csrc = os.path.join(ROOT, "dgpr_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wno-unknown-attributes",
                    "-Wno-unused-function", "-I" + os.path.join(ROOT, "tests", "cpu", "wave"),
                    "-I" + csrc, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpu", "wave_check.cpp"),
                    os.path.join(csrc, "dgx_tables.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
