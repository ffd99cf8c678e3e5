"""Launchers refuse arguments that their kernels would read or write past (host code only: the
refusals come before any GPU call)."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
LIB = ROOT / "agent-serve_amd" / "lib"


@pytest.mark.skipif(shutil.which("hipcc") is None and not pathlib.Path("/opt/rocm/bin/hipcc").exists(),
                    reason="hipcc not available")
def test_refused_arguments(pkg, tmp_path):
    pkg.hip_lib()
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = tmp_path / "launch_check"
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", f"-I{ROOT / 'agent-serve_amd' / 'csrc'}",
                    f"-I{ROOT / 'include'}", "-o", str(exe), str(ROOT / "tests" / "launch_check.cpp"), f"-L{LIB}", "-ltf_hip",
                    f"-Wl,-rpath,{LIB}"], check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60)
    assert out.stdout.splitlines() and all(line.endswith(" 1") for line in out.stdout.splitlines()), out.stdout
