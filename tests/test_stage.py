"""Host transfers on the CPU, with requests for host memory and copies that
fail in turn: an error code or the arrays bit for bit, never an exception or
an abort out of the C functions that call them (tests/stage_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failing_requests(tmp_path):
    exe = str(tmp_path / "stage_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "stage_check.cpp"), "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), (r.returncode, r.stdout, r.stderr)
