"""fib_set_impact on the CPU with failing copies (tests/impact_check.cpp): a
call that succeeds leaves the device's record equal to the host's, also the
one after a call that failed, with the same value."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failing_copies(tmp_path):
    exe = str(tmp_path / "impact_check")
    # (the kernels and the rest of HIP stay unresolved: nothing here calls them)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "impact_check.cpp"), "-o", exe, "-lpthread", "-no-pie",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
