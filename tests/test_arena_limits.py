"""fib_force_noalloc's device memory on the CPU (tests/arena_check.cpp): a
configuration of which any array does not fit is refused, also when the arrays
after it would."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_configurations_that_do_not_fit(tmp_path):
    exe = str(tmp_path / "arena_check")
    # (the kernels and HIP stay unresolved: nothing here calls them)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "arena_check.cpp"), "-o", exe, "-lpthread", "-no-pie",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
