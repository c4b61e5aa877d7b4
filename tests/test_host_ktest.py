"""The kernel test harness on a HIP runtime of host memory (tests/host)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rrqr_without_columns(tmp_path):
    exe = str(tmp_path / "ktest_test")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O0", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + rocm + "/include",
                    "-I" + os.path.join(ROOT, "spaqr_public_amd", "csrc", "ktest"),
                    os.path.join(ROOT, "tests", "host", "ktest_test.cpp"), "-o", exe, "-no-pie",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
