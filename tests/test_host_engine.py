"""The engine's host code on a HIP runtime of host memory (tests/host): state after
allocation failures, what queued launches read, and what the process-wide pool
keeps.  No device."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "spaqr_public_amd", "csrc", "host")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="session")
def engine_test(tmp_path_factory):
    out = tmp_path_factory.mktemp("host")
    sources = [os.path.join(ROOT, "tests", "host", "engine_test.cpp")]
    sources += [os.path.join(HOST, f + ".cpp") for f in ("common", "krylov", "parallel", "partition", "hypergraph",
                                                         "profile", "tuner")]

    def compile_(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        subprocess.run(["g++", "-std=c++17", "-O0", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include", "-I" + HOST,
                        "-c", src, "-o", obj], check=True)
        return obj

    with ThreadPoolExecutor(4) as ex:
        objs = list(ex.map(compile_, sources))
    exe = str(out / "engine_test")
    # the launchers that no case reaches stay unresolved
    subprocess.run(["g++", *objs, "-o", exe, "-no-pie", "-pthread", "-ldl", "-Wl,--unresolved-symbols=ignore-all"],
                   check=True)
    return exe


CASES = ["transposed", "segments", "no_memory", "rrqr_ring", "timeout", "trim", "stream", "tuner", "offsets",
         "codes"]


@pytest.mark.parametrize("case", CASES)
def test_host(engine_test, case, tmp_path):
    env = dict(os.environ, SPAQR_TUNE_FILE="/dev/null")
    r = subprocess.run([engine_test, case, str(tmp_path / "tune.json")], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
