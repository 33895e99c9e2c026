"""Host side of the resident 2D time loop, without a GPU: resident2d.cpp and the read-backs' staging
compiled against a stand-in for the HIP runtime (tests/host/resident_host.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "wave-simulation_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "resident_host")
    subprocess.run(["/opt/rocm/bin/amdclang++", "-x", "c++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + CSRC, os.path.join(ROOT, "tests", "host", "resident_host.cpp"),
                    os.path.join(CSRC, "resident2d.cpp"), "-o", exe], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("test", ["no_memory", "memory_asked_for", "timing", "failure", "refusal", "queue", "plan",
                                  "step_bytes", "staging"])
def test_resident_host(program, test):
    r = subprocess.run([program, test], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stderr
