"""The workspace pool (csrc/device_memory.hpp) compiled for the host against a stand-in for the HIP
allocator: reuse and its bounds, a full device, and blocks that solvers hold."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(f'#include "{HERE / "host" / "hip_stub.h"}"\n')
    exe = d / "workspace_pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-I", str(d), "-I",
                    str(HERE.parent / "cfd_solvers_amd" / "csrc"), str(HERE / "host" / "workspace_pool.cpp"), "-o",
                    str(exe), "-pthread"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["reuse", "full_device", "foreign_capture", "held_bound", "held_close_fit",
                                      "held_close_fit_over_the_bound", "held_bound_two_threads",
                                      "held_again_after_a_full_device", "held_again_after_a_failed_call",
                                      "reclaimable", "release"])
def test_pool(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, r.stderr
