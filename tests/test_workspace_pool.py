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


def test_a_full_device_gives_the_kept_memory_to_torch(monkeypatch):
    """An allocation of the gradient path that PyTorch cannot serve is tried again, once, after the
    library has given back what it keeps."""
    torch = pytest.importorskip("torch")
    from cfd_solvers_amd import autograd

    released, tried = [], []
    monkeypatch.setattr(autograd, "release_workspaces", lambda: released.append(1))

    def allocate(full):
        tried.append(1)
        if len(tried) <= full:
            raise torch.cuda.OutOfMemoryError("full")
        return "memory"

    assert autograd._with_room(lambda: allocate(0)) == "memory" and not released
    tried.clear()
    assert autograd._with_room(lambda: allocate(1)) == "memory" and len(released) == 1
    tried.clear()
    with pytest.raises(torch.cuda.OutOfMemoryError):
        autograd._with_room(lambda: allocate(2))
    assert len(tried) == 2


def test_release_without_kept_memory():
    """On any machine, a GPU or none, there may be nothing to give back."""
    import cfd_solvers_amd

    cfd_solvers_amd.release_workspaces()
