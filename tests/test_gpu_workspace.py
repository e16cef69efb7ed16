"""The adjoint's working memory is handed from call to call: runs that find a block another solver's
run left behind return what a first run returns, bit for bit, and the device-memory gradient of the
two-level plan is the host one."""
import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu


def _solver(hip, n, storage):
    from cfd_solvers_amd import geometry

    nx, ny, nz = n
    s = hip.EsotericPullHipSolver("d3q19", nx, ny, nz, 0.6, storage=storage)
    flags = geometry.channel_flags(nx, ny, nz, inlet_outlet=True)
    s.set_flags(flags)
    s.set_porosity(np.where(flags == 0, 0.004, 0.0).astype(np.float32))
    s.set_inlet_outlet(0.04, 1.0)
    return s


def _run(s, every, snapshots):
    s.initialize_uniform()
    if every:
        return s.adjoint_run(12, 4, every, 1, s.shape[-1] - 2)
    return s.adjoint_run_binomial(12, 4, snapshots)[:3]


def _same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and a[2] == b[2]


@pytest.mark.parametrize("storage", ["fp32", "fp16s"])
def test_reused_blocks_change_nothing(hip, storage):
    plans = [(4, 0), (0, 3), (5, 0), (0, 2)]
    # Each shape's first result comes from a process state in which its solver is the only one, so
    # that the pool is empty when it starts.
    shapes = [(19, 14, 12), (33, 12, 11)]
    first = {}
    for n in shapes:
        for plan in plans:
            report("workspace_first", storage=storage, n=n, plan=plan)
            s = _solver(hip, n, storage)
            first[n, plan] = _run(s, *plan)
            s.close()
    solvers = {n: _solver(hip, n, storage) for n in shapes}
    for plan in plans:
        for n in shapes:
            report("workspace_again", storage=storage, n=n, plan=plan)
            assert _same(_run(solvers[n], *plan), first[n, plan])


def test_device_gradient_of_the_two_level_plan(hip, dev):
    n = (19, 14, 12)
    s = _solver(hip, n, "fp32")
    want = _run(s, 4, 0)
    grad = dev.upload(np.full(s.cells, np.nan))
    report("two_level_device", n=n)
    s.initialize_uniform()
    J, du = s.adjoint_run_device(12, 4, 4, grad)
    assert J == want[0] and du == want[2]
    assert np.array_equal(dev.download(grad, s.shape, np.float64), want[1])
    with pytest.raises(RuntimeError, match="aligned"):
        s.adjoint_run_device(12, 4, 4, 0)


@pytest.mark.parametrize("every", [1, 4, 5, 11, 12, 40])
def test_two_level_plans_agree(hip, every):
    """The last segment's states are those of the forward sweep, the others' are recomputed: whatever
    the interval (one state a segment, a short last segment, one segment), the binomial plan's J and
    gradients, bit for bit."""
    report("two_level_plan", every=every)
    s = _solver(hip, (19, 14, 12), "fp32")
    assert _same(_run(s, every, 0), _run(s, 0, 3))


def test_release(hip):
    """Kept memory goes back to the device on request, and the next calls return what they returned."""
    import ctypes as C

    report("workspace_release")
    rt = C.CDLL("libamdhip64.so.7")

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    s = _solver(hip, (33, 40, 41), "fp32")
    flow = hip.EsotericPullHipSolver("d2q9", 2048, 1024, 1, 0.6)
    flow.initialize_taylor_green(0.02, 1e-4, 3)
    want = _run(s, 4, 0)
    flow.step(16)
    fields = flow.download_macroscopic()
    before, held = free_bytes(), flow.resident_bytes()
    hip.release_workspaces()
    assert flow.resident_bytes() <= held - flow.population_bytes()
    assert free_bytes() >= before + flow.population_bytes()
    assert _same(_run(s, 4, 0), want)
    flow.initialize_taylor_green(0.02, 1e-4, 3)
    flow.step(16)
    again = flow.download_macroscopic()
    assert flow.resident_bytes() == held
    assert np.array_equal(again.rho, fields.rho) and np.array_equal(again.ux, fields.ux)
    flow.close()
    s.close()


@pytest.mark.parametrize("plan", [(4, 0), (0, 3)])
@pytest.mark.parametrize("storage", ["fp32", "fp16s"])
def test_a_reused_block_may_hold_anything(hip, storage, plan):
    """A run that finds a block full of NaN (states, lambda and sums of a run on NaN populations) returns
    what a run in fresh memory returned; that it is the same block shows in the device's free memory."""
    import ctypes as C

    report("workspace_poisoned", storage=storage, plan=plan)
    rt = C.CDLL("libamdhip64.so.7")

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n = (65, 48, 40)
    s, bad = _solver(hip, n, storage), _solver(hip, n, storage)
    hip.release_workspaces()
    before = free_bytes()
    want = _run(s, *plan)
    kept = free_bytes()
    assert kept < before
    bad.initialize_uniform()
    bad.upload_populations(np.full((19, bad.cells), np.nan, np.float32))
    poisoned = (bad.adjoint_run(12, 4, plan[0], 1, n[0] - 2) if plan[0] else bad.adjoint_run_binomial(12, 4, plan[1]))
    assert np.isnan(poisoned[0]) and free_bytes() == kept
    assert _same(_run(s, *plan), want) and free_bytes() == kept
    s.close()
    bad.close()


TORCH_TWO_LEVEL = r"""
import sys
import numpy as np
import torch  # first: the library then shares torch's HIP runtime

torch.ones(1, device="cuda:0").sum().item()
sys.path.insert(0, sys.argv[1])
import cfd_solvers_amd as hip
from cfd_solvers_amd import geometry
from cfd_solvers_amd.autograd import LbmAdjointProblem, lbm_objective

n = (19, 14, 12)
flags = geometry.channel_flags(*n, inlet_outlet=True)
blend = np.where(flags == 0, 0.01 * np.random.default_rng(4).uniform(0.3, 0.7, flags.shape), 0.0).astype(np.float32)
prob = LbmAdjointProblem(flags=flags, shape=n, storage="fp32", steps=20, window=5, checkpoint_every=7)
gamma = torch.tensor(blend, device="cuda:0", requires_grad=True)
u_peak = torch.tensor(0.04, device="cuda:0", requires_grad=True)
J = lbm_objective(gamma, u_peak, prob)
J.backward()
s = hip.EsotericPullHipSolver("d3q19", *n, 0.6)
s.set_flags(flags)
s.set_inlet_outlet(float(u_peak.item()), 1.0)
s.set_porosity(blend)
s.initialize_uniform()
ref_J, ref_grad, ref_du = s.adjoint_run(20, 5, 7, 1, n[0] - 2)
assert J.item() == ref_J, (J.item(), ref_J)
assert gamma.grad.device.type == "cuda" and gamma.grad.shape == gamma.shape and gamma.grad.dtype == torch.float32
assert np.array_equal(gamma.grad.cpu().numpy(), ref_grad.astype(np.float32))
assert u_peak.grad.item() == np.float32(ref_du)
value, grad, du = prob.run(gamma.detach(), u_peak.item())  # the public call hands out host memory
assert isinstance(grad, np.ndarray) and value == ref_J and np.array_equal(grad, ref_grad) and du == ref_du
print("two-level ok")
"""


def test_two_level_gradient_of_a_device_tensor():
    """lbm_objective with checkpoint_every > 0 and gamma on the GPU: J and both gradients are those of
    adjoint_run, bit for bit.  In a child process that imports torch first, as a torch user would."""
    import subprocess
    import sys
    from pathlib import Path

    report("two_level_torch")
    root = Path(__file__).resolve().parents[1]
    out = subprocess.run([sys.executable, "-c", TORCH_TWO_LEVEL, str(root)], capture_output=True, text=True,
                         timeout=240, cwd=root)
    assert out.returncode == 0 and "two-level ok" in out.stdout, out.stderr[-3000:]
