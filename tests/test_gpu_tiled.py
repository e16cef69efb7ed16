"""Several D2Q9 steps in one launch (LDS tiles) against the same number of single steps, bit for bit:
the raw slots (those left behind at walls included), populations and fields, over both tile sizes,
lattices at the halo's width, at tile edges and beyond them, odd and even starts and counts, and
every option the step has."""
import ctypes as C

import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu

# A tile's interior is 56 wide (2 steps: 60); the small one has 2 to 8 rows (2 steps: to 12) by the
# lattice's size, the large one 26 (30).
SMALL = [(8, 8), (24, 8), (25, 17), (57, 9), (131, 40), (2300, 15), (171, 700)]
LARGE = [(448, 520), (449, 469), (9, 22300)]


def _solver(hip, shape, storage, scene):
    nx, ny = shape
    accel = (1e-5, -2e-6, 0.0) if scene in ("forced", "les") else (0.0, 0.0, 0.0)
    g = hip.EsotericPullHipSolver("d2q9", nx, ny, 1, 0.6, accel, storage=storage)
    f = np.zeros((1, ny, nx), np.uint8)
    if scene in ("cavity", "forced"):
        f[:, :, 0] = f[:, :, -1] = f[:, 0, :] = 0x80
        f[:, -1, :] = 0x81
        f[:, ny // 2, nx // 2] = 0x80
        g.set_flags(f)
        g.set_wall_velocity(1, (0.05, 0.0, 0.0))
    if scene == "channel":
        f[:, 0, :] = f[:, -1, :] = 0x80
        f[:, 1:-1, 0], f[:, 1:-1, -1] = 1, 2
        g.set_flags(f)
        g.set_inlet_outlet(0.04, 1.0)
    if scene == "local":
        rng = np.random.default_rng(3)
        g.set_local_body_acceleration(*(1e-5 * rng.standard_normal((3, nx * ny))).astype(np.float32))
    if scene == "les":
        g.set_smagorinsky(True)
    g.initialize_taylor_green(0.02, 1e-4, 3)
    return g


def _state(g):
    m = g.download_macroscopic()
    return [g.raw_storage(), g.logical_populations(), m.rho, m.ux, m.uy]


def _compare(hip, shape, storage, scene, counts):
    report("tiled", shape=shape, storage=storage, scene=scene, counts=counts)
    many, one = (_solver(hip, shape, storage, scene) for _ in range(2))
    before = many.resident_bytes()
    for count in counts:
        many.step(count)
        for _ in range(count):
            one.step(1)
        for got, want in zip(_state(many), _state(one)):
            assert np.array_equal(got, want), f"differs after a call of {count} steps"
    # The comparison is one of two paths: only `many` has taken a second lattice.
    assert many.resident_bytes() >= before + many.population_bytes() > one.resident_bytes()
    many.close()
    one.close()


@pytest.mark.parametrize("scene", ["periodic", "cavity", "channel", "forced", "local"])
@pytest.mark.parametrize("storage", ["fp32", "fp16s", "fp32s"])
@pytest.mark.parametrize("shape", SMALL)
def test_small_tiles(hip, shape, storage, scene):
    _compare(hip, shape, storage, scene, (4, 5, 8, 1, 23))


@pytest.mark.parametrize("scene", ["periodic", "cavity", "channel", "forced"])
@pytest.mark.parametrize("storage", ["fp32", "fp16s", "fp32s"])
@pytest.mark.parametrize("shape", LARGE)
def test_large_tiles(hip, shape, storage, scene):
    _compare(hip, shape, storage, scene, (4, 13))


def test_smagorinsky(hip):
    _compare(hip, (57, 9), "fp32", "les", (12,))


@pytest.mark.parametrize("kind", ["narrow", "fp64", "porous"])
def test_other_lattices_take_single_steps(hip, kind):
    report("tiled_not", kind=kind)
    g = _solver(hip, (7, 9) if kind == "narrow" else (25, 17), "fp64" if kind == "fp64" else "fp32", "periodic")
    if kind == "porous":
        g.set_porosity(np.full(25 * 17, 0.1, np.float32))
    before = g.resident_bytes()
    g.step(8)
    assert g.resident_bytes() == before


def test_first_call_during_a_capture_of_another_stream(hip):
    """The call that takes the second lattice neither ends a global-mode capture of an unrelated
    stream nor is recorded in it."""
    report("tiled_capture")
    g, one = (_solver(hip, (57, 9), "fp32", "cavity") for _ in range(2))
    rt = C.CDLL("libamdhip64.so.7")
    stream, graph, nodes = C.c_void_p(), C.c_void_p(), C.c_size_t(99)
    rt.hipStreamDestroy.argtypes = rt.hipGraphDestroy.argtypes = [C.c_void_p]
    assert rt.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    g.wait()
    one.wait()
    assert rt.hipStreamBeginCapture(stream, 0) == 0  # hipStreamCaptureModeGlobal
    before = g.resident_bytes()
    g.step(8)
    assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert rt.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 0
    assert rt.hipGraphDestroy(graph) == 0 and rt.hipStreamDestroy(stream) == 0
    assert g.resident_bytes() >= before + g.population_bytes()
    for _ in range(8):
        one.step(1)
    for got, want in zip(_state(g), _state(one)):
        assert np.array_equal(got, want)


@pytest.mark.parametrize("shape,storage,scene,count,taken", [
    ((60, 4000), "fp16s", "cavity", 8, False), ((60, 4000), "fp32", "cavity", 8, True),
    ((60, 4000), "fp32", "forced", 8, False), ((64, 4000), "fp32", "les", 8, False),
    ((65, 4000), "fp16s", "periodic", 8, True), ((60, 4000), "fp16s", "periodic", 8, False),
    ((128, 2000), "fp16s", "cavity", 8, False), ((128, 2000), "fp16s", "periodic", 8, True),
    ((128, 2000), "fp32", "forced", 8, True), ((449, 469), "fp32", "periodic", 7, False),
    ((449, 469), "fp16s", "periodic", 8, True), ((100, 500), "fp16s", "periodic", 4, True),
    ((100, 500), "fp16s", "periodic", 3, False), ((1000, 8000), "fp16s", "cavity", 8, True),
    ((256, 31250), "fp16s", "cavity", 8, False), ((256, 31250), "fp16s", "periodic", 8, True)])
def test_lattices_that_take_several_steps_a_launch(hip, shape, storage, scene, count, taken):
    """The rule by width, storage, forcing and size: only lattices that gain take a second array."""
    report("tiled_rule", shape=shape, storage=storage, scene=scene, count=count)
    g = _solver(hip, shape, storage, scene)
    before = g.resident_bytes()
    g.step(count)
    grown = g.resident_bytes() - before
    assert grown >= g.population_bytes() if taken else grown == 0
    g.close()


@pytest.mark.parametrize("storage", ["fp32", "fp16s"])
@pytest.mark.parametrize("shape", [(57, 9), (448, 520)])
def test_plain_planes(hip, monkeypatch, shape, storage):
    """The layout of lattices beyond 4 GiB."""
    monkeypatch.setenv("CFD_LBM_LAYOUT", "planes")
    _compare(hip, shape, storage, "cavity", (8, 9))
