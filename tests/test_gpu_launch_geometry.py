"""The step kernels' tiles and their order over the XCDs change no result: every row width where the
rule for the tile changes (below, at and beyond one to nine 64-cell segments), lattices of fewer
tiles than XCDs and tile counts that fill no whole run of tiles, against 64-cell tiles dealt
round-robin, bit for bit: populations after both parities, fields, and the adjoint's gradient."""
import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu

SHAPES = [(19, 2, 3, 2), (27, 56, 5, 7), (19, 63, 4, 3), (19, 65, 5, 3), (9, 130, 9, 1), (19, 257, 4, 3),
          (19, 301, 5, 7), (27, 384, 3, 2), (19, 400, 3, 5), (9, 512, 11, 1), (9, 513, 13, 1), (9, 1100, 7, 1)]


def _run(hip, monkeypatch, shape, storage, walls, env):
    q, nx, ny, nz = shape
    for k in ("CFD_LBM_BX", "CFD_LBM_XCD_REMAP"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    g = hip.EsotericPullHipSolver(q, nx, ny, nz, 0.6, storage=storage)
    if walls:
        f = np.zeros((nz, ny, nx), np.uint8)
        f[:, 0, :] = 0x80
        f[:, -1, :] = 0x81
        f[:, ny // 2, nx // 2] = 0x80
        g.set_flags(f)
        g.set_wall_velocity(1, (0.05, 0.0, 0.0))
    g.initialize_taylor_green(0.02, 1e-4, 3)
    out = []
    for steps in (3, 1):
        g.step(steps)
        m = g.download_macroscopic()
        out += [g.logical_populations(), m.rho, m.ux, m.uy, m.uz]
    g.close()
    return out


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("storage", ["fp32", "fp16s", "fp64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_tiles_change_no_result(hip, monkeypatch, shape, storage, walls):
    if walls and shape[1] < 8:
        pytest.skip("the obstacle needs a wider lattice")
    report("launch_geometry", shape=shape, storage=storage, walls=walls)
    plain = _run(hip, monkeypatch, shape, storage, walls, {"CFD_LBM_BX": "64", "CFD_LBM_XCD_REMAP": "0"})
    for env in ({}, {"CFD_LBM_XCD_REMAP": "3"}):
        for got, want in zip(_run(hip, monkeypatch, shape, storage, walls, env), plain):
            assert np.array_equal(got, want), env


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "fp64"])
@pytest.mark.parametrize("nx", [65, 301])
def test_tiles_change_no_gradient(hip, monkeypatch, nx, storage):
    from cfd_solvers_amd import geometry

    flags = geometry.channel_flags(nx, 9, 8, inlet_outlet=True)
    results = []
    for env in ({"CFD_LBM_BX": "64", "CFD_LBM_XCD_REMAP": "0"}, {}, {"CFD_LBM_XCD_REMAP": "3"}):
        report("launch_geometry_adjoint", nx=nx, storage=storage, env=env)
        for k in ("CFD_LBM_BX", "CFD_LBM_XCD_REMAP"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        s = hip.EsotericPullHipSolver("d3q19", nx, 9, 8, 0.6, storage=storage)
        s.set_flags(flags)
        s.set_porosity(np.where(flags == 0, 0.004, 0.0).astype(np.float32))
        s.set_inlet_outlet(0.04, 1.0)
        s.initialize_uniform()
        results.append(s.adjoint_run(6, 3, 3, 1, nx - 2))
        s.close()
    for r in results[1:]:
        assert r[0] == results[0][0] and np.array_equal(r[1], results[0][1]) and r[2] == results[0][2]
