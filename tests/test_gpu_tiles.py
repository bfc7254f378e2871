"""The staged tile kernels at the edges of their tables: meshes of one cell
to a few tiles, tiles cut short, strips whose tiles have long borders, and
geometry that the tile kernels leave to the separate ones.  Against the
oracle, bit for bit, with the tiles on and off."""
import numpy as np
import pytest

import swe_fvm_amd as swe
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def state(xyz, topo, seed):
    rng = np.random.default_rng(seed)
    xyz[:, 2] = 0.3 * np.sin(3.0 * xyz[:, 0]) * np.cos(2.0 * xyz[:, 1])
    tp = topo.tables()["tp"]
    c = 1.0 / 3.0
    z = xyz[tp, 2]
    bc = (z[:, 0] * c + z[:, 1] * c) + z[:, 2] * c
    w = np.maximum(bc, 0.15 + 0.02 * rng.standard_normal(tp.shape[0]))
    return np.stack([w, rng.uniform(-0.2, 0.2, w.shape[0]), rng.uniform(-0.2, 0.2, w.shape[0])], 1)


def opened(xyz, topo):
    t = topo.tables()
    b = np.nonzero(t["et"][:, 1] < 0)[0]
    x = 0.5 * (xyz[t["ep"][b, 0], 0] + xyz[t["ep"][b, 1], 0])
    return topo.with_boundary_tag(b[x < x.min() + 1e-9], swe.FREE_FLOW)


def one_triangle():
    xyz = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 1.0, 0.0]])
    return xyz, swe.Topology.build(3, [[0, 1, 2]], [[0, 1], [1, 2], [2, 0]])


MESHES = {"1": one_triangle, "4": lambda: swe.StructTriangMesh(1, 1, 0.5), "256": lambda: swe.StructTriangMesh(8, 8, 0.1),
          "260": lambda: swe.StructTriangMesh(13, 5, 0.1), "strip256": lambda: swe.StructTriangMesh(64, 1, 0.1),
          "strip260": lambda: swe.StructTriangMesh(1, 65, 0.1), "1020": lambda: swe.StructTriangMesh(3, 85, 0.1),
          "rows": lambda: swe.StructTriangMesh(100, 7, 0.1), "jittered": lambda: swe.jittered_mesh(23, 0.3, 8)}


@pytest.mark.parametrize("opts", [0, swe.OPT_DRAIN_LENGTH | swe.OPT_FRICTION, swe.OPT_EXACT_BALANCE])
@pytest.mark.parametrize("flux", ["HLL", "HLLC"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_tiles_match_the_oracle(mesh, flux, opts):
    xyz, topo = MESHES[mesh]()
    prim = state(xyz, topo, 3)
    topo = opened(xyz, topo)
    fl = getattr(swe.Fluxes, flux)[swe.Wavespeeds.Einfeldt]
    sd = swe.SpaceDisc(fl, swe.Domain(xyz, topo), prim, cor=0.1, tau=0.2, options=opts)
    assert sd.set_fused(True)
    orc = O.OracleSolver(xyz, topo.tables(), flux, "Einfeldt", cor=0.1, tau=0.2, opts=opts)
    orc.set_state(prim)
    for scheme, dt in (("SSPRK3", 0.0), ("Euler", 1e-3), ("SSPRK2", 1e-3)):
        sd.run(scheme, 2, dt=dt)
        orc.run(scheme, 2, dt=dt, cfl=0.15)
        got = sd.GetVolField()
        assert np.array_equal(got, orc.state()), scheme
    z = xyz[:, 2] + 0.01 * np.cos(xyz[:, 0])  # the tiles' copies of the geometry follow the bathymetry
    sd.set_bathymetry(z)
    moved = xyz.copy()
    moved[:, 2] = z
    orc = O.OracleSolver(moved, topo.tables(), flux, "Einfeldt", cor=0.1, tau=0.2, opts=opts)
    orc.set_state(got)
    sd.run("SSPRK2", 2, dt=0.0)
    orc.run("SSPRK2", 2, dt=0.0, cfl=0.15)
    assert np.array_equal(sd.GetVolField(), orc.state())


@pytest.mark.parametrize("change", ["negative zero", "tiny", "huge"])
def test_unusual_coordinates_keep_the_separate_kernels(change):
    xyz, topo = swe.StructTriangMesh(8, 8, 0.1)
    prim = state(xyz, topo, 4)
    if change == "negative zero":
        xyz[np.nonzero(xyz[:, 0] == 0.0)[0][0], 0] = -0.0
    else:
        xyz[:, :2] *= 1e-150 if change == "tiny" else 1e150
    sd = swe.SpaceDisc(swe.Fluxes.HLLC[swe.Wavespeeds.Davis], swe.Domain(xyz, topo), prim)
    assert not sd.set_fused(True)
    orc = O.OracleSolver(xyz, topo.tables(), "HLLC", "Davis")
    orc.set_state(prim)
    dt = 1e-3 if change != "tiny" else 1e-154
    sd.run("SSPRK2", 2, dt=dt)
    orc.run("SSPRK2", 2, dt=dt)
    assert np.array_equal(sd.GetVolField(), orc.state(), equal_nan=True)


@pytest.mark.parametrize("opts", [0, swe.OPT_DRAIN_LENGTH])
@pytest.mark.parametrize("nx, ny", [(127, 129), (128, 128), (129, 128)])  # 256 tiles, the last cut short or not; 258
def test_around_a_tile_per_compute_unit(nx, ny, opts):
    xyz, topo = swe.StructTriangMesh(nx, ny, 0.02)
    prim = state(xyz, topo, 5)
    sd = swe.SpaceDisc(swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt], swe.Domain(xyz, topo), prim, options=opts)
    orc = O.OracleSolver(xyz, topo.tables(), "HLLC", "Einfeldt", opts=opts)
    orc.set_state(prim)
    for scheme, dt in (("SSPRK2", 0.0), ("Euler", 1e-3)):
        sd.run(scheme, 2, dt=dt)
        orc.run(scheme, 2, dt=dt, cfl=0.15)
        assert np.array_equal(sd.GetVolField(), orc.state()), scheme
