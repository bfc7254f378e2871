"""Partially wet cells in numbers that the other meshes do not reach: whole
workgroups of them, their levels asked for across workgroup borders, nodes
with many cells around them, and lists on both sides of the length at which
the second pass changes its split.  Against the oracle, bit for bit."""
import numpy as np
import pytest

import swe_fvm_amd as swe
from oracle import oracle as O
from swe_fvm_amd import _lib
from swe_fvm_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu


def film(xyz, topo, seed, wet_share):
    """Rough bottom; a share of the cells under deep water, the others with the surface between their vertices."""
    rng = np.random.default_rng(seed)
    xyz[:, 2] = rng.uniform(0.0, 0.2, xyz.shape[0])
    tp = topo.tables()["tp"]
    z = xyz[tp, 2]
    c = 1.0 / 3.0
    bc = (z[:, 0] * c + z[:, 1] * c) + z[:, 2] * c
    T = tp.shape[0]
    h = rng.uniform(0.05, 0.9, T) * (z.max(axis=1) - bc)
    h[rng.random(T) < wet_share] = 1.0
    h[rng.random(T) < 0.02] = 0.0
    return np.stack([bc + h, rng.uniform(-0.1, 0.1, T), rng.uniform(-0.1, 0.1, T)], axis=1)


def fan(n):
    """n triangles around one node."""
    a = 2 * np.pi * np.arange(n) / n
    xyz = np.zeros((n + 1, 3))
    xyz[1:, 0], xyz[1:, 1] = np.cos(a), np.sin(a)
    rim = 1 + np.arange(n)
    nxt = np.roll(rim, -1)
    topo = swe.Topology.build(n + 1, np.stack([np.zeros(n, int), rim, nxt], 1), np.stack([rim, nxt], 1))
    return xyz, topo


MESHES = {"fan4": lambda: fan(4), "fan6": lambda: fan(6), "fan9": lambda: fan(9), "fan41": lambda: fan(41),
          "512": lambda: swe.jittered_mesh(16, 0.3, 4), "8450": lambda: swe.jittered_mesh(65, 0.3, 5),
          "28800": lambda: swe.jittered_mesh(120, 0.3, 6)}  # its list exceeds a quarter of the 65,536 lanes


@pytest.mark.parametrize("opts", [0, swe.OPT_HEAD_GRADIENT, swe.OPT_HEAD_PARTWET2])
@pytest.mark.parametrize("wet_share", [0.0, 0.5])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_partially_wet_lists_match_the_oracle(mesh, wet_share, opts):
    xyz, topo = MESHES[mesh]()
    prim = film(xyz, topo, 9, wet_share)
    sd = swe.SpaceDisc(swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt], swe.Domain(xyz, topo), prim, options=opts)
    orc = O.OracleSolver(xyz, topo.tables(), "HLLC", "Einfeldt", opts=opts)
    orc.set_state(prim)
    sd.ComputeInterfaceValues()
    if wet_share == 0.0 and not mesh.startswith("fan"):
        assert (sd.CellClass() == 1).mean() > 0.9
    for steps in (1, 2):
        sd.run("SSPRK2", steps, dt=0.0, cfl=0.15)
        orc.run("SSPRK2", steps, dt=0.0, cfl=0.15)
        assert np.array_equal(sd.GetVolField(), orc.state())


def test_list_reuse_across_getters_and_steps():
    """Steps leave the list empty for the next reconstruction, the getters in use; any order of the two agrees."""
    xyz, topo = swe.jittered_mesh(16, 0.3, 4)
    prim = film(xyz, topo, 11, 0.3)
    fl = swe.Fluxes.HLL[swe.Wavespeeds.Davis]
    sd = swe.SpaceDisc(fl, swe.Domain(xyz, topo), prim)
    orc = O.OracleSolver(xyz, topo.tables(), "HLL", "Davis")
    orc.set_state(prim)
    for scheme, fused, dt in (("SSPRK3", True, 0.0), ("Euler", True, 1e-4), ("SSPRK2", False, 0.0), ("SSPRK2", True, 0.0)):
        sd.set_fused(fused)
        sd.Integrals()
        sd.run(scheme, 1, dt=dt)
        sd.ComputeInterfaceValues()
        sd.run(scheme, 2, dt=dt)
        orc.run(scheme, 3, dt=dt, cfl=0.15)
        assert np.array_equal(sd.GetVolField(), orc.state()), (scheme, fused)


@pytest.mark.parametrize("graph", [False, True])
def test_ensemble_steps_interrupted_by_a_reconstruction(graph):
    members = [swe.jittered_mesh(n, 0.3, n) for n in (5, 16, 23)]
    states = [film(x, t, k, 0.5) for k, (x, t) in enumerate(members)]
    doms = [swe.Domain(x, t) for x, t in members]
    fl = swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt]
    out = []
    for interrupt in (False, True):
        ens = Ensemble(fl, doms, states)
        for _ in range(3):
            ens.run("SSPRK2", cfl=0.15, t_end=1.0, max_steps=4, graph=graph)
            if interrupt:
                assert _lib.load().swe_compute_interface_values(ens._h) == 0
        out.append(np.concatenate(ens.states() + [ens.times()[0][:, None].repeat(3, 1)]))
    assert np.array_equal(out[0], out[1])
