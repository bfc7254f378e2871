"""Tiles with long borders (strips of a row-ordered mesh, a tile of scattered
cells) in launches of more tiles than the chip holds at two workgroups per CU,
where the stage kernel leaves the cells beyond the ring out of LDS: against the
oracle, and its storing launches against the separate kernels, bit for bit."""
import numpy as np
import pytest

import swe_fvm_amd as swe
from oracle import oracle as O
from swe_fvm_amd.ensemble import Ensemble
from tests.test_gpu_tiles import opened, state
from tests.test_stage_tables_host import scattered

pytestmark = pytest.mark.gpu


def rows():  # 132,480 cells: 517 tiles and a half
    return swe.StructTriangMesh(184, 180, 0.02)


def ends():  # 180,000 cells, 73 of them at the end out of order
    topo = scattered(300, 73)
    return np.array(swe.jittered_mesh(300, 0.25, 8)[0]), topo


@pytest.mark.parametrize("opts", [0, swe.OPT_DRAIN_LENGTH | swe.OPT_FRICTION, swe.OPT_EXACT_BALANCE])
@pytest.mark.parametrize("flux", ["HLL", "HLLC"])
@pytest.mark.parametrize("mesh", [rows, ends])
def test_long_tiles_match_the_oracle(mesh, flux, opts):
    xyz, topo = mesh()
    prim = state(xyz, topo, 6)
    topo = opened(xyz, topo)
    sd = swe.SpaceDisc(getattr(swe.Fluxes, flux)[swe.Wavespeeds.Einfeldt], swe.Domain(xyz, topo), prim, cor=0.1,
                       tau=0.2, options=opts)
    assert sd.set_fused(True)
    orc = O.OracleSolver(xyz, topo.tables(), flux, "Einfeldt", cor=0.1, tau=0.2, opts=opts)
    orc.set_state(prim)
    for scheme, dt in (("SSPRK3", 0.0), ("Euler", 1e-4)):
        sd.run(scheme, 1, dt=dt)
        orc.run(scheme, 1, dt=dt, cfl=0.15)
        assert np.array_equal(sd.GetVolField(), orc.state()), scheme


@pytest.mark.parametrize("opts", [0, swe.OPT_DRAIN_LENGTH])
def test_long_tiles_store_the_fluxes_of_the_separate_kernels(opts):
    xyz, topo = rows()
    prim = state(xyz, topo, 7)
    bar = np.random.default_rng(1).standard_normal(prim.shape)
    got = []
    for fused in (True, False):
        sd = swe.SpaceDisc(swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt], swe.Domain(xyz, topo), prim, options=opts)
        assert sd.set_fused(fused) == fused
        got.append(sd.adjoint_run(bar, 3, dt=1e-5, checkpoint_every=2)[:2])
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("scheme", ["SSPRK2", "SSPRK3"])
def test_ensembles_of_long_tiles(scheme, graph):
    # 160,320 cells, 627 tiles while all members run, 470 and fewer once the
    # first has finished: the launches change form on the way
    fl = swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt]
    doms, prims = [], []
    for k, (nx, ny, h) in enumerate([(100, 101, 0.08), (100, 99, 0.02), (101, 100, 0.02), (100, 100, 0.03)]):
        xyz, topo = swe.StructTriangMesh(nx, ny, h)
        prims.append(state(xyz, topo, 8 + k))
        doms.append(swe.Domain(xyz, topo))
    ens = Ensemble(fl, doms, prims)
    ens.run(scheme, cfl=0.15, t_end=0.03, graph=graph)
    steps = ens.times()[1]
    assert steps.min() < steps.max()
    for k, got in enumerate(ens.states()):
        one = Ensemble(fl, [doms[k]], [prims[k]])
        one.run(scheme, cfl=0.15, t_end=0.03, graph=False)
        assert one.times()[1][0] == steps[k]
        assert np.array_equal(got, one.states()[0])
