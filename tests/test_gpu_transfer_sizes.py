"""States that cross through a free state buffer (22,000 cells and more) and
those below, turned on the host: the round trip on both sides of the line, and
what other calls still read in the buffers, in every layout."""
import numpy as np
import pytest

import swe_fvm_amd as swe
from swe_fvm_amd.ensemble import Ensemble
from tests.test_gpu_transfers import FLUX, humps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [0, 64, 8, 1])
@pytest.mark.parametrize("mesh", [(1, 1), (3, 1833), (110, 50), (3, 1835), (101, 99)])  # 21,996 | 22,000, 22,020
def test_round_trip(mesh, block):
    xyz, topo = swe.StructTriangMesh(*mesh, 0.1)
    T = topo.NumTriangles()
    sd = swe.SpaceDisc(FLUX, swe.Domain(xyz, topo), humps(T, 1))
    sd.set_layout(block)
    for seed in (2, 3):
        prim = humps(T, seed)
        sd.SetVolField(prim)
        assert np.array_equal(sd.GetVolField(), prim)


@pytest.mark.parametrize("scheme", ["Euler", "SSPRK2", "SSPRK3"])
@pytest.mark.parametrize("dt", [0.0, 1e-4])
def test_getters_after_a_crossing(scheme, dt):
    xyz, topo = swe.jittered_mesh(110, 0.3, 8)
    prim = humps(topo.NumTriangles(), 4)
    seen = []
    for cross in (False, True):
        sd = swe.SpaceDisc(FLUX, swe.Domain(xyz, topo), prim)
        sd.run(scheme, 2, dt=dt)
        if cross:
            sd.SetVolField(sd.GetVolField())
        seen.append((sd.GetFluxes(), sd.GetMinLenToWavespeed(), sd.GetVolField()))
    assert np.array_equal(seen[0][0], seen[1][0]) and seen[0][1] == seen[1][1]
    assert np.array_equal(seen[0][2], seen[1][2])


@pytest.mark.parametrize("block", [0, 64])
@pytest.mark.parametrize("scheme", ["Euler", "SSPRK2"])
def test_finished_members_survive_a_crossing(scheme, block):
    members = [swe.jittered_mesh(n, 0.3, n) for n in (6, 20, 110)]
    prims = [humps(t.NumTriangles(), k) for k, (_, t) in enumerate(members)]
    out = []
    for cross in (False, True):
        ens = Ensemble(FLUX, [swe.Domain(x, t) for x, t in members], prims)
        ens.set_layout(block)
        for _ in range(8):
            _, active = ens.run(scheme, cfl=0.15, t_end=0.01, max_steps=3, graph=False)
            if cross:
                ens.set_states(ens.states())
        out.append(np.concatenate(ens.states()))
    assert active < 3  # some members finished on the way
    assert np.array_equal(out[0], out[1])
