"""swe_release_workspaces: the device gets back what solvers keep between
their adjoint, tangent and diagnostic calls, and the next call is the same."""
import numpy as np
import pytest
import torch

import swe_fvm_amd as swe
from tests import _common as C

pytestmark = pytest.mark.gpu


def test_memory_given_back_between_calls():
    xyz, topo, prim = C.wet_dry_mesh(60, seed=5)
    sd = swe.SpaceDisc(swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt], swe.Domain(xyz, topo), prim)
    bar = np.random.default_rng(4).standard_normal(prim.shape)
    out = []
    for _ in range(2):
        sd.SetVolField(prim)
        out.append(sd.adjoint_run(bar, 40, dt=1e-4, checkpoint_every=40)[:2])
        free = torch.cuda.mem_get_info()[0]
        swe.release_workspaces()
        assert torch.cuda.mem_get_info()[0] > free
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
