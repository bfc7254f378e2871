"""Coordinates that the tile kernels take: negative zeros (mirrored and rounded
meshes, both zeros on one edge) and the extremes of the accepted exponents.
Against the oracle, and against the separate kernels with their full square
root and division down to the signs of zeros."""
import numpy as np
import pytest

import swe_fvm_amd as swe
from oracle import oracle as O
from tests.test_gpu_tiles import opened, state

pytestmark = pytest.mark.gpu


def centred(n):
    return swe.StructTriangMesh(n, n, 0.25, -0.125 * n, -0.125 * n)


def mirrored():
    xyz, topo = centred(16)
    xyz[:, 0] *= -1.0
    return xyz, topo


def mixed():  # zeros of both signs along both axes
    xyz, topo = centred(16)
    rng = np.random.default_rng(2)
    for a in (0, 1):
        zero = xyz[:, a] == 0.0
        xyz[zero, a] = np.where(rng.random(zero.sum()) < 0.5, -0.0, 0.0)
    return xyz, topo


def rounded():
    xyz, topo = swe.jittered_mesh(20, 0.25, 3)
    xyz = np.array(xyz)
    xyz[:, :2] = -np.round(xyz[:, :2] - 0.5, 2)
    return xyz, topo


def scaled(ex, ey):
    def mesh():
        xyz, topo = swe.StructTriangMesh(9, 8, 1.0)
        xyz = np.array(xyz)
        xyz[:, 0] = np.ldexp(xyz[:, 0], ex)
        xyz[:, 1] = np.ldexp(xyz[:, 1], ey)
        return xyz, topo
    return mesh


# differences of a scaled mesh are 1 and 1/2 times its scale, up to 2^-400 and 2^400
MESHES = {"mirrored": (mirrored, 1e-3), "mixed": (mixed, 1e-3), "rounded": (rounded, 1e-3),
          "2^-399": (scaled(-399, -399), 2.0**-410), "2^400": (scaled(400, 400), 1e-3),
          "2^-399, 2^400": (scaled(-399, 400), 2.0**-410), "2^-399, 1": (scaled(-399, 0), 2.0**-410),
          "1, 2^400": (scaled(0, 400), 1e-3)}


@pytest.mark.parametrize("flux", ["HLL", "HLLC"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_accepted_coordinates(mesh, flux):
    make, dt = MESHES[mesh]
    xyz, topo = make()
    with np.errstate(all="ignore"):
        prim = state(xyz, topo, 4)
    prim[::5, 1:] = 0.0
    prim[1::5, 1:] = -0.0
    topo = opened(xyz, topo)
    fl = getattr(swe.Fluxes, flux)[swe.Wavespeeds.Davis]
    sd = swe.SpaceDisc(fl, swe.Domain(xyz, topo), prim, cor=0.1)
    assert sd.set_fused(True)
    separate = swe.SpaceDisc(fl, swe.Domain(xyz, topo), prim, cor=0.1)
    separate.set_fused(False)
    orc = O.OracleSolver(xyz, topo.tables(), flux, "Davis", cor=0.1)
    orc.set_state(prim)
    for scheme, step in (("SSPRK2", dt), ("SSPRK3", 0.0)):
        for x in (sd, separate):
            x.run(scheme, 2, dt=step)
        orc.run(scheme, 2, dt=step, cfl=0.15)
        got = sd.GetVolField()
        assert np.isfinite(got).all()
        assert np.array_equal(got, orc.state()), scheme
        assert np.array_equal(got.view(np.int64), separate.GetVolField().view(np.int64)), scheme
