"""Device memory kept between the adjoint, tangent and diagnostic calls of a
solver: every call's results are those of a solver that makes it first, in
any order of calls and sizes, on several threads, and past the kept size."""
import threading

import numpy as np
import pytest

import swe_fvm_amd as swe
from tests import _common as C

pytestmark = pytest.mark.gpu


def _solver(n, seed):
    xyz, topo, prim = C.wet_dry_mesh(n, seed=seed)
    fl = swe.Fluxes.HLLC[swe.Wavespeeds.Einfeldt]
    return swe.SpaceDisc(fl, swe.Domain(xyz, topo), prim, device=0), prim


CALLS = {
    "stats": lambda sd, p, g: tuple(sd.Stats().values()),
    "totals": lambda sd, p, g: sd.Integrals(),
    "cells": lambda sd, p, g: sd.Integrals(per_cell=True)[1],
    "adjoint3": lambda sd, p, g: sd.adjoint_run(g, 3, dt=1e-4, checkpoint_every=2)[:2],
    "adjoint9": lambda sd, p, g: sd.adjoint_run(g, 9, dt=1e-4, checkpoint_every=9)[:2],
    "tangent": lambda sd, p, g: sd.tangent_run(g, 2, z_dot=None, dt=1e-4)[0],
}


def _one(sd, prim, bar, name):
    sd.SetVolField(prim)
    return [np.array(x) for x in np.atleast_1d(CALLS[name](sd, prim, bar))] if name in ("stats", "totals") else \
        [np.array(x) for x in (lambda r: r if isinstance(r, tuple) else (r,))(CALLS[name](sd, prim, bar))]


def _equal(a, b):
    return len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))


def _order(n, seed, out):
    sd, prim = _solver(n, seed)
    bar = np.random.default_rng(seed).standard_normal(prim.shape)
    ref = {}
    for name in CALLS:
        ref[name] = _one(_solver(n, seed)[0], prim, bar, name)
    bad = []
    for name in ["stats", "adjoint3", "cells", "adjoint9", "tangent", "totals", "adjoint3", "stats", "cells", "adjoint9"]:
        if not _equal(_one(sd, prim, bar, name), ref[name]):
            bad.append(name)
    out[n] = bad


@pytest.mark.parametrize("sizes", [(5,), (40,), (16, 33, 60)])
def test_calls_in_any_order_equal_a_fresh_solver(sizes):
    out = {}
    th = [threading.Thread(target=_order, args=(n, 3 + k, out)) for k, n in enumerate(sizes)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert out == {n: [] for n in sizes}


def test_a_call_larger_than_what_is_kept():
    # 1,400 SSP-RK2 steps of 80,000 cells in one segment: about 20 GB
    sd, prim = _solver(200, 2)
    bar = np.random.default_rng(0).standard_normal(prim.shape)
    res = []
    for k in (50, 1400, 50):
        sd.SetVolField(prim)
        res.append(sd.adjoint_run(bar, 1400, dt=1e-5, checkpoint_every=k)[:2])
    for r in res[1:]:
        assert np.array_equal(r[0], res[0][0]) and np.array_equal(r[1], res[0][1])
