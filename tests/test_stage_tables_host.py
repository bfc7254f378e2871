"""Tables of the stage kernels' tiles and the LDS that a tile takes, checked on
the host (tests/cpp/stage_tables_check.cpp): every local index names the mesh's
own cell, node and edge, and meshes whose tiles have long borders keep the
workgroups per CU that the gathering kernel before them had."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import swe_fvm_amd as swe

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CU = 160 * 1024


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stage") / "libstage_check.so")
    res = subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-pthread", "-Wall", "-Wextra",
                          os.path.join(ROOT, "tests", "cpp", "stage_tables_check.cpp"),
                          os.path.join(ROOT, "swe_fvm_amd", "csrc", "swe_tiles.cpp"), "-o", out],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return ctypes.CDLL(out)


def check(lib, topo):
    t = topo.tables()
    T = t["tp"].shape[0]
    c = lambda a, ty=np.int32: np.ascontiguousarray(a, dtype=ty)
    et0 = c(t["et"][:, 0])
    fl = np.zeros(T, np.uint32)
    for k in range(3):
        fl |= (et0[t["te"][:, k]] == np.arange(T)).astype(np.uint32) << k
    args = [c(t["tp"].T), c(t["tt"].T), c(t["te"].T), fl, et0, c(t["et"][:, 1]), c(t["ep"][:, 0]), c(t["ep"][:, 1])]
    out = np.zeros(7, np.int64)
    msg = ctypes.create_string_buffer(128)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    rc = lib.stage_tables_check(ctypes.c_int64(T), *[p(a) for a in args], p(out), msg, 128)
    assert rc == 0, msg.value.decode()
    return out


def scattered(n, k):
    """A Morton-ordered mesh with k cells moved to its end."""
    xyz, topo = swe.jittered_mesh(n, 0.25, 8)
    T = topo.NumTriangles()
    idx = np.random.default_rng(0).choice(T, k, replace=False)
    dom = swe.reorder_cells(swe.Domain(xyz, topo), np.concatenate([np.setdiff1d(np.arange(T), idx), idx]))
    return (dom[0] if isinstance(dom, tuple) else dom).topology


MESHES = {"one square": lambda: swe.StructTriangMesh(1, 1, 0.1)[1], "rows7": lambda: swe.StructTriangMesh(100, 7, 0.1)[1],
          "jittered": lambda: swe.jittered_mesh(61, 0.3, 2)[1], "rows300": lambda: swe.StructTriangMesh(300, 300, 0.1)[1],
          "rows185": lambda: swe.StructTriangMesh(185, 180, 0.1)[1], "jittered300": lambda: swe.jittered_mesh(300, 0.3, 8)[1],
          "scattered": lambda: scattered(300, 73)}


@pytest.mark.parametrize("mesh", list(MESHES))
def test_tables_and_lds(lib, mesh):
    tiles, *lds = check(lib, MESHES[mesh]())
    for whole, far, is_far in (lds[:3], lds[3:]):
        print(f"{mesh}: {tiles} tiles, {whole} B whole, {far} B far, far {is_far}")
        taken = far if is_far else whole
        assert far <= whole and taken <= 64 * 1024
        # three workgroups to a CU, or every tile on the chip at once
        assert taken * 3 <= CU or tiles <= 256 * (CU // taken)


def test_morton_ordered_tiles_are_staged_whole(lib):
    _, *lds = check(lib, MESHES["jittered300"]())
    assert lds[0] <= CU // 4 and not lds[2] and not lds[5]


@pytest.mark.parametrize("mesh", ["rows300", "rows185", "scattered"])
def test_long_tiles_leave_the_cells_beyond_the_ring_out(lib, mesh):
    _, *lds = check(lib, MESHES[mesh]())
    assert lds[2] and lds[5]
