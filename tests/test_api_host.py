"""The library's host code over a device that is host memory
(tests/cpp/api_on_host.cpp): what it does where a launch fails, where threads
meet, and over sequences of calls."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"
EULER, SSPRK2, SSPRK3 = 0, 1, 2


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(os.path.join(HIP, "hip", "hip_runtime.h")):
        pytest.skip("no HIP headers")
    out = str(tmp_path_factory.mktemp("api") / "libapi_on_host.so")
    src = os.path.join(ROOT, "swe_fvm_amd", "csrc")
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                          "-Wl,-z,lazy", "-Wl,-Bsymbolic", "-I", HIP, os.path.join(ROOT, "tests", "cpp", "api_on_host.cpp"),
                          os.path.join(src, "swe_mesh.cpp"), os.path.join(src, "swe_tiles.cpp"), "-o", out],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return ctypes.CDLL(out, mode=os.RTLD_LAZY | os.RTLD_LOCAL)


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("scheme, fused, launch", [(EULER, 1, "flux"), (EULER, 1, "fused"), (SSPRK2, 1, "fused"),
                                                   (SSPRK2, 0, "flux"), (SSPRK3, 0, "drain"), (SSPRK2, 0, "update"),
                                                   (SSPRK2, 1, "recon1"), (SSPRK2, 1, "recon2")])
def test_a_failed_launch_leaves_no_longer_list(lib, scheme, fused, launch, graph):
    lib.list_after_failed_launch.restype = ctypes.c_int64
    cells = ctypes.c_int64()
    longest = lib.list_after_failed_launch(launch.encode(), scheme, fused, graph, ctypes.byref(cells))
    assert cells.value == 192 and longest == cells.value


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("layouts", range(5))
def test_euler_ensembles_after_layout_changes(lib, layouts, graph):
    lib.euler_steps_after_layouts.restype = ctypes.c_int64
    for runs, steps in ((1, 6), (2, 3), (1, 67)):
        assert lib.euler_steps_after_layouts(layouts, graph, runs, ctypes.c_int64(steps)) == runs * steps


@pytest.mark.parametrize("kind", [0, 1, 2], ids=["hipMalloc", "hipFree of a destroyed solver", "hipFree of memory given back"])
def test_solvers_do_not_wait_for_each_others_device_calls(lib, kind):
    assert lib.other_solver_goes_on(kind) == 1


def test_kept_memory_is_given_back(lib):
    kept = (ctypes.c_int64 * 5)()
    assert lib.kept_bytes(3, kept) == 0
    assert kept[0] == 3 * 256 and list(kept)[1:] == [256, 0, 3 * 256, 0]


@pytest.mark.parametrize("n, two", [(10, 1), (147, 1), (148, 2)])  # 129,948 and 131,720 edges
def test_the_tuning_that_is_read_can_be_set_again(lib, n, two):
    items, got = (ctypes.c_int * 5)(), (ctypes.c_int * 5)()
    assert lib.flux_items_launched(n, items, got) == 0
    assert list(got) == [2, 2, 4, 2, 1]
    assert list(items) == [two, two, 4, two, 1]


@pytest.mark.parametrize("layout", [0, 64, 8, 1])
@pytest.mark.parametrize("n, launches", [(1, 0), (10, 0), (74, 0), (75, 2), (80, 2)])  # 21,904 and 22,500 cells
def test_small_states_cross_without_a_launch(lib, n, launches, layout):
    assert lib.launches_of_a_crossing(n, layout) == launches
