"""Host paths of the engine on the CPU: pt_host.cpp and pt_terms.cpp built
with a stand-in for the HIP runtime and the kernel launchers
(tests/c/fake_hip.cpp), in which device memory ends where a test says and a
tile launch leaves 1 + ijk as the energy of each ijk it runs."""

import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "libpt_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
RPT, UPT, RFT, UFT = range(4)
FP64, FP32, BF16X3, F16X3 = range(4)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "host.so")
    subprocess.run(
        ["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wl,-Bsymbolic",
         "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
         "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
         os.path.join(ROOT, "tests", "c", "fake_hip.cpp"),
         os.path.join(CSRC, "pt_host.cpp"), os.path.join(CSRC, "pt_terms.cpp"),
         "-lpthread", "-o", out], check=True)
    h = ctypes.CDLL(out)
    vp, i64, sz = ctypes.c_void_p, ctypes.c_int64, ctypes.c_size_t
    h.libpt_amd_plan_create.restype = vp
    h.libpt_amd_plan_create.argtypes = [ctypes.c_int] * 2 + [sz] * 4 + [vp]
    h.libpt_amd_plan_destroy.argtypes = [vp]
    h.libpt_amd_plan_nijk.restype = i64
    h.libpt_amd_plan_nijk.argtypes = [vp, ctypes.c_int]
    h.libpt_amd_plan_run.argtypes = [vp, ctypes.c_int, i64, i64]
    h.libpt_amd_plan_ijk_energies.argtypes = [vp, ctypes.c_int, vp]
    h.libpt_amd_last_error.restype = ctypes.c_char_p
    h.fake_count.restype = ctypes.c_long
    h.fake_limit.argtypes = [sz]
    yield h
    h.fake_limit(1 << 40)


def _arrays(n=10):
    """device pointers that nothing reads"""
    return (ctypes.c_void_p * n)(*[4096] * n)


def _plan(lib, call, form, dims):
    dims = tuple(dims) + (0,) * (4 - len(dims))
    return lib.libpt_amd_plan_create(call, form, *dims, _arrays())


def _ijk(lib, plan, sc):
    e = np.zeros(lib.libpt_amd_plan_nijk(plan, sc))
    assert lib.libpt_amd_plan_ijk_energies(plan, sc, e.ctypes.data) == 0
    return e


def test_ranges_of_one_plan_from_two_threads(lib):
    """Both threads make the launch order of their range before either runs
    its tiles, unless a range is one unit."""
    plan = _plan(lib, RPT, FP64, (12, 200))
    n = lib.libpt_amd_plan_nijk(plan, 1)
    cut = n // 3
    rc = []
    lib.fake_meet(2)
    th = [threading.Thread(target=lambda r: rc.append(
        lib.libpt_amd_plan_run(plan, 1, *r)), args=(r,))
        for r in ((0, cut), (cut, n))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    lib.fake_meet(0)
    assert rc == [0, 0]
    got = _ijk(lib, plan, 1)
    lib.libpt_amd_plan_destroy(plan)
    assert np.array_equal(got, 1.0 + np.arange(n))
