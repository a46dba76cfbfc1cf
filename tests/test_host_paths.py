"""Host paths of the engine on the CPU: pt_host.cpp and pt_terms.cpp built
with a stand-in for the HIP runtime and the kernel launchers
(tests/c/fake_hip.cpp), in which device memory ends where a test says and a
tile launch leaves 1 + ijk as the energy of each ijk it runs."""

import ctypes
import os
import subprocess
import threading
import time

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
    h.libpt_amd_batch_create.restype = vp
    h.libpt_amd_batch_create.argtypes = [ctypes.c_int] * 3 + [vp] * 2
    h.libpt_amd_batch_destroy.argtypes = [vp]
    h.libpt_amd_batch_energies.argtypes = [vp] * 2
    h.pt_noalloc_energy.restype = ctypes.c_double
    h.pt_noalloc_energy.argtypes = ([ctypes.c_int] * 2 + [sz] * 4 +
                                    [vp, vp, sz, vp])
    h.libpt_amd_energy.restype = ctypes.c_double
    h.libpt_amd_energy.argtypes = [ctypes.c_int] * 2 + [sz] * 4 + [vp] * 2
    h.libpt_rpt.restype = ctypes.c_double
    h.libpt_rpt.argtypes = [sz] * 2 + [vp] * 7
    h.fake_arena.restype = sz
    h.fake_region.restype = vp
    h.fake_region.argtypes = [sz]
    h.fake_region_free.argtypes = [vp, sz]
    h.fake_count.restype = ctypes.c_long
    h.fake_limit.argtypes = [sz]
    return h


@pytest.fixture(autouse=True)
def _memory(lib):
    yield
    lib.fake_limit(1 << 40)


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


@pytest.fixture
def region(lib):
    """scratch of the allocation-free call, as large as its static array"""
    size = lib.fake_arena()
    p = lib.fake_region(size)
    yield p, size
    lib.fake_region_free(p, size)


def _noalloc(lib, call, form, dims, scratch, cap):
    dims = tuple(dims) + (0,) * (4 - len(dims))
    lib.pt_set_error(None)
    return lib.pt_noalloc_energy(call, form, *dims, _arrays(), scratch, cap,
                                 None)


def _expected(lib, dims):
    """the restricted energy of the stand-in: 2 (n (n + 1) / 2) per case"""
    o = dims[0]
    n = (o * (o - 1) * (o - 2) // 6, o * (o - 1) // 2 * o)
    return float(sum(x * (x + 1) for x in n))


def test_plan_without_room_for_the_copies(lib):
    """With less memory than the transposed copies take, the plan is made
    without them, gives the same energies and leaves no error text."""
    dims = (6, 40)
    lib.fake_limit(1 << 40)
    base = lib.fake_count(0)
    full = _plan(lib, RPT, FP64, dims)
    ref = [_ijk(lib, full, 0), _ijk(lib, full, 1)]
    size = lib.fake_count(0) - base
    lib.libpt_amd_plan_destroy(full)
    before = lib.libpt_amd_last_error()
    lib.fake_limit(base + size - 1)
    plan = _plan(lib, RPT, FP64, dims)
    lib.fake_limit(1 << 40)
    assert plan and lib.fake_count(0) - base < 0.8 * size
    assert lib.libpt_amd_last_error() == before
    assert [lib.libpt_amd_plan_run(plan, sc, 0, len(e))
            for sc, e in enumerate(ref)] == [0, 0]
    for sc, e in enumerate(ref):
        assert np.array_equal(_ijk(lib, plan, sc), 1.0 + np.arange(len(e)))
    lib.libpt_amd_plan_destroy(plan)
    assert lib.fake_count(0) == base


def test_drop_in_call_without_room_for_the_copies(lib):
    """The same through pt.h, with an energy that is NaN (inputs of the
    caller): it is returned, and no allocation error ends the program."""
    o, v = 4, 30
    n = [o * v] * 3 + [2 * o * o * v * v, 2 * o * o * v * o,
                       2 * o * o * v * v,
                       o * v * (v * (v - 1) // 2) + o * v * v * v]
    arr = [np.zeros(k) for k in n]
    ptr = [a.ctypes.data for a in arr]
    base = lib.fake_count(0)
    lib.fake_limit(1 << 40)
    assert lib.libpt_rpt(o, v, *ptr) == _expected(lib, (o, v))
    peak = lib.fake_count(1)
    for nan in (0, 1):
        lib.fake_nan(nan)
        lib.fake_limit(peak - 1)
        e = lib.libpt_rpt(o, v, *ptr)
        lib.fake_limit(1 << 40)
        lib.fake_nan(0)
        assert np.isnan(e) if nan else e == _expected(lib, (o, v))
        assert lib.libpt_amd_last_error() == b""
    assert lib.fake_count(0) == base


def test_calls_after_a_device_reset(lib):
    """Streams kept from earlier calls end with the device's other state: a
    later call notices and makes its own."""
    o, v = 3, 8
    n = [o * v] * 3 + [2 * o * o * v * v, 2 * o * o * v * o,
                       2 * o * o * v * v,
                       o * v * (v * (v - 1) // 2) + o * v * v * v]
    arr = [np.zeros(k) for k in n]
    ptr = (ctypes.c_void_p * 7)(*[a.ctypes.data for a in arr])

    def call():
        e = lib.libpt_amd_energy(RPT, FP64, o, v, o, v, ptr, None)
        assert e == _expected(lib, (o, v)), lib.libpt_amd_last_error()

    call()
    made, bad = lib.fake_count(2), lib.fake_count(3)
    call()
    assert lib.fake_count(2) == made
    lib.fake_reset_streams()
    call()
    assert lib.fake_count(2) == made + 1 and lib.fake_count(3) == bad


def test_progress_lines_name_what_was_done(lib, monkeypatch, capfd):
    o, v = 4, 8
    n = [o * v] * 3 + [2 * o * o * v * v, 2 * o * o * v * o,
                       2 * o * o * v * v,
                       o * v * (v * (v - 1) // 2) + o * v * v * v]
    arr = [np.zeros(k) for k in n]
    ptr = (ctypes.c_void_p * 7)(*[a.ctypes.data for a in arr])
    monkeypatch.setenv("LIBPT_AMD_PROGRESS", "1")
    for fail in (0, 1):
        lib.fake_fail_tiles(fail)
        e = lib.libpt_amd_energy(RPT, FP64, o, v, o, v, ptr, None)
        lib.fake_fail_tiles(0)
        lines = capfd.readouterr().err.count("done")
        # 16 parts a spin case; of 4 ijk the first three parts are empty
        assert (np.isnan(e), lines) == ((True, 3) if fail else
                                        (False, 32)), lines


def test_scratch_without_room_for_the_copies(lib, region):
    """The allocation-free call drops the copies where its scratch ends."""
    dims = (6, 40)
    copies = lib.fake_count(5)
    assert _noalloc(lib, RPT, FP64, dims, *region) == _expected(lib, dims)
    assert lib.fake_count(5) > copies
    copies = lib.fake_count(5)
    cap = 8 << 20
    while _noalloc(lib, RPT, FP64, dims, region[0], cap) != _expected(lib,
                                                                      dims):
        assert b"scratch" in lib.libpt_amd_last_error()
        cap += 1 << 20
    assert lib.fake_count(5) == copies
    assert lib.libpt_amd_last_error() == b""


def _batch(lib, call, form, sizes):
    dims = np.array([(o, v, o, v) for o, v in sizes], dtype=np.int64)
    return lib.libpt_amd_batch_create(call, form, len(sizes),
                                      dims.ctypes.data,
                                      _arrays(10 * len(sizes)))


@pytest.mark.parametrize("call,form", [(RPT, FP64), (RFT, F16X3)])
def test_batch_without_room_for_the_copies(lib, monkeypatch, call, form):
    """Wherever memory ends, a batch that fits without the transposed copies
    is made; one that does not is refused, and nothing stays allocated."""
    sizes = [(5, 40), (4, 33), (6, 64), (3, 20)]
    base = lib.fake_count(0)

    def size():
        lib.fake_limit(1 << 40)
        b = _batch(lib, call, form, sizes)
        used = lib.fake_count(0) - base
        lib.libpt_amd_batch_destroy(b)
        return used

    full = size()
    monkeypatch.setenv("LIBPT_AMD_VC_TRANSPOSED", "0")
    bare = size()
    monkeypatch.delenv("LIBPT_AMD_VC_TRANSPOSED")
    assert bare < 0.9 * full
    for q in range(21):
        before = lib.libpt_amd_last_error()
        lib.fake_limit(base + bare + (full - bare) * q // 20)
        b = _batch(lib, call, form, sizes)
        assert b and lib.libpt_amd_last_error() == before, q
        e = np.zeros(len(sizes))
        assert lib.libpt_amd_batch_energies(b, e.ctypes.data) == 0
        assert list(e) == [_expected(lib, s) for s in sizes]
        lib.libpt_amd_batch_destroy(b)
    lib.fake_limit(base + bare - 1)
    assert not _batch(lib, call, form, sizes)
    assert b"hipMalloc" in lib.libpt_amd_last_error()
    lib.fake_limit(1 << 40)
    assert lib.fake_count(0) == base


def test_save_areas_of_a_batch_fit_its_largest_launch(lib):
    """24 small (fT) systems: spin cases share launches of up to 8192 items, so
    that many areas of 128 KB beside the systems' own 75 MB each, and not one
    for each of the batch's items."""
    sizes = [(6, 64)] * 24
    base = lib.fake_count(0)
    tiles = lib.fake_count(7)
    b = _batch(lib, RFT, FP64, sizes)
    assert b and lib.fake_count(7) > tiles
    assert lib.fake_count(0) - base < (8192 << 17) + 24 * (76 << 20)
    e = np.zeros(len(sizes))
    assert lib.libpt_amd_batch_energies(b, e.ctypes.data) == 0
    assert list(e) == [_expected(lib, s) for s in sizes]
    lib.libpt_amd_batch_destroy(b)


@pytest.mark.parametrize("call,dims,plain,transposed", [
    (RPT, (4, 5), 4, 3), (RPT, (2, 5), 4, 2), (UPT, (4, 5, 3, 6), 8, 6),
    # no case reads the second spin's own blocks: its pairs have no orbitals
    (UPT, (2, 2, 50, 1), 4, 2), (UPT, (1, 5, 4, 6), 4, 3),
    (UPT, (2, 1, 1, 5), 0, 0), (UFT, (4, 5, 1, 1), 8, 6)])
def test_only_blocks_that_a_case_reads_are_packed(lib, call, dims, plain,
                                                  transposed):
    a, b = lib.fake_count(4), lib.fake_count(5)
    plan = _plan(lib, call, FP64, dims)
    assert plan
    lib.libpt_amd_plan_destroy(plan)
    assert (lib.fake_count(4) - a, lib.fake_count(5) - b) == (plain,
                                                              transposed)


# sizes at the limit, from one virtual orbital of a spin up, and what they were
# taken with before rows were padded: 16-fold for one orbital
@pytest.mark.parametrize("call,form,dims", [
    (UPT, FP64, (2, 2, 5770, 1)), (UFT, FP64, (1825, 1, 69, 19)),
    (UFT, FP64, (3641, 1, 36, 2)), (UFT, FP64, (1, 1, 1896, 2)),
    (UFT, FP32, (2, 2, 5752, 1)), (UPT, BF16X3, (1, 3, 257, 3)),
    (UFT, FP64, (1, 13, 206, 17)), (UFT, FP64, (1, 33, 179, 17)),
    (RPT, FP32, (259, 8)), (RPT, FP64, (8, 134)), (RFT, F16X3, (31, 64))])
def test_sizes_at_the_limit_fit_the_scratch(lib, region, call, form, dims):
    e = _noalloc(lib, call, form, dims, *region)
    assert lib.libpt_amd_last_error() == b"" and np.isfinite(e)


@pytest.mark.parametrize("call,form,dims", [
    (UPT, FP64, (2, 2, 5771, 1)), (UFT, FP64, (1, 13, 207, 17)),
    (RPT, FP64, (9, 134)), (RFT, F16X3, (32, 64))])
def test_sizes_beyond_the_limit_are_refused(lib, region, call, form, dims):
    assert np.isnan(_noalloc(lib, call, form, dims, *region))
    assert b"%d bytes of static scratch" % (256 << 20) in \
        lib.libpt_amd_last_error()


@pytest.mark.parametrize("call,dims", [(RPT, (10, 100000)),
                                       (UFT, (1 << 20, 1 << 20, 9, 7))])
def test_far_too_large_sizes_are_refused_at_once(lib, region, call, dims):
    t0 = time.monotonic()
    assert np.isnan(_noalloc(lib, call, FP64, dims, *region))
    assert time.monotonic() - t0 < 1.0
    assert b"static scratch" in lib.libpt_amd_last_error()


def test_copies_leave_room_for_save_areas(lib, region):
    """(fT): a launch holds as many items as there are save areas, so the
    copies are left out where they would take the room of these: more
    scratch never means more launches."""
    most = None
    for cap in list(range(60 << 20, 400 << 20, 4 << 20)) + [region[1]]:
        tiles = lib.fake_count(7)
        if not np.isnan(_noalloc(lib, RFT, FP64, (6, 64), region[0], cap)):
            launches = lib.fake_count(7) - tiles
            assert most is None or launches <= most, cap
            most = launches
    assert most == 1


@pytest.mark.parametrize("form,dims,width,ordered", [
    (FP64, (12, 200), 64, 1), (BF16X3, (12, 64), 40, 1),
    (FP64, (12, 200), 32, 0),              # one group
    (FP64, (60, 8), 256, 0), (FP32, (60, 24), 500, 0),
    (BF16X3, (45, 48), 40, 0), (BF16X3, (45, 48), 2000, 1)])
def test_short_ranges_of_long_lists_go_in_list_order(lib, form, dims, width,
                                                     ordered):
    """Picking a range's launch order walks the whole list: only where the
    range's work outweighs that.  Either way each ijk runs once."""
    plan = _plan(lib, RPT, form, dims)
    n, made = lib.libpt_amd_plan_nijk(plan, 1), lib.fake_count(6)
    b = n // 3 + 1
    assert lib.libpt_amd_plan_run(plan, 1, b, b + width) == 0
    got = _ijk(lib, plan, 1)
    lib.libpt_amd_plan_destroy(plan)
    assert lib.fake_count(6) - made == ordered
    want = np.zeros(n)
    want[b:b + width] = 1.0 + np.arange(b, b + width)
    assert np.array_equal(got, want)


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
