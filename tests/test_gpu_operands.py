"""Operand fragments of the tile kernel at the edges of their tiles.

- Sizes on both sides of the 16-row blocks, the 4- and 8-wide parts of the c
  range, the 32-wide tiles and the kappa chunks (8 or 16), the smallest ones
  included, in every form: tiles cut by the diagonal and by the end of every
  index skip the blocks outside the triangle and read only fragments that
  exist.  Bounds: FP64 as for the other parity tests; FP32 and the split
  forms by their operand precision (FP32 2^-24, split 2^-16 per product).
- Open-shell sizes with fewer orbitals than a 16-row block in one spin or
  both, down to spin cases that do not exist.
- Without the transposed copies (LIBPT_AMD_VC_TRANSPOSED=0, or too little
  memory for them) the same values come from the plain copies in scattered
  pieces: per-ijk energies are equal bit for bit."""

import ctypes
import os

import numpy as np
import pytest

import oracle
from libpt_amd import api

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5, "bf16x3": 1e-4, "f16x3": 1e-4}
SIZES = [(3, 3), (4, 8), (3, 15), (5, 16), (4, 17), (3, 20), (9, 32), (4, 33),
         (3, 36), (17, 24), (3, 47), (4, 48), (3, 49), (3, 65)]


def _energy(kind, form, dims, dev):
    with api.Plan(kind, form, dims, dev) as pl:
        pl.run_all()
        return pl.energy(), [pl.ijk_energies(sc) for sc in range(pl.ncases)]


@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16x3", "f16x3"])
@pytest.mark.parametrize("dims", SIZES, ids=[f"{o}x{v}" for o, v in SIZES])
def test_tile_edges_match_the_oracle(dims, form):
    spec = api.make_spec("rpt", dims, seed=sum(dims), sig_f=1e-2)
    arr = api.synth_host("rpt", spec)
    eo = oracle.energy("rpt", dims, arr, mp=form == "fp32")
    dev = api.to_device("rpt", arr, fp32=form == "fp32")
    try:
        e, _ = _energy("rpt", form, dims, dev)
    finally:
        dev.close()
    print(dims, form, e, eo)
    assert abs(e - eo) <= TOL[form] * abs(eo)


# energies of a few 1e-5 to 1e-1, summed from terms of both signs: the bounds
# above, on the sum of the per-ijk energies' sizes
@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16x3", "f16x3"])
@pytest.mark.parametrize("copies", ["1", "0"])
@pytest.mark.parametrize("kind,dims", [
    ("upt", (2, 2, 5, 1)), ("upt", (3, 1, 4, 3)), ("upt", (1, 5, 4, 6)),
    ("uft", (5, 17, 2, 1)), ("uft", (3, 1, 5, 2)), ("upt", (3, 3, 4, 2)),
    ("uft", (4, 7, 3, 9)), ("upt", (3, 15, 4, 8)), ("uft", (3, 9, 3, 16)),
    ("upt", (6, 4, 2, 21))])
def test_few_orbitals_match_the_oracle(kind, dims, copies, form, monkeypatch):
    monkeypatch.setenv("LIBPT_AMD_VC_TRANSPOSED", copies)
    spec = api.make_spec(kind, dims, seed=sum(dims), sig_f=1e-2,
                         omega=0.3 if kind == "uft" else 0.0)
    arr = api.synth_host(kind, spec)
    eo = oracle.energy(kind, dims, arr, mp=form == "fp32")
    dev = api.to_device(kind, arr, fp32=form == "fp32")
    try:
        e, ijk = _energy(kind, form, dims, dev)
    finally:
        dev.close()
    size = sum(float(np.sum(np.abs(x))) for x in ijk)
    print(kind, dims, form, copies, e, eo, size)
    assert abs(e - eo) <= TOL[form] * size


@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16x3", "f16x3"])
@pytest.mark.parametrize("kind,dims", [
    ("rpt", (5, 45)), ("upt", (4, 33, 5, 20)), ("uft", (4, 18, 3, 37))])
def test_plain_copies_give_the_same_bits(kind, dims, form):
    spec = api.make_spec(kind, dims, seed=7, sig_f=1e-2,
                         omega=0.3 if kind == "uft" else 0.0)
    dev = api.synth_device(kind, spec, fp32=form == "fp32")
    old = os.environ.get("LIBPT_AMD_VC_TRANSPOSED")
    try:
        e0, ijk0 = _energy(kind, form, dims, dev)
        os.environ["LIBPT_AMD_VC_TRANSPOSED"] = "0"
        e1, ijk1 = _energy(kind, form, dims, dev)
    finally:
        if old is None:
            os.environ.pop("LIBPT_AMD_VC_TRANSPOSED", None)
        else:
            os.environ["LIBPT_AMD_VC_TRANSPOSED"] = old
        dev.close()
    assert e0 == e1
    for a, b in zip(ijk0, ijk1):
        assert np.array_equal(a, b)


class _PackJob(ctypes.Structure):
    """struct pt_pack_job of the engine"""
    _fields_ = ([("src", ctypes.c_void_p), ("dst", ctypes.c_void_p)] +
                [(n, ctypes.c_int64) for n in ("R", "K", "rows", "cols")] +
                [("scale", ctypes.c_double), ("at", ctypes.c_int64)] +
                [(n, ctypes.c_int32) for n in ("tri", "tr", "fr")])


def test_more_slabs_than_one_launch_packs():
    """More workgroups than a launch can hold (2^24 of 256 threads): the job
    goes in runs, and the slabs at the ends of these arrive."""
    lib = api.lib()
    slabs, rows = (1 << 24) + 70, 2
    src = lib.libpt_amd_dev_alloc(8 * slabs * rows)
    dst = lib.libpt_amd_dev_alloc(64 * slabs * rows)
    assert src and dst
    try:
        first = [0, (1 << 24) - 8, slabs - 8]
        for s in first:
            x = (1.0 + np.arange(8 * rows)) + 1000.0 * s
            assert lib.libpt_amd_memcpy(src + 8 * rows * s, x.ctypes.data,
                                        x.nbytes, 1) == 0
        job = _PackJob(src=src, dst=dst, R=slabs, K=1, rows=rows, cols=1,
                       scale=1.0)
        print("pack", slabs, "slabs", flush=True)
        assert lib.pt_launch_pack(ctypes.byref(job), 1, 0, None) == 0
        for s in first:
            # a fragment: four quarters of 2 rows, the first kappa of the
            # first quarter is the only one
            got = api.from_device(dst + 64 * rows * s, 8 * 8 * rows)
            want = np.zeros((8, 4, rows, 2))
            want[:, 0, :, 0] = (1.0 + np.arange(8 * rows) + 1000.0 * s
                                ).reshape(8, rows)
            assert np.array_equal(got, want.ravel()), s
    finally:
        lib.libpt_amd_dev_free(src)
        lib.libpt_amd_dev_free(dst)
