"""Launch order of the ijk: whole lists and ranges of every length relative
to a group (32), starting anywhere, run each ijk once; every range leaves the
other energies alone and gives the whole list's per-ijk energies bit for
bit (the order only decides which items run together).  At small sizes the
ranges go in list order, at larger ones in the launch order picked out of the
list's."""

import numpy as np
import pytest

from libpt_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dims", [("rpt", (11, 20)), ("upt", (9, 17, 6, 19)),
                                       ("rft", (9, 18))])
def test_ranges_run_every_ijk_once(kind, dims):
    _ranges(kind, "fp64", dims)


@pytest.mark.parametrize("kind,form,dims", [
    ("rpt", "fp64", (9, 65)), ("rpt", "fp32", (9, 70)),
    ("upt", "bf16x3", (8, 48, 6, 50)), ("uft", "f16x3", (7, 50, 8, 47))])
def test_ordered_ranges_run_every_ijk_once(kind, form, dims):
    _ranges(kind, form, dims)


def _ranges(kind, form, dims):
    spec = api.make_spec(kind, dims, seed=3, sig_f=1e-2)
    dev = api.synth_device(kind, spec, fp32=form == "fp32")
    try:
        with api.Plan(kind, form, dims, dev) as pl:
            pl.run_all()
            ref = [pl.ijk_energies(sc) for sc in range(pl.ncases)]
        for sc in range(len(ref)):
            n = len(ref[sc])
            ranges = [(0, 1), (0, 31), (3, 35), (1, 34), (5, 38), (7, n),
                      (0, n - 1), (n - 33, n), (0, n)]
            for b, e in ranges:
                b, e = max(0, min(b, n)), min(e, n)
                with api.Plan(kind, form, dims, dev) as pl:
                    pl.run(sc, b, e)
                    got = pl.ijk_energies(sc)
                want = np.zeros(n)
                want[b:e] = ref[sc][b:e]
                assert np.array_equal(got, want), (sc, b, e)
    finally:
        dev.close()
