"""Pairs of items per workgroup (split forms, large virtual extents): the
persistent grid runs the same items one at a time, so the per-ijk energies
are equal bit for bit.  Odd and even numbers of items, both spin cases, one
and two W sets, and a range that ends inside a group; at o=5 also a range of
more than a group that starts inside one (43 mixed-spin ijk, in launch order,
a whole group and a part), which for two W sets is cut where the save areas
end (32768 of 43 x 1183 items) and leaves an odd number for the second
launch."""

import os

import numpy as np
import pytest

from libpt_amd import api

pytestmark = pytest.mark.gpu


def _ijk(kind, form, dims, dev, persistent, cut):
    os.environ["LIBPT_AMD_PERSISTENT"] = "1" if persistent else "0"
    with api.Plan(kind, form, dims, dev) as pl:
        for sc in range(pl.ncases):
            n = pl.nijk(sc)
            at = min(cut, n)
            pl.run(sc, 0, at)
            pl.run(sc, at, n)
        return [pl.ijk_energies(sc) for sc in range(pl.ncases)]


@pytest.mark.parametrize("kind,form,dims,cut", [
    ("rpt", "bf16x3", (3, 384), 0), ("rpt", "f16x3", (3, 385), 4),
    ("upt", "bf16x3", (3, 417, 2, 7), 1), ("uft", "f16x3", (3, 391, 2, 9), 0),
    ("rpt", "bf16x3", (5, 385), 7), ("rft", "f16x3", (5, 385), 7)])
def test_pairs_give_the_same_bits(kind, form, dims, cut):
    spec = api.make_spec(kind, dims, seed=5, sig_f=1e-2,
                         omega=0.3 if kind.endswith("ft") else 0.0)
    dev = api.synth_device(kind, spec)
    old = os.environ.get("LIBPT_AMD_PERSISTENT")
    try:
        one = _ijk(kind, form, dims, dev, True, cut)
        two = _ijk(kind, form, dims, dev, False, cut)
    finally:
        if old is None:
            os.environ.pop("LIBPT_AMD_PERSISTENT", None)
        else:
            os.environ["LIBPT_AMD_PERSISTENT"] = old
        dev.close()
    for a, b in zip(one, two):
        assert np.array_equal(a, b)
        assert np.all(np.isfinite(a))
