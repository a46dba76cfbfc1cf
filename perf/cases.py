"""Performance cases of the perturbative-triples engine: what its users have
it compute, through the public entry points of ``libpt_amd.api``.

Four ways in:

* ``call``: one pt.h call on host arrays (``libpt_rpt`` and family, their
  ``_mp`` variants, or ``libpt_amd_energy`` for the split forms), copies to
  the GPU and operand packing included;
* ``noalloc``: one allocation-free call on device-resident inputs;
* ``plan``: a kept plan over device-resident inputs, run over a range of
  the occupied triples of each spin case (all of them at small sizes; a
  share at large ones, as a job that splits the work list runs it);
* ``batch``: a kept batch of independent systems, one graph launch.

The inputs obey the relations that coupled-cluster programs give theirs:
antisymmetric same-spin blocks, closed-shell relations of the restricted
blocks, orbital-energy denominators, and for (fT) left amplitudes and
integrals that resemble the right ones.
"""

import math
import random

import numpy as np
import torch

from libpt_amd import api

SIG_T1, SIG_T2, SIG_INT, SIG_F = 1e-2, 1e-2, 5e-2, 1e-2
OMEGA = 0.3          # excitation energy folded into the (fT) denominators
LIKE = 0.8           # share of the right operands in the left ones

# flops of a pass of the largest cases, by form (0.2 to 0.3 s each)
MOST_FLOPS = {"fp64": 1.2e13, "fp32": 2.4e13, "bf16x3": 3.6e13,
              "f16x3": 3.6e13}
MOST_BYTES = 14e9    # inputs of one system


def listed():
    return [
        # a molecule in a minimal basis (the size of a known-answer input):
        # the whole call is launches, copies and host work
        _case("tiny rpt call", "call", "rpt", "fp64", (5, 19)),
        # the smallest open-shell excited-state call, single precision
        _case("tiny uft_mp call", "call", "uft", "fp32", (7, 3, 6, 4)),
        # a small molecule evaluated over and over on inputs that another
        # GPU code leaves in device memory
        _case("noalloc rpt 8/64", "noalloc", "rpt", "fp64", (8, 64)),
        # the same size in the mixed-precision form, per-triple energies
        # read back for a local analysis
        _case("plan rpt 8/64 bf16x3", "plan", "rpt", "bf16x3", (8, 64),
              per_ijk=True),
        # ordinary closed-shell molecule, from the coupled-cluster
        # program's host arrays
        _case("call rpt 20/120", "call", "rpt", "fp64", (20, 120)),
        # the single-precision drop-in at an odd virtual size
        _case("call rpt_mp 24/101", "call", "rpt", "fp32", (24, 101)),
        # the basis of the nine-water benchmark (v = 477) in double
        # precision, a share of the triples
        _case("plan rpt 10/477", "plan", "rpt", "fp64", (10, 477), ijk=22,
              at=0.4),
        # and in the split form that is there for this size
        _case("plan rpt 10/477 bf16x3", "plan", "rpt", "bf16x3", (10, 477),
              ijk=64, at=0.4, per_ijk=True),
        # open-shell radical, single precision, a share of four spin cases
        _case("plan upt 24/200 fp32", "plan", "upt", "fp32",
              (24, 200, 20, 204), ijk=420, at=0.25),
        # closed-shell excited state, split FP16
        _case("plan rft 12/300 f16x3", "plan", "rft", "f16x3", (12, 300),
              ijk=80, at=0.2),
        # open-shell excited state in double precision
        _case("plan uft 16/160 fp64", "plan", "uft", "fp64",
              (16, 160, 14, 160), ijk=200, at=0.5, per_ijk=True),
        # a set of small molecules (o 4 to 20, v 40 to 160) in one launch
        _case("batch rpt", "batch", "rpt", "fp64", (12, 100), n=8, sizes=64),
    ]


def draw(rng):
    """One more case: entry, call, form and sizes drawn over their ranges,
    the pass held to the flops of the largest listed cases."""
    entry = rng.choice(["call", "call", "noalloc", "plan", "plan", "plan",
                        "plan", "batch"])
    kind = rng.choice(["rpt", "rpt", "upt", "rft", "uft"])
    form = rng.choice(["fp64", "fp64", "fp32", "bf16x3", "f16x3"])
    if entry == "batch":
        return _case(None, entry, kind, form, (12, 100), n=rng.randint(4, 10),
                     sizes=rng.randrange(1 << 20))
    if entry == "call":
        o, v = _log(rng, 3, 24), _log(rng, 3, 160)
    elif entry == "noalloc":
        o, v = _log(rng, 3, 9), _log(rng, 8, 70)
    else:
        o, v = _log(rng, 6, 30), _log(rng, 40, 477)
    dims = (o, v)
    if kind in ("upt", "uft"):
        dims = (o, v, max(1, o - rng.randint(0, 3)), v + rng.randint(0, 4))
    while _input_bytes(kind, form, dims) > MOST_BYTES / (
            10 if entry == "call" else 2 if kind in ("rft", "uft") else 1):
        dims = _shrink(dims)
    if entry == "noalloc" and kind in ("rft", "uft"):
        dims = tuple(min(d, 45) for d in dims)
    if entry != "plan":
        while _flops(kind, dims) > MOST_FLOPS[form] / 3:
            dims = _shrink(dims)
        return _case(None, entry, kind, form, dims)
    per = sum(f for _, f in _per_ijk(kind, dims))
    ijk = max(1, int(MOST_FLOPS[form] * rng.uniform(0.2, 0.9) / per))
    return _case(None, entry, kind, form, dims, ijk=min(ijk, 100000),
                 at=round(rng.random(), 3), per_ijk=rng.random() < 0.5)


def prepare(case, seed):
    """Inputs of the seed; for plans and batches also the plan or batch."""
    return State(case, seed)


def run(state):
    """One pass: the energy (and per-triple energies) it computes."""
    c = state.case
    if c["entry"] == "call":
        if c["form"] in ("fp64", "fp32"):
            e = api.dropin(c["kind"], state.dims, state.arrays,
                           mp=c["form"] == "fp32")
        else:
            e = api.energy(c["kind"], c["form"], state.dims, state.arrays)
        return {"energy": np.array([e])}
    if c["entry"] == "noalloc":
        e = api.energy_noalloc(c["kind"], c["form"], state.dims, state.dev)
        return {"energy": np.array([e])}
    if c["entry"] == "batch":
        state.batch.run()
        return {"energy": state.batch.energies()}
    plan = state.plan
    for sc, (b, e) in enumerate(state.ranges):
        plan.run(sc, b, e)
    out = {"energy": np.array([plan.energy()])}
    if c["per_ijk"]:
        out["ijk"] = [plan.ijk_energies(sc)[b:e]
                      for sc, (b, e) in enumerate(state.ranges)]
    return out


def work(case):
    """Inputs that the pass touches, read once, and its energies, written
    once; multiply-adds of the contractions, as libpt counts its GEMMs."""
    if case["entry"] == "batch":
        dims = _batch_dims(case)
        return {"bytes": sum(_input_bytes(case["kind"], case["form"], d)
                             for d in dims) + 8.0 * len(dims),
                "flops": sum(_flops(case["kind"], d) for d in dims)}
    kind, dims = case["kind"], _dims(case)
    nbytes = _input_bytes(kind, case["form"], dims)
    if case["entry"] != "plan":
        return {"bytes": nbytes + 8.0, "flops": _flops(kind, dims)}
    ranges = _ranges(case)
    oa, va, ob, vb = _four(kind, dims)
    used = set()
    n = 0
    for (same, sp), (b, e) in zip(_spin_cases(kind), ranges):
        o1, o2 = (oa, ob) if sp == 0 else (ob, oa)
        for i, j, k in _triples(same, o1, o2)[b:e]:
            used |= {(sp, i), (sp, j), (sp if same else 1 - sp, k)}
        n += e - b
    if kind in ("rpt", "rft"):   # one set of slabs for both spins
        used = {(0, i) for _, i in used}
    share = len(used) / (oa if kind in ("rpt", "rft") else oa + ob)
    flops = sum((e - b) * f for (b, e), (_, f) in
                zip(ranges, _per_ijk(kind, dims)))
    return {"bytes": nbytes * share + 8.0 * (n + 1), "flops": flops}


def tolerance(case):
    """Above what was measured against 64 bits over the ranges: FP64 1e-16
    to 1e-15, FP32 up to 1e-8, split BF16 and FP16 up to 1.1e-7 (per-triple
    energies of the smallest sizes; the energies of larger ones average
    their elements' rounding down)."""
    return {"fp64": {"rel": 1e-13}, "fp32": {"rel": 1e-6},
            "bf16x3": {"rel": 1e-6}, "f16x3": {"rel": 1e-6}}[case["form"]]


def exact(case, seed):
    """The energies from torch in 64 bits; None where that takes long."""
    if case["entry"] == "batch":
        dims = _batch_dims(case)
        if sum(_flops(case["kind"], d) for d in dims) > 2e13:
            return None
        es = []
        for n, d in enumerate(dims):
            arrays = _inputs(case["kind"], d, _sub(seed, n), case["form"])
            es.append(_energies(case["kind"], d, arrays, None)[0])
        return {"energy": np.array(es)}
    kind, dims = case["kind"], _dims(case)
    ranges = _ranges(case) if case["entry"] == "plan" else None
    pairs = sum(e - b for b, e in ranges) if ranges else sum(
        n for n, _ in _per_ijk(kind, dims))
    flops = work(case)["flops"]
    if flops > 4e13 or pairs > 20000:
        return None
    arrays = _inputs(kind, dims, seed, case["form"])
    e, per = _energies(kind, dims, arrays, ranges)
    out = {"energy": np.array([e])}
    if case["per_ijk"]:
        out["ijk"] = per
    return out


# --------------------------------------------------------------- the cases

def _case(name, entry, kind, form, dims, ijk=0, at=0.0, per_ijk=False, n=0,
          sizes=0):
    """A case; ijk: triples of each spin case in a plan's pass (0: all),
    from the fraction `at` of its list; n, sizes: a batch's systems."""
    c = {"entry": entry, "kind": kind, "form": form, "oa": dims[0],
         "va": dims[1], "ob": dims[2] if len(dims) == 4 else dims[0],
         "vb": dims[3] if len(dims) == 4 else dims[1], "ijk": ijk, "at": at,
         "per_ijk": per_ijk, "n": n, "sizes": sizes}
    if name:
        c["name"] = name
    return c


def _log(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def _shrink(dims):
    return tuple(d if n % 2 == 0 and d < 8 else max(1, d - max(1, d // 12))
                 for n, d in enumerate(dims))


def _four(kind, dims):
    return tuple(dims) if len(dims) == 4 else (dims[0], dims[1]) * 2


def _dims(case):
    if case["kind"] in ("rpt", "rft"):
        return (case["oa"], case["va"])
    return (case["oa"], case["va"], case["ob"], case["vb"])


def _batch_dims(case):
    """Sizes of a batch's systems: o in [4, 20], v in [40, 160] (FP64
    (T); smaller for the other calls, which have twice or four times the
    work per size), spread over their logarithm."""
    rng = random.Random(case["sizes"])
    kind = case["kind"]
    o_hi = 20 if kind == "rpt" else 12
    v_hi = 160 if kind == "rpt" else 100
    out = []
    for _ in range(case["n"]):
        o, v = _log(rng, 4, o_hi), _log(rng, 40, v_hi)
        out.append((o, v) if kind in ("rpt", "rft") else
                   (o, v, max(1, o - rng.randint(0, 2)),
                    v + rng.randint(0, 3)))
    return out


def _spin_cases(kind):
    """(same spin, spin) in the order of the plan's spin cases"""
    if kind in ("rpt", "rft"):
        return [(True, 0), (False, 0)]
    return [(True, 0), (True, 1), (False, 0), (False, 1)]


def _triples(same, o1, o2):
    return [(i, j, k) for i in range(o1) for j in range(i + 1, o1)
            for k in (range(j + 1, o1) if same else range(o2))]


def _per_ijk(kind, dims):
    """(triples, flops of one) of each spin case"""
    oa, va, ob, vb = _four(kind, dims)
    sets = 2 if kind in ("rft", "uft") else 1
    out = []
    for same, sp in _spin_cases(kind):
        o1, v1, o2, v2 = (oa, va, ob, vb) if sp == 0 else (ob, vb, oa, va)
        if same:
            n = o1 * (o1 - 1) * (o1 - 2) // 6
            f = 3.0 * v1**3 * (v1 - 1) + 6.0 * o1 * v1**3
            n = n if v1 >= 3 else 0
        else:
            n = o1 * (o1 - 1) // 2 * o2
            f = (2.0 * v1**3 * v2 + 4.0 * v1**2 * v2**2 +
                 2.0 * v2 * v1**2 * (v1 - 1) + 6.0 * o1 * v1**2 * v2 +
                 4.0 * o2 * v1**2 * v2)
            n = n if v1 >= 2 else 0
        out.append((n, f * sets))
    return out


def _flops(kind, dims):
    return float(sum(n * f for n, f in _per_ijk(kind, dims)))


def _ranges(case):
    """[begin, end) of the triples of each spin case in a plan's pass"""
    out = []
    for n, _ in _per_ijk(case["kind"], _dims(case)):
        m = min(n, case["ijk"]) if case["ijk"] else n
        b = int(case["at"] * (n - m))
        out.append((b, b + m))
    return out


def _input_bytes(kind, form, dims):
    oa, va, ob, vb = _four(kind, dims)
    if kind in ("rpt", "rft"):
        ov = oa * va
        oovv = 2 * oa * oa * va * va
        oovo = 2 * oa**3 * va
        ovvv = oa * va * (va * (va - 1) // 2) + oa * va**3
    else:
        ov = oa * va + ob * vb
        oovv = (oa * va)**2 + 2 * oa * ob * va * vb + (ob * vb)**2
        oovo = oa**3 * va + oa * ob * ob * va + ob**3 * vb + ob * oa * oa * vb
        ovvv = (oa * va * (va * (va - 1) // 2) + oa * vb * va * vb +
                ob * vb * (vb * (vb - 1) // 2) + ob * va * vb * va)
    n = 3 * ov + 2 * oovv + oovo + ovvv
    if kind in ("rft", "uft"):
        n += oovv + oovo + ovvv
    return float(n) * (4 if form == "fp32" else 8)


# -------------------------------------------------------------- the inputs

def _sub(seed, n):
    return (int(seed) * 1000003 + 7919 * n) % (1 << 62)


class _Rng:
    def __init__(self, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))

    def normal(self, sig, *shape):
        x = torch.randn(*shape, generator=self.g, device=self.dev,
                        dtype=torch.float64)
        return x.mul_(sig)

    def uniform(self, lo, hi, *shape):
        x = torch.rand(*shape, generator=self.g, device=self.dev,
                       dtype=torch.float64)
        return x.mul_(hi - lo).add_(lo)


def _tri(v, dev):
    """rows and columns of the packed pairs b > c (index b(b-1)/2 + c)"""
    t = torch.tril_indices(v, v, -1, device=dev)
    return t[0], t[1]


def _oovv(r, sig, kind, oa, va, ob, vb):
    """blocks of an amplitude-like [o][o][v][v] family"""
    if kind in ("rpt", "rft"):
        x = r.normal(sig, oa, oa, va, va)
        ab = (x + x.permute(1, 0, 3, 2)) / math.sqrt(2.0)
        return [ab - ab.permute(0, 1, 3, 2), ab]
    out = []
    for o, v in ((oa, va), (ob, vb)):
        x = r.normal(sig, o, o, v, v)
        x = x - x.permute(1, 0, 2, 3)
        out.append((x - x.permute(0, 1, 3, 2)) / 2.0)
    ab = r.normal(sig, oa, ob, va, vb)
    return [out[0], ab, out[1], ab.permute(1, 0, 3, 2)]


def _oovo(r, sig, kind, oa, va, ob, vb):
    """blocks of [o][o][v][o] integrals"""
    if kind in ("rpt", "rft"):
        ab = r.normal(sig, oa, oa, va, oa)
        return [ab - ab.permute(1, 0, 2, 3), ab]
    out = []
    for o, v in ((oa, va), (ob, vb)):
        x = r.normal(sig, o, o, v, o)
        out.append((x - x.permute(1, 0, 2, 3)) / math.sqrt(2.0))
    return [out[0], r.normal(sig, oa, ob, va, ob), out[1],
            r.normal(sig, ob, oa, vb, oa)]


def _ovvv(r, sig, kind, oa, va, ob, vb):
    """blocks of [o][v][v][v] integrals, same spin packed over b > c"""
    if kind in ("rpt", "rft"):
        ab = r.normal(sig, oa, va, va, va)
        b, c = _tri(va, ab.device)
        aa = torch.empty(oa, va, b.numel(), device=ab.device,
                         dtype=torch.float64)
        for k in range(oa):
            aa[k] = ab[k][:, b, c] - ab[k][:, c, b]
        return [aa, ab]
    return [r.normal(sig, oa, va, va * (va - 1) // 2),
            r.normal(sig, oa, vb, va, vb),
            r.normal(sig, ob, vb, vb * (vb - 1) // 2),
            r.normal(sig, ob, va, vb, va)]


def _flat(blocks):
    return torch.cat([b.reshape(-1) for b in blocks])


def _inputs(kind, dims, seed, form):
    """The arrays of one call in pt.h order, flat, on the GPU, in the
    call's element type."""
    oa, va, ob, vb = _four(kind, dims)
    restricted, ft = kind in ("rpt", "rft"), kind in ("rft", "uft")
    r = _Rng(seed)
    spins = [(oa, va)] if restricted else [(oa, va), (ob, vb)]

    def ov(sig):
        return torch.cat([r.normal(sig, o * v) for o, v in spins])

    d = torch.cat([(r.uniform(-1.5, -0.3, o, 1) - r.uniform(0.1, 3.0, 1, v) +
                    (OMEGA / 3 if ft else 0.0)).reshape(-1)
                   for o, v in spins])
    args = (kind, oa, va, ob, vb)

    def like(x, make, sig):
        """a left operand: the right one and a draw of its own"""
        return _flat(make(r, sig * math.sqrt(1 - LIKE**2), *args)).add_(
            x, alpha=LIKE)

    f, t1 = ov(SIG_F), ov(SIG_T1)
    t2 = _flat(_oovv(r, SIG_T2, *args))
    if not ft:
        out = [d, f, t1, t2, _flat(_oovo(r, SIG_INT, *args)),
               _flat(_oovv(r, SIG_INT, *args)),
               _flat(_ovvv(r, SIG_INT, *args))]
    else:
        l2 = like(t2, _oovv, SIG_T2)
        oovv = _flat(_oovv(r, SIG_INT, *args))
        i2 = _flat(_oovo(r, SIG_INT, *args))
        i3 = _flat(_ovvv(r, SIG_INT, *args))
        out = [d, f, t1, t2, l2, oovv, i2, i3, like(i2, _oovo, SIG_INT),
               like(i3, _ovvv, SIG_INT)]
    if form == "fp32":
        out = [x.float() for x in out]
    return out


class State:
    """What a user's program holds before a pass; frees its plan or batch."""

    def __init__(self, case, seed):
        self.case, self.plan, self.batch = case, None, None
        kind, form = case["kind"], case["form"]
        if case["entry"] == "batch":
            self.systems = []
            for n, d in enumerate(_batch_dims(case)):
                t = _inputs(kind, d, _sub(seed, n), form)
                self.systems.append((d, t, self._device(kind, form, t)))
            torch.cuda.synchronize()
            self.batch = api.Batch(kind, form,
                                   [(d, dev) for d, _, dev in self.systems])
            return
        self.dims = _dims(case)
        tensors = _inputs(kind, self.dims, seed, form)
        if case["entry"] == "call":
            self.arrays = [t.cpu().numpy() for t in tensors]
            return
        self.tensors = tensors
        self.dev = self._device(kind, form, tensors)
        torch.cuda.synchronize()
        if case["entry"] == "plan":
            self.ranges = _ranges(case)
            self.plan = api.Plan(kind, form, self.dims, self.dev)

    @staticmethod
    def _device(kind, form, tensors):
        return api.DeviceArrays(kind, None, [t.data_ptr() for t in tensors],
                                [t.numel() for t in tensors], form == "fp32")

    def __del__(self):
        for held in (self.plan, self.batch):
            if held is not None:
                held.close()


# ------------------------------------------------- energies in 64 bits

def _blocks(kind, dims, arrays):
    """The arrays as blocks [aaaa, abab, bbbb, baba] (ov: [a, b]), double."""
    oa, va, ob, vb = _four(kind, dims)
    restricted = kind in ("rpt", "rft")
    sp = [(oa, va, ob, vb), (ob, vb, oa, va)]

    def cut(x, shapes):
        x, out = x.double(), []
        at = 0
        for s in shapes:
            n = math.prod(s)
            out.append(x[at:at + n].reshape(s))
            at += n
        return out

    def ov(x):
        if restricted:
            return cut(x, [(oa, va)]) * 2
        return cut(x, [(oa, va), (ob, vb)])

    def four(x, same, mixed):
        if restricted:
            return cut(x, [same(*sp[0]), mixed(*sp[0])]) * 2
        return cut(x, [f(*s) for s in sp for f in (same, mixed)])

    def oovv(x):
        return four(x, lambda o, v, p, w: (o, o, v, v),
                    lambda o, v, p, w: (o, p, v, w))

    def oovo(x):
        return four(x, lambda o, v, p, w: (o, o, v, o),
                    lambda o, v, p, w: (o, p, v, p))

    def ovvv(x):
        return four(x, lambda o, v, p, w: (o, v, v * (v - 1) // 2),
                    lambda o, v, p, w: (o, w, v, w))

    if kind in ("rpt", "upt"):
        d, f, u, t2, o3, g, v3 = arrays
        z, sets = oovv(t2), [(oovv(t2), oovo(o3), ovvv(v3))]
    else:
        d, f, u, t2, l2, g, i2, i3, i6, i7 = arrays
        z = oovv(l2)
        sets = [(z, oovo(i6), ovvv(i7)), (oovv(t2), oovo(i2), ovvv(i3))]
    return ov(d), ov(f), ov(u), oovv(g), z, sets


def _w_same(T, O, V, i, j, ks, tri):
    """Connected triples W[k][a][b][c] of the same-spin case (a > b > c)."""
    v, nk = T.shape[-1], len(ks)
    w = torch.zeros(nk, v, v, v, device=T.device, dtype=torch.float64)

    def full(packed):
        q = torch.zeros(packed.shape[0], v, v * v, device=T.device,
                        dtype=torch.float64)
        q[:, :, tri[0] * v + tri[1]] = packed
        return q

    # sum_d T[p, q, x, d] V[r, d, (y, z)] for (p, q; r) = (i, j; k),
    # -(i, k; j), -(k, j; i)
    for s, t, q in ((1.0, T[i, j][None], full(V[ks])),
                    (-1.0, T[i, ks], full(V[j:j + 1])),
                    (-1.0, T[ks, j], full(V[i:i + 1]))):
        y = torch.matmul(t, q).reshape(nk, v, v, v)
        w += s * (y.permute(0, 2, 3, 1) - y.permute(0, 2, 1, 3) + y)
    # sum_l O[q, r, z, l] T[p, l, x, y] for (p; q, r) = (i; j, k),
    # -(j; i, k), -(k; j, i)
    o = T.shape[0]
    for s, t, q in ((1.0, T[i:i + 1], O[j, ks]), (-1.0, T[j:j + 1], O[i, ks]),
                    (-1.0, T[ks], O[j, i][None])):
        x = torch.matmul(q, t.reshape(-1, o, v * v)).reshape(nk, v, v, v)
        w += s * (x - x.permute(0, 2, 1, 3) - x.permute(0, 3, 2, 1))
    return w


def _w_mixed(A, B, C, i, j, ks, tri):
    """Connected triples W[k][a][b][c] of the mixed-spin case (a > b; i, j
    of the pair's spin): A, B, C = (T, O, V) of the blocks aaaa, abab and
    baba of the pair's spin."""
    (TA, OA, VA), (TB, OB, VB), (TC, OC, VC) = A, B, C
    oa, va, ob, vb = TB.shape[0], TB.shape[2], TB.shape[1], TB.shape[3]
    nk = len(ks)

    def full(packed):
        q = torch.zeros(va, va * va, device=TA.device, dtype=torch.float64)
        q[:, tri[0] * va + tri[1]] = packed
        return q

    # m[a][b][c], antisymmetrised in a and b below
    m = torch.matmul(TB[j, ks], VB[i].reshape(vb, va * vb))
    m -= torch.matmul(TB[i, ks], VB[j].reshape(vb, va * vb))
    m += torch.matmul(OB[j, ks], TB[i].reshape(ob, va * vb))
    m -= torch.matmul(OB[i, ks], TB[j].reshape(ob, va * vb))
    m = m.reshape(nk, va, va, vb)
    n = torch.matmul(OA[j, i][None], TC[ks].reshape(nk, oa, vb * va))
    n -= torch.matmul(TA[i, j][None], VC[ks].reshape(nk, va, vb * va))
    m += n.reshape(nk, va, vb, va).transpose(2, 3)
    w = m - m.transpose(1, 2)
    # c[c][a][b]
    c = torch.matmul(TC[ks, i], full(VA[j])) - torch.matmul(TC[ks, j],
                                                            full(VA[i]))
    c += torch.matmul(OC[ks, i], TA[j].reshape(oa, va * va))
    c -= torch.matmul(OC[ks, j], TA[i].reshape(oa, va * va))
    return w + c.reshape(nk, vb, va, va).permute(0, 2, 3, 1)


def _z_same(u, f, G, Z, i, j, ks):
    """Disconnected triples of the same-spin case"""
    z = 0.0
    for x, M in ((u, G), (f, Z)):
        xi, xj, xk = x[i][None], x[j][None], x[ks]
        jk, ik, ji = M[j, ks], M[i, ks], M[j, i][None]
        for s, y, q in ((1, xi, jk), (-1, xj, ik), (-1, xk, ji)):
            z = z + s * (y[:, :, None, None] * q[:, None, :, :] -
                         y[:, None, :, None] * q[:, :, None, :] -
                         y[:, None, None, :] * q.transpose(1, 2)[:, :, :, None])
    return z


def _z_mixed(u, f, GA, GB, ZA, ZB, s, i, j, ks):
    """Disconnected triples of the mixed-spin case, pair spin s"""
    z = 0.0
    for x, MA, MB in ((u, GA, GB), (f, ZA, ZB)):
        xi, xj, xc = x[s][i][None], x[s][j][None], x[1 - s][ks]
        jk, ik, ji = MB[j, ks], MB[i, ks], MA[j, i][None]
        z = z + (xi[:, :, None, None] * jk[:, None, :, :] -
                 xi[:, None, :, None] * jk[:, :, None, :] -
                 xj[:, :, None, None] * ik[:, None, :, :] +
                 xj[:, None, :, None] * ik[:, :, None, :] +
                 xc[:, None, None, :] * ji.transpose(1, 2)[:, :, :, None])
    return z


def _energies(kind, dims, arrays, ranges):
    """(energy, per-triple energies of each spin case) over the ranges"""
    d, f, u, g, z, sets = _blocks(kind, dims, arrays)
    total, per = 0.0, []
    factor = 2.0 if kind in ("rpt", "rft") else 1.0
    for sc, (same, s) in enumerate(_spin_cases(kind)):
        o1, o2 = d[s].shape[0], d[1 - s].shape[0]
        v1, v2 = d[s].shape[1], d[s if same else 1 - s].shape[1]
        todo = _triples(same, o1, o2)
        if _per_ijk(kind, dims)[sc][0] == 0:
            todo = []
        if ranges:
            todo = todo[ranges[sc][0]:ranges[sc][1]]
        dev = d[s].device
        tri = _tri(v1, dev)
        a = torch.arange(v1, device=dev)
        keep = (a[:, None] > a[None, :])[:, :, None]
        if same:
            keep = keep & (a[:, None] > a[None, :])[None]
        # slots of aaaa, abab and baba as this pair spin sees them
        A, B, C = (0, 1, 3) if s == 0 else (2, 3, 1)
        es = []
        at = 0
        most = max(1, int(2e8 / (v1 * v1 * v2)))   # triples at a time
        while at < len(todo):
            i, j, _ = todo[at]
            n = at
            while n < len(todo) and todo[n][:2] == (i, j) and n - at < most:
                n += 1
            ks = [t[2] for t in todo[at:n]]
            at = n
            if same:
                ws = [_w_same(T[A], O[A], V[A], i, j, ks, tri)
                      for T, O, V in sets]
                zz = _z_same(u[s], f[s], g[A], z[A], i, j, ks)
                dk = d[s][ks]
            else:
                ws = [_w_mixed(*[(T[x], O[x], V[x]) for x in (A, B, C)],
                               i, j, ks, tri) for T, O, V in sets]
                zz = _z_mixed(u, f, g[A], g[B], z[A], z[B], s, i, j, ks)
                dk = d[1 - s][ks]
            dn = (d[s][i][None, :, None, None] + d[s][j][None, None, :, None] +
                  dk[:, None, None, :])
            e = (ws[0] - zz).mul_(ws[-1]).div_(dn).mul_(keep)
            es.append(e.sum(dim=(1, 2, 3)))
        es = torch.cat(es).cpu().numpy() if es else np.zeros(0)
        per.append(es)
        total += factor * float(es.sum())
    return total, per
