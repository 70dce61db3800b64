"""The measured cases: what programs that use this library have it do.

A case names one kind of call with its sizes and options:

* ``step``      one HowFar + Perform step of a batch of tracks (Context.step), written to a second batch;
* ``split``     the same step through howfar and perform with the caller's geometry between them;
* ``substeps``  TrackElectron's MSC sub-step loop over a batch of e-/e+, driven by the caller;
* ``batches``   many uneven batches stepped by one BatchPlan;
* ``lookup``    energy-loss and cross-section lookups of e-/e+;
* ``gamma``     gamma cross-section lookups with the selected interaction;
* ``showers``   electron showers in a sampling calorimeter, from the primaries to the deposits.

Each comes in the FP64 form and in the FP32-table form (``fp32``). Tracks are fresh ones as the stepping benchmark
draws them: e-:e+:gamma = 4:1:5, energies log-uniform in [100 keV, 10 GeV], isotropic directions, couples uniform
over four materials, safeties log-uniform in [1 um, 10 mm]; ``ordered`` batches hold the e-/e+ first, as a device
track stack hands them over, the others interleave the kinds by track id.
"""
import json
import math

import numpy as np
import torch

from g4hepem_amd import HEPEM_FP32T, HEPEM_FP64, BatchPlan, Context, Tables
from g4hepem_amd._native import HOWFAR_FIELDS, OUT_FIELDS, SUBSTEP_FIELDS, TRACK_FIELDS, slab_setup
from g4hepem_amd.tracks import HowFarSoA, StepOutSoA, SubstepSoA, TrackSoA

CALORIMETER = ("G4_Pb", "G4_lAr")                      # the lookup and shower configurations
FOUR = ("G4_PbWO4", "G4_Pb", "G4_lAr", "G4_Si")        # the stepping configurations
PROD_CUT_MM = 0.7
MIX = (4, 1, 5)                                        # e- : e+ : gamma
SAFETY_MM = (1e-3, 10.0)
STEP_E = (0.1, 1.0e4)                                  # MeV
LOOKUP_E = (1e-3, 1.0e8)


def listed():
    return [
        # a worker's own small batch, or the tail of a shower: the smallest batch of the batched configuration
        {"name": "step_1k", "kind": "step", "n": 1000, "fp32": False, "ordered": False},
        # a host thread's batch when many of them share the GPU, odd in size
        {"name": "step_16k", "kind": "step", "n": 16411, "fp32": True, "ordered": True},
        # one wave of events of a detector simulation
        {"name": "step_131k", "kind": "step", "n": 131072, "fp32": False, "ordered": False},
        # the headline configuration in its two forms
        {"name": "step_1m", "kind": "step", "n": 1000000, "fp32": False, "ordered": False},
        {"name": "step_1m_fp32", "kind": "step", "n": 1000000, "fp32": True, "ordered": False},
        # a device stack's generation, in the stack's own order
        {"name": "step_3m_ordered", "kind": "step", "n": 3000017, "fp32": False, "ordered": True},
        # a tracking loop with its own geometry between HowFar and Perform
        {"name": "split_300k", "kind": "split", "n": 300007, "fp32": False, "ordered": False},
        # TrackElectron's loop driven by the caller
        {"name": "substeps_100k", "kind": "substeps", "n": 100003, "fp32": False},
        # the batched configuration: 64 uneven batches in one plan
        {"name": "batches_64", "kind": "batches", "batches": 64, "smallest": 1000, "largest": 1000000, "sizes": 7, "fp32": False},
        # table lookups of a whole tracking pass
        {"name": "lookup_10m", "kind": "lookup", "n": 10000000, "particle": 0, "fp32": False},
        {"name": "gamma_1m", "kind": "gamma", "n": 1000003, "fp32": False},
        # showers of 10 GeV electrons in 50 x (2.3 mm Pb + 5.7 mm lAr)
        {"name": "showers_1k", "kind": "showers", "events": 1000, "layers": 50, "ekin": 1.0e4, "woodcock": 0.0, "fp32": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "split", "substeps", "batches", "lookup", "gamma", "showers"])
    fp32 = rng.random() < 0.4
    if kind == "step":
        return {"kind": kind, "n": _log_int(rng, 700, 3.0e6), "fp32": fp32, "ordered": rng.random() < 0.5}
    if kind == "split":
        return {"kind": kind, "n": _log_int(rng, 2000, 1.0e6), "fp32": fp32, "ordered": rng.random() < 0.5}
    if kind == "substeps":
        return {"kind": kind, "n": _log_int(rng, 2000, 2.0e5), "fp32": fp32}
    if kind == "batches":
        return {"kind": kind, "batches": rng.randrange(3, 65), "smallest": _log_int(rng, 300, 3000),
                "largest": _log_int(rng, 1.0e4, 3.0e5), "sizes": rng.randrange(1 << 20), "fp32": fp32}
    if kind == "lookup":
        return {"kind": kind, "n": _log_int(rng, 1.0e4, 1.0e7), "particle": rng.randrange(2), "fp32": fp32}
    if kind == "gamma":
        return {"kind": kind, "n": _log_int(rng, 1.0e4, 1.0e7), "fp32": fp32}
    return {"kind": kind, "events": _log_int(rng, 20, 1000), "layers": rng.randrange(20, 51), "ekin": float(_log_int(rng, 1000, 10000)),
            "woodcock": 0.2 if rng.random() < 0.3 else 0.0, "fp32": fp32}


# ---- what a program holds for its whole run: the tables and their device images ------------------------------------

_tables, _contexts = {}, {}


def _get_tables(materials):
    if materials not in _tables:
        _tables[materials] = Tables(list(materials), PROD_CUT_MM)
    return _tables[materials]


def _get_context(materials, fp32):
    if (materials, fp32) not in _contexts:
        _contexts[materials, fp32] = Context(_get_tables(materials), HEPEM_FP32T if fp32 else HEPEM_FP64)
    return _contexts[materials, fp32]


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _generator(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _uniform(g, n):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _kinds(n, electrons_only):
    """Particle types by track id: e-, e+, gamma in the ratio MIX (without the gammas: e- and e+ in theirs)."""
    mix = MIX[:2] if electrons_only else MIX
    period = torch.tensor([k for k, m in enumerate(mix) for _ in range(m)], dtype=torch.int8, device="cuda")
    return period.repeat(-(-n // len(period)))[:n]


class _Block:
    """A SoA whose arrays lie in one allocation, so that a whole batch is restored by one copy."""

    def __init__(self, cls, n):
        offs, end = {}, 0
        for name, (dt, k) in cls.FIELDS.items():
            offs[name] = end
            end += (np.dtype(dt).itemsize * k * n + 255) & ~255
        self.bytes = torch.zeros(max(end, 1), dtype=torch.uint8, device="cuda")
        arrays = {}
        for name, (dt, k) in cls.FIELDS.items():
            part = self.bytes[offs[name]:offs[name] + np.dtype(dt).itemsize * k * n]
            arrays[name] = part.view(getattr(torch, dt))
        self.soa = cls(n, "torch", "cuda", arrays)


def _fill_tracks(t, seed, salt, first_id=0, ordered=False, electrons_only=False, ncouples=len(FOUR)):
    n = t.n
    g = _generator(seed, salt)
    ids = torch.arange(n, device="cuda", dtype=torch.int64)
    pt = _kinds(n, electrons_only)
    if ordered:
        order = torch.cat([torch.nonzero(pt != 2).view(-1), torch.nonzero(pt == 2).view(-1)])
        ids, pt = ids[order], pt[order]
    t["ptype"].copy_(pt)
    t["id"].copy_((ids + first_id).to(torch.int32))
    t["imc"].copy_(torch.randint(0, ncouples, (n,), generator=g, device="cuda", dtype=torch.int32))
    t["ekin"].copy_(torch.exp(_uniform(g, n) * math.log(STEP_E[1] / STEP_E[0]) + math.log(STEP_E[0])))
    cost = 2.0 * _uniform(g, n) - 1.0
    phi = 2.0 * math.pi * _uniform(g, n)
    sint = torch.sqrt((1.0 - cost) * (1.0 + cost))
    t["dir"].copy_(torch.cat([sint * torch.cos(phi), sint * torch.sin(phi), cost]))
    t["safety"].copy_(torch.exp(_uniform(g, n) * math.log(SAFETY_MM[1] / SAFETY_MM[0]) + math.log(SAFETY_MM[0])))
    # start-of-track state
    t["num_ia_left"].fill_(-1.0)
    t["msc_init_range"].fill_(1.0e21)
    t["msc_dyn_range_factor"].fill_(0.04)
    t["msc_tlimit_min"].fill_(1.0e-7)
    t["msc_first_step"].fill_(1)


def _queries(case, seed):
    n, g = case["n"], _generator(seed, 5)
    imc = torch.randint(0, len(CALORIMETER), (n,), generator=g, device="cuda", dtype=torch.int32)
    lekin = _uniform(g, n) * math.log(LOOKUP_E[1] / LOOKUP_E[0]) + math.log(LOOKUP_E[0])
    return imc, torch.exp(lekin), lekin, _uniform(g, n)


def _batch_sizes(case):
    rng = np.random.Generator(np.random.Philox(case["sizes"]))
    lo, hi = math.log(case["smallest"]), math.log(case["largest"])
    return np.exp(rng.uniform(lo, hi, case["batches"])).astype(np.int64).tolist()


def _pool(fields, total):
    return {k: torch.zeros(c * total, dtype=getattr(torch, dt), device="cuda") for k, (dt, c) in fields.items()}


def _part(cls, pool, first, n):
    """Batch `n` tracks from `first` on of a pool: k planes of n values at k * first."""
    return cls(n, "torch", "cuda", {k: pool[k][c * first:c * (first + n)] for k, (_, c) in cls.FIELDS.items()})


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        s = {"ctx": _get_context(FOUR, case["fp32"]), "tin": TrackSoA(case["n"], "torch", "cuda"), "tout": TrackSoA(case["n"], "torch", "cuda"),
             "res": StepOutSoA(case["n"], "torch", "cuda"), "work": Context.work_buffer(case["n"], "cuda")}
        _fill_tracks(s["tin"], seed, 1, ordered=case["ordered"])
    elif kind == "split":
        n = case["n"]
        fresh, tracks = _Block(TrackSoA, n), _Block(TrackSoA, n)
        _fill_tracks(fresh.soa, seed, 2, ordered=case["ordered"])
        # the caller's geometry: how far each track may go before its volume ends
        dist = torch.exp(_uniform(_generator(seed, 3), n) * math.log(1e4) + math.log(1e-2))
        s = {"ctx": _get_context(FOUR, case["fp32"]), "fresh": fresh, "tracks": tracks, "hs": HowFarSoA(n, "torch", "cuda"),
             "res": StepOutSoA(n, "torch", "cuda"), "work": Context.work_buffer(n, "cuda"), "dist": dist}
    elif kind == "substeps":
        n = case["n"]
        fresh, tracks = _Block(TrackSoA, n), _Block(TrackSoA, n)
        _fill_tracks(fresh.soa, seed, 4, electrons_only=True)
        s = {"ctx": _get_context(FOUR, case["fp32"]), "fresh": fresh, "tracks": tracks, "hs": HowFarSoA(n, "torch", "cuda"),
             "ss": SubstepSoA(n, "torch", "cuda"), "res": StepOutSoA(n, "torch", "cuda"), "work": Context.work_buffer(n, "cuda")}
    elif kind == "batches":
        sizes = _batch_sizes(case)
        total = sum(sizes)
        pin, pout, pres = _pool(TRACK_FIELDS, total), _pool(TRACK_FIELDS, total), _pool(OUT_FIELDS, total)
        batches, first = [], 0
        for k, n in enumerate(sizes):
            tin = _part(TrackSoA, pin, first, n)
            _fill_tracks(tin, seed, 100 + k, first_id=first)
            batches.append((tin, _part(TrackSoA, pout, first, n), _part(StepOutSoA, pres, first, n)))
            first += n
        ctx = _get_context(FOUR, case["fp32"])
        s = {"plan": BatchPlan(ctx, batches), "pout": pout, "pres": pres}
    elif kind in ("lookup", "gamma"):
        imc, ekin, lekin, u = _queries(case, seed)
        s = {"ctx": _get_context(CALORIMETER, case["fp32"]), "imc": imc, "ekin": ekin, "lekin": lekin, "u": u}
        if kind == "lookup":
            s["out"] = torch.empty(5 * case["n"], dtype=torch.float64, device="cuda")
            s["particle"] = case["particle"]
    else:
        s = {"ctx": _get_context(CALORIMETER, case["fp32"]), "events": case["events"],
             "setup": slab_setup(case["layers"], [2.3, 5.7], [0, 1], 0, case["ekin"], capacity=1 << 22, events_per_chunk=4096,
                                 refill_below=1 << 20, woodcock_min_ekin=case["woodcock"])}
    s["kind"] = kind
    s["seed"] = int(seed) & 0x7FFFFFFF
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------

def _outputs(tracks, res, more=None):
    # draw counters as signed words: torch indexes no unsigned 32-bit tensors
    out = {"state." + k: v.view(torch.int32) if v.dtype == torch.uint32 else v for k, v in tracks.items()}
    out.update({"step." + k: v for k, v in res.items()})
    out.update(more or {})
    return out


def run(s):
    kind, seed = s["kind"], s["seed"]
    if kind == "step":
        s["ctx"].step(seed, s["tin"], s["tout"], s["res"], s["work"])
        return _outputs(s["tout"].a, s["res"].a)
    if kind == "split":
        ctx, t, hs = s["ctx"], s["tracks"].soa, s["hs"]
        s["tracks"].bytes.copy_(s["fresh"].bytes)  # the calls step in place: stands for the fill of the batch
        ctx.howfar(seed, t, hs, s["work"])
        torch.minimum(hs["geom_step"], s["dist"], out=hs["geom_step"])
        t["on_boundary"].copy_(hs["geom_step"] >= s["dist"])
        ctx.perform(seed, t, hs, s["res"], s["work"])
        return _outputs(t.a, s["res"].a, {"howfar." + k: v for k, v in hs.a.items()})
    if kind == "substeps":
        ctx, t, hs, ss, work = s["ctx"], s["tracks"].soa, s["hs"], s["ss"], s["work"]
        s["tracks"].bytes.copy_(s["fresh"].bytes)
        ctx.electron_step_begin(seed, t, hs, ss, work)
        while True:
            ctx.electron_substep_howfar(seed, t, hs, ss, work)
            ctx.electron_substep_along(seed, t, hs, ss, work)
            if ctx.electron_substep_active(work) == 0:
                break
        ctx.electron_step_end(seed, t, hs, ss, s["res"], work)
        return _outputs(t.a, s["res"].a, {"loop." + k: v for k, v in ss.a.items()})
    if kind == "batches":
        s["plan"].run(seed)
        return _outputs(s["pout"], s["pres"])
    if kind == "lookup":
        return s["ctx"].lookup(s["particle"], s["imc"], s["ekin"], s["lekin"], s["out"])
    if kind == "gamma":
        return s["ctx"].lookup_gamma(s["imc"], s["ekin"], s["lekin"], s["u"])
    r = s["ctx"].slab_run(s["setup"], s["events"], seed, per_event=True)
    return {k: r[k] for k in ("edep_event", "leak_event", "edep_sum", "edep_sum2", "steps", "tracks", "substeps")}


# ---- the least that a pass has to move -------------------------------------------------------------------------------

def _size(fields, names):
    return sum(np.dtype(fields[k][0]).itemsize * fields[k][1] for k in names)


_MSC = [k for k in TRACK_FIELDS if k.startswith("msc_")]
_COMMON = [k for k in TRACK_FIELDS if not k.startswith("msc_")]
_CHANGED = ("ekin", "dir", "num_ia_left", "rng_ctr", "rng_gauss", "rng_has_gauss")
_RESULT = [k for k in OUT_FIELDS if not k.startswith("sec_")]
_SECONDARY = 33                                        # type, energy and direction of one
_PER_TRACK = 1.14                                      # secondaries of a mixed batch's step
_STEPS_PER_GEV = 5400                                  # steps of a shower in the calorimeter


def work(case):
    kind = case["kind"]
    electron = 0.5 if kind != "substeps" else 1.0
    msc = electron * _size(TRACK_FIELDS, _MSC)
    read = _size(TRACK_FIELDS, _COMMON) + msc
    changed = _size(TRACK_FIELDS, _CHANGED) + msc
    result = _size(OUT_FIELDS, _RESULT) + _SECONDARY * _PER_TRACK
    if kind == "step":
        return {"bytes": case["n"] * (read + _size(TRACK_FIELDS, _COMMON) + msc + result), "flops": 0}
    if kind == "split":
        hand = electron * _size(HOWFAR_FIELDS, [k for k in HOWFAR_FIELDS if k != "pe_xsec"]) + 0.5 * (8 + 8 + 4 + 8)
        return {"bytes": case["n"] * (2 * read + 2 * changed + 2 * hand + result), "flops": 0}
    if kind == "substeps":
        loop = _size(SUBSTEP_FIELDS, SUBSTEP_FIELDS) + _size(HOWFAR_FIELDS, HOWFAR_FIELDS)
        return {"bytes": case["n"] * (2 * read + 2 * changed + 2 * loop + result), "flops": 0}
    if kind == "batches":
        return {"bytes": sum(_batch_sizes(case)) * (read + _size(TRACK_FIELDS, _COMMON) + msc + result), "flops": 0}
    if kind == "lookup":
        return {"bytes": case["n"] * (4 + 2 * 8 + 5 * 8), "flops": 0}
    if kind == "gamma":
        return {"bytes": case["n"] * (4 + 3 * 8 + 2 * 8 + 4), "flops": 0}
    return {"bytes": case["events"] * case["ekin"] * 1e-3 * _STEPS_PER_GEV * (read + changed), "flops": 0}


# ---- the same values in 64 bits --------------------------------------------------------------------------------------
# Table lookups have such values: splines over the tables' own numbers. A sampled step has none but what HowFar
# looks up before its first random number decides anything (the range and the mean free paths).

class _Exact:
    def __init__(self, materials):
        d = json.loads(_get_tables(materials).to_json())["fData"]
        self.el = (d["fTheElectronData"], d["fThePositronData"])
        self.gamma = d["fTheGammaData"]
        self.cuts = d["fTheMatCutData"]["fMatCutData"]
        self.mats = d["fTheMaterialData"]["fMaterialData"]

    @staticmethod
    def of(values):
        return torch.tensor(values, dtype=torch.float64, device="cuda")

    @staticmethod
    def spline(x1, x2, y1, y2, s1, s2, x):
        h = x2 - x1
        b = ((x - x1) / h).clamp(0.0, 1.0)
        return y1 + b * (y2 - y1) + b * (b - 1.0) * ((2.0 - b) * s1 + (1.0 + b) * s2) * (h * h * 0.166666666667)

    @staticmethod
    def bins(le, lmin, ild, n):
        return ((le - lmin) * ild).clamp(0.0, n - 2).to(torch.int64)

    def loss(self, e, imc, column, x, le):
        """Range (0) or dE/dx (1) of the queries of couple imc."""
        grid, data = self.of(e["fELossEnergyGrid"]), self.of(e["fELossData"])
        n = len(grid)
        i = self.bins(le, e["fELossLogMinEkin"], e["fELossEILDelta"], n)
        d = data[n * (5 * imc + 2 * column):][:2 * n]
        y = self.spline(grid[i], grid[i + 1], d[2 * i], d[2 * i + 2], d[2 * i + 1], d[2 * i + 3], x.clamp(grid[0].item(), grid[-1].item()))
        return y.clamp_min(0.0)

    def inverse(self, e, imc, r):
        grid, data = self.of(e["fELossEnergyGrid"]), self.of(e["fELossData"])
        n = len(grid)
        ranges, second = data[5 * n * imc:][:2 * n:2].contiguous(), data[n * (5 * imc + 4):][:n]
        i = (torch.searchsorted(ranges, r, right=True) - 1).clamp(0, n - 2)
        y = self.spline(ranges[i], ranges[i + 1], grid[i], grid[i + 1], second[i], second[i + 1], r).clamp_min(0.0)
        return torch.where(r < ranges[0], grid[0] * (r / ranges[0]) ** 2, y)

    def macroscopic(self, e, imc, ioni, x, le, stepping=False):
        """Restricted cross section of couple imc; for the step limit, its largest value down to 0.8 of the energy."""
        data = e["fResMacXSecData"]
        at = e["fResMacXSecStartIndexPerMatCut"][imc]
        if not ioni:
            at += 3 * int(data[at]) + 5
        n, emax, vmax, lmin, ild = int(data[at]), data[at + 1], data[at + 2], data[at + 3], data[at + 4]
        d = self.of(data[at + 5:at + 5 + 3 * n])
        flat = None
        if stepping:
            above = x > emax
            flat = above & (0.8 * x < emax)
            x, le = torch.where(above, 0.8 * x, x), torch.where(above, le + math.log(0.8), le)
        i = 3 * self.bins(le, lmin, ild, n)
        y = self.spline(d[i], d[i + 3], d[i + 1], d[i + 4], d[i + 2], d[i + 5], x.clamp(d[0].item(), d[-3].item())).clamp_min(0.0)
        y = torch.where(x < d[0], torch.zeros_like(y), y)
        return y if flat is None else torch.where(flat, torch.full_like(y, vmax), y)

    def gammas(self, imat, x, le):
        """Total and photoelectric cross section of material imat, and the four columns of the high-energy window."""
        g = self.gamma
        data = self.of(g["fMacXsecData"])[imat * g["fDataPerMat"]:][:g["fDataPerMat"]]
        n0, n1 = g["fNumData0"] // 2, g["fNumData1"] // 3
        n2 = (g["fDataPerMat"] - g["fNumData0"] - g["fNumData1"]) // 9
        d0, d1, d2 = data[:2 * n0].view(n0, 2), data[2 * n0:][:3 * n1].view(n1, 3), data[2 * n0 + 3 * n1:].view(n2, 9)

        def linear(d, i, c):
            return d[i, c] + ((x - d[i, 0]) / (d[i + 1, 0] - d[i, 0])).clamp(0.0, 1.0) * (d[i + 1, c] - d[i, c])

        i0, i1, i2 = (self.bins(le, g["fLogEMin%d" % k], g["fEILDelta%d" % k], n) for k, n in enumerate((n0, n1, n2)))
        m = self.mats[imat]
        edges, coefs = self.of(m["fSandiaEnergies"]), self.of(m["fSandiaCoefficients"]).view(-1, 4)
        k = (torch.searchsorted(edges, x, right=True) - 1).clamp_min(0)
        pe0 = sum(coefs[k, c] / x ** (c + 1) for c in range(4)).clamp_min(0.0)
        mid = [linear(d1, i1, c).clamp_min(0.0) for c in (1, 2)]
        high = [self.spline(d2[i2, 0], d2[i2 + 1, 0], d2[i2, c], d2[i2 + 1, c], d2[i2, c + 1], d2[i2 + 1, c + 1], x) for c in (1, 3, 5, 7)]
        top, middle = x > g["fEMax1"], x > g["fEMax0"]
        total = torch.where(top, high[0], torch.where(middle, mid[0], linear(d0, i0, 1) + pe0))
        return total, torch.where(middle, mid[1], pe0), high, top


def _exact_lookup(case, seed):
    imc, x, le, _ = _queries(case, seed)
    E = _Exact(CALORIMETER)
    e = E.el[case["particle"]]
    out = torch.empty((5, case["n"]), dtype=torch.float64, device="cuda")
    for k in range(len(CALORIMETER)):
        at = torch.nonzero(imc == k).view(-1)
        xk, lk = x[at], le[at]
        r = E.loss(e, k, 0, xk, lk)
        for row, v in enumerate((E.loss(e, k, 1, xk, lk), r, E.inverse(e, k, r), E.macroscopic(e, k, True, xk, lk), E.macroscopic(e, k, False, xk, lk))):
            out[row, at] = v
    return out


def _exact_gamma(case, seed):
    imc, x, le, u = _queries(case, seed)
    E = _Exact(CALORIMETER)
    xs, pe = torch.empty_like(x), torch.empty_like(x)
    for k in range(len(CALORIMETER)):
        at = torch.nonzero(imc == k).view(-1)
        total, photo, high, top = E.gammas(E.cuts[k]["fHepEmMatIndex"], x[at], le[at])
        # above the pair threshold the track holds the cross section of the last process tried
        first, second = high[1] / total, (high[1] + high[2]) / total
        last = torch.where(u[at] <= first, high[1], torch.where(u[at] <= second, high[2], high[3]))
        xs[at], pe[at] = total, torch.where(top, last, photo)
    return xs, pe, None


def _exact_howfar(case, seed):
    t = TrackSoA(case["n"], "torch", "cuda")
    _fill_tracks(t, seed, 2, ordered=case["ordered"])
    E, n = _Exact(FOUR), case["n"]
    ranges, mfp = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.zeros((4, n), dtype=torch.float64, device="cuda")
    pt, imc, x = t["ptype"], t["imc"], t["ekin"]
    big = 1.0e20
    for k in range(len(FOUR)):
        imat = E.cuts[k]["fHepEmMatIndex"]
        for p in range(3):
            at = torch.nonzero((pt == p) & (imc == k)).view(-1)
            xk, lk = x[at], torch.log(x[at])
            if p == 2:
                mfp[0, at] = 1.0 / E.gammas(imat, xk, lk)[0]
                continue
            ranges[at] = E.loss(E.el[p], k, 0, xk, lk)
            for row in (0, 1):
                m = E.macroscopic(E.el[p], k, row == 0, xk, lk, stepping=True)
                mfp[row, at] = torch.where(m > 0.0, 1.0 / m, torch.full_like(m, big))
            mfp[2, at] = mfp[3, at] = big
            if p == 1:
                tau = 0.8 * xk / 5.1099890999999997e-01
                gam, bg2 = tau + 1.0, tau * (tau + 2.0)
                bg = torch.sqrt(bg2)
                m = E.mats[imat]["fElectronDensity"] * 2.4946724123674787e-23 * (
                    (gam * gam + 4.0 * gam + 1.0) * torch.log(gam + bg) - (gam + 3.0) * bg) / (bg2 * (gam + 1.0))
                mfp[2, at] = 1.0 / m
    return {"howfar.range": ranges, "howfar.mfp": mfp.view(-1)}


def exact(case, seed):
    if case["kind"] == "lookup":
        return _exact_lookup(case, seed)
    if case["kind"] == "gamma":
        return _exact_gamma(case, seed)
    if case["kind"] == "split":
        return _exact_howfar(case, seed)
    return None  # sampled: no value in closed form
