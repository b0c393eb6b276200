"""The work a user of petite_amd has it do, as cases that can be timed.

Each case is one call (or the two calls of a step) of a public entry point on
inputs of a stated size: whole showers (Shower.generate_showers), batched
accept/reject draws (DeviceContext.draw), the dark vectors of a shower record
and of a meson beam (DarkShower.generate_dark_showers), the m_V-continuous
yield with its gradient (DarkShower.dark_yield) and the detector acceptance
(detector.cut_masks).  Sizes follow bench.py's workloads and the tests, scaled
so that a pass stays below a second, and their neighbourhood: one primary,
thousands, tens of thousands; ragged counts; every species; the two table
sets; scattering on and off; few and many detector planes.

Records come back in the order in which the device finished them, which
differs between runs.  A program that wants the same record every time sorts
it by the particles' 64-bit stream ids, or puts a vector at its parent's
place; the passes here do that, into arrays of a size that depends on the case
alone (zeros past the last record), and return every field of every record.
"""
import math

import numpy as np
import torch

from petite_amd import DarkShower, Shower
from petite_amd.batch import PRIMARY_DTYPE, ParticleBatch
from petite_amd.constants import all_process_code, mass_dict
from petite_amd.detector import cut_masks

SPECIES = {"e-": (11,), "photon": (22,), "e-/e+/photon": (11, -11, 22), "mu-/e-": (13, 11)}
# accept/reject draws of a shower by process, as they occur in lead at a 10 MeV cutoff
DRAW_SHARES = (("Brem", 0.75), ("PairProd", 0.21), ("Comp", 0.02), ("Moller", 0.01), ("Ann", 0.005),
               ("Bhabha", 0.005))
DARK_PROCESSES = ("DarkBrem", "DarkAnn", "DarkComp")
# records of a shower per unit of energy over cutoff: value at a 10 MeV cutoff
# and its growth with the cutoff (measured, 0.3-30 GeV); a muon leaves up to 5
RECORDS = {"graphite": (0.71, 0.55), "lead": (1.50, 0.33), "iron": (1.16, 0.42)}
MESONS = {111: 0.1349768, 221: 0.547862}  # GeV
MESON_BR = {111: 0.98823, 221: 0.3936}    # to two photons


def listed():
    return [
        # an interactive look at one shower: the reference's quick-start call
        dict(name="one_electron", kind="showers", material="graphite", tables="100GeV", cutoff=0.010, n=1,
             species="e-", e_lo=10.0, e_hi=10.0, scattering=True),
        # the reference's own timing case, one shower per seed
        dict(name="graphite_1000x10GeV", kind="showers", material="graphite", tables="100GeV", cutoff=0.010, n=1000,
             species="e-", e_lo=10.0, e_hi=10.0, scattering=True),
        # a beam dump's mixed, uneven primaries in one batch: the benchmark's workload
        dict(name="lead_40000_mixed", kind="showers", material="lead", tables="100GeV", cutoff=0.010, n=40000,
             species="e-/e+/photon", e_lo=0.1, e_hi=100.0, scattering=True),
        # photons of meson decays without multiple scattering, a ragged count
        dict(name="iron_3331_photons", kind="showers", material="iron", tables="100GeV", cutoff=0.020, n=3331,
             species="photon", e_lo=1.0, e_hi=60.0, scattering=False),
        # a 400 GeV muon and electron beam: the longest chains of generations
        dict(name="lead_2000x400GeV", kind="showers", material="lead", tables="400GeV", cutoff=0.100, n=2000,
             species="mu-/e-", e_lo=400.0, e_hi=400.0, scattering=True),
        # the sampler alone: a caller's own transport asks for a million vertices
        dict(name="draws_1000003", kind="draws", material="lead", n=1000003, e_lo=0.02, e_hi=50.0, noalloc=False),
        # the same in a serving loop, a few hundred at a time, without allocations
        dict(name="draws_300", kind="draws", material="graphite", n=300, e_lo=0.02, e_hi=50.0, noalloc=True),
        # dark vectors of an existing shower record
        dict(name="dark_2000x10GeV", kind="dark", material="graphite", n=2000, e_lo=10.0, e_hi=10.0, mV=0.03),
        # dark vectors of a meson beam file
        dict(name="mesons_4000000", kind="mesons", n=4000000, mV=0.03),
        # a scan over m_V with its gradient on a fixed record (one step of a fit)
        dict(name="yield_20000_32_masses", kind="yield", material="lead", n=20000, e_lo=1.0, e_hi=20.0, masses=32),
        # acceptance of a large record at three planes with an energy window
        dict(name="detector_30000001_3_planes", kind="detector", n=30000001, planes=3, window=True),
        # a ragged record against a row of planes
        dict(name="detector_1000003_12_planes", kind="detector", n=1000003, planes=12, window=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["showers", "showers", "showers", "draws", "dark", "mesons", "yield", "detector"])
    if kind == "showers":
        species = rng.choice(sorted(SPECIES))
        material = rng.choice(["graphite", "lead", "iron"])
        if species == "mu-/e-":
            e = rng.uniform(50.0, 400.0)
            return dict(kind=kind, material=material, tables="400GeV", cutoff=0.1, n=_log_int(rng, 2, 1500),
                        species=species, e_lo=e, e_hi=e, scattering=True)
        e_lo = math.exp(rng.uniform(math.log(0.05), math.log(10.0)))
        e_hi = e_lo * math.exp(rng.uniform(0.0, math.log(10.0)))
        cutoff = rng.choice([0.010, 0.015, 0.030, 0.100])
        # at most the energy of the largest listed batch per cutoff
        most = 5.0e7 * cutoff / (0.5 * (e_lo + e_hi))
        return dict(kind=kind, material=material, tables="100GeV", cutoff=cutoff,
                    n=_log_int(rng, 1, min(40000.0, most)), species=species, e_lo=e_lo, e_hi=e_hi,
                    scattering=rng.random() < 0.8)
    material = rng.choice(["graphite", "lead", "iron"])
    if kind == "draws":
        noalloc = rng.random() < 0.4
        return dict(kind=kind, material=material, n=_log_int(rng, 1, 16384 if noalloc else 1000000),
                    e_lo=rng.uniform(0.02, 0.1), e_hi=rng.uniform(1.0, 90.0), noalloc=noalloc)
    if kind == "dark":
        e_lo = rng.uniform(1.0, 8.0)
        return dict(kind=kind, material="graphite", n=_log_int(rng, 1, 2000), e_lo=e_lo,
                    e_hi=e_lo + rng.uniform(0.0, 4.0), mV=rng.choice([0.01, 0.03, 0.1]))
    if kind == "mesons":
        return dict(kind=kind, n=_log_int(rng, 100, 4000000), mV=rng.uniform(0.003, 0.12))
    if kind == "yield":
        return dict(kind=kind, material="lead", n=_log_int(rng, 10, 20000), e_lo=rng.uniform(0.5, 2.0),
                    e_hi=rng.uniform(5.0, 20.0), masses=rng.randint(1, 32))
    return dict(kind=kind, n=_log_int(rng, 100, 20000000), planes=rng.randint(1, 12), window=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs --
def _primaries(case, rng):
    """Primaries along +z with 1 mrad of angular spread, log-uniform energies."""
    n = int(case["n"])
    pids = np.array(SPECIES[case.get("species", "e-")], dtype=np.int32)
    pid = rng.choice(pids, size=n) if n > 1 else pids[:1]
    E = np.exp(rng.uniform(math.log(case["e_lo"]), math.log(case["e_hi"]), n))
    m = np.select([pid == q for q in pids], [mass_dict[int(q)] for q in pids])
    tx, ty = rng.normal(0.0, 1e-3, n), rng.normal(0.0, 1e-3, n)
    p = np.sqrt(E * E - m * m) / np.sqrt(tx * tx + ty * ty + 1.0)
    prim = np.zeros(n, dtype=PRIMARY_DTYPE)
    prim["E"], prim["px"], prim["py"], prim["pz"] = E, p * tx, p * ty, p
    prim["mass"], prim["weight"], prim["pid"] = m, 1.0, pid
    prim["shower"] = np.arange(n)
    prim["sid"] = np.arange(n)
    return prim


def _mean_energy(case):
    lo, hi = case["e_lo"], case["e_hi"]
    return lo if hi <= lo * 1.0001 else (hi - lo) / math.log(hi / lo)


def _records(case, energy):
    """Expected records of showers of this total energy."""
    a, b = RECORDS[case["material"]]
    cutoff = case.get("cutoff", 0.010)
    return energy / cutoff * (3.5 if case.get("species") == "mu-/e-" else a * (cutoff / 0.010) ** b)


def _rows(case):
    """Rows that hold the record of any seed: the energies of few primaries vary."""
    n = int(case["n"])
    energy = n * min(case["e_hi"], _mean_energy(case) * (1.0 + 8.0 / math.sqrt(n)))
    pad = 1.5 if case.get("species") == "mu-/e-" else 1.1
    return int(pad * _records(case, energy)) + 2 * n + 256


def _take(t, order, rows=0):
    """Rows of t in the given order, zeros up to `rows`; 16-byte rows as one element each."""
    n = order.numel()
    out = t.new_empty((max(rows, n),) + tuple(t.shape[1:]))
    flat, to = (t, out) if t.dim() == 1 else (t.view(torch.complex128).view(-1), out.view(torch.complex128).view(-1))
    torch.index_select(flat, 0, order, out=to[:n])
    out[n:] = 0
    return out


def _by_stream(batch, rows):
    """The record in the order of the stream ids, zeros past its end; parents
    by their stream ids (-1: none)."""
    order = torch.argsort(batch.sid)
    parent = batch.parent.long()
    parent = torch.where(parent >= 0, batch.sid[parent.clamp(min=0)], parent)
    out = {k: _take(batch.tensor(k), order, rows) for k in ("p0", "r0", "pf", "rf", "pid", "meta", "shower", "sid")}
    out["parent"] = _take(parent, order, rows)
    return out


def _record(shower, case, rng, seed):
    """A shower record as a checkpoint would give it, in the order of the stream ids."""
    batch = shower.generate_showers(_primaries(case, rng), seed=seed)
    order = torch.argsort(batch.sid)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(order.numel(), device=order.device)
    store = {k: _take(batch.tensor(k), order) for k in ("p0", "r0", "pf", "rf", "pid", "meta", "shower", "sid")}
    parent = batch.parent[order].long()
    store["parent"] = torch.where(parent >= 0, rank[parent.clamp(min=0)], parent).int()
    return ParticleBatch(store, batch.n)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _meson_beam(case, seed):
    """3:1 pi0/eta rows (E, px, py, pz) within 20 mrad, on the host as a beam file gives them."""
    rng = np.random.default_rng([int(seed), 7])
    n = int(case["n"])
    pid = np.where(rng.random(n) < 0.75, 111, 221).astype(np.int32)
    m = np.where(pid == 111, MESONS[111], MESONS[221])
    E = np.maximum(np.exp(rng.uniform(math.log(0.2), math.log(120.0), n)), 1.001 * m)
    th, ph = np.abs(rng.normal(0.0, 0.02, n)), rng.uniform(0.0, 2.0 * np.pi, n)
    p = np.sqrt(E * E - m * m)
    return np.stack([E, p * np.sin(th) * np.cos(ph), p * np.sin(th) * np.sin(ph), p * np.cos(th)], axis=1), pid


def _detector_inputs(case, seed):
    """Momenta and points of an m_V = 30 MeV vector beam, and the detector."""
    g = _generator(seed)
    n = int(case["n"])

    def u():
        return torch.rand(n, device="cuda", generator=g)

    E = torch.exp(math.log(0.03) + u() * math.log(100.0 / 0.03))
    th, ph = 0.15 * torch.sqrt(-2.0 * torch.log1p(-u())), 2.0 * math.pi * u()
    P = torch.sqrt(torch.clamp(E * E - 9.0e-4, min=1e-8))
    p = torch.stack([E, P * torch.sin(th) * torch.cos(ph), P * torch.sin(th) * torch.sin(ph), P * torch.cos(th)], 1)
    r = torch.stack([0.02 * (u() - 0.5), 0.02 * (u() - 0.5), 0.5 * u(), u() * 1e-3], 1)
    planes = [1.0 + 0.75 * k for k in range(int(case["planes"]))]
    return p.contiguous(), r.contiguous(), planes, 0.5, 0.01, ((0.1, 50.0) if case["window"] else None)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([int(seed), 3])
    key = int(seed) * 1000003 + 17
    s = {"case": dict(case), "seed": key}
    if kind == "showers":
        s["shower"] = Shower(case["tables"], case["material"], case["cutoff"], seed=key)
        s["shower"].device_context(MS=bool(case["scattering"]))
        s["primaries"] = _primaries(case, rng)
    elif kind == "draws":
        s["ctx"] = Shower("100GeV", case["material"], 0.010, seed=key).device_context()
        n = int(case["n"])
        codes = np.array([all_process_code[P] for P, _ in DRAW_SHARES], dtype=np.int32)
        share = np.array([f for _, f in DRAW_SHARES])
        s["proc"] = torch.from_numpy(rng.choice(codes, size=n, p=share / share.sum()).astype(np.int32)).cuda()
        s["E"] = torch.from_numpy(np.exp(rng.uniform(math.log(case["e_lo"]), math.log(case["e_hi"]), n))).cuda()
        s["sid"] = torch.from_numpy(rng.integers(0, 2 ** 62, n)).cuda()
    elif kind == "dark":
        s["dark"] = DarkShower("100GeV", case["material"], 0.010, case["mV"], seed=key,
                               active_processes=list(DARK_PROCESSES))
        s["record"] = _record(s["dark"], case, rng, key)
    elif kind == "mesons":
        s["dark"] = DarkShower("100GeV", "graphite", 0.010, case["mV"], mode="approx", seed=key,
                               active_processes=["TwoBody_BSMDecay"])
        s["dark"].device_context()
        s["record"] = ParticleBatch.from_arrays(*_meson_beam(case, seed))
    elif kind == "yield":
        s["dark"] = DarkShower("100GeV", case["material"], 0.010, 0.01, seed=key)
        s["record"] = _record(s["dark"], case, rng, key)
        s["mV"] = torch.from_numpy(np.sort(np.exp(rng.uniform(math.log(1.0e-3), math.log(0.1), int(case["masses"])))))
        s["weights"] = torch.from_numpy(rng.uniform(0.5, 1.5, int(case["masses"])))
        s["dark"].dark_yield(s["record"], s["mV"][:1], 1.0)  # the model, kept by the DarkShower
    else:
        s["detector"] = _detector_inputs(case, seed)
    return s


# -------------------------------------------------------------------- pass --
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "showers":
        batch = state["shower"].generate_showers(state["primaries"], seed=state["seed"],
                                                 GlobalMS=bool(case["scattering"]))
        out = _by_stream(batch, _rows(case))
        out["energy"] = batch.energy
        out["steps"] = int(batch.stats["n_steps"])
        return out
    if kind == "draws":
        x, trials, w, _ = state["ctx"].draw(state["proc"], state["E"], state["sid"], state["seed"],
                                            noalloc=bool(case["noalloc"]))
        return {"x": x, "trials": trials, "w": w}
    if kind in ("dark", "mesons"):
        d = state["dark"].generate_dark_showers(state["record"], seed=state["seed"])
        # one place per (SM record, process)
        at, rows = d.parent.long(), int(case["n"])
        if kind == "dark":
            at, rows = at * len(DARK_PROCESSES) + (d.process.long() - 8), _rows(case) * len(DARK_PROCESSES)
        out = {"yields": [float(v) for v in d.stats["yield"]]}
        for k, t in (("p", d.p), ("r", d.tensor("r")), ("process", d.process), ("valid", d.valid)):
            out[k] = t.new_zeros((rows,) + tuple(t.shape[1:]))
            out[k][at] = t
        return out
    if kind == "yield":
        mV = state["mV"].clone().requires_grad_(True)
        eps2 = torch.tensor(1.0e-6, dtype=torch.float64, requires_grad=True)
        Y = state["dark"].dark_yield(state["record"], mV, eps2)
        (Y * state["weights"]).sum().backward()
        return {"yield": Y.detach(), "d_mV": mV.grad, "d_eps2": eps2.grad}
    p, r, planes, radius, inner, window = state["detector"]
    mask, wsum = cut_masks(p, r, planes, radius, window, inner)
    return {"mask": mask, "wsum": wsum}


# -------------------------------------------------------------------- work --
def work(case):
    """Bytes: inputs read and outputs written once.  Operations: floating-point
    operations of the physics.  Counts that depend on the random numbers are
    the means measured with bench.py's workloads (records per unit of energy
    over cutoff; 9 particle-steps and 13 candidates per record)."""
    kind, n = case["kind"], float(case["n"])
    if kind in ("showers", "dark", "yield"):
        rec = n + _records(case, n * _mean_energy(case))
    if kind == "showers":
        return {"bytes": 88.0 * rec + 88.0 * n, "flops": rec * (9.0 * 120.0 + 13.0 * 150.0)}
    if kind == "draws":
        return {"bytes": n * (4 + 8 + 8 + 16 + 4 + 4), "flops": n * 16.0 * 150.0}
    if kind == "dark":
        return {"bytes": rec * (64.0 + 48.0), "flops": rec * 20.0 * 400.0}
    if kind == "mesons":
        return {"bytes": n * 100.0, "flops": n * 150.0}
    if kind == "yield":
        return {"bytes": rec * 12.0, "flops": rec * float(case["masses"]) * 40.0}
    return {"bytes": n * 40.0, "flops": n * (4.0 + 10.0 * float(case["planes"]))}


# ------------------------------------------------------------------- exact --
def _philox(sid, index, purpose, seed):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (sid, index, purpose)."""
    low = np.uint64(0xFFFFFFFF)
    c = [sid & low, sid >> np.uint64(32), np.full_like(sid, index), np.full_like(sid, purpose)]
    k0, k1 = int(seed) & 0xFFFFFFFF, (int(seed) >> 32) & 0xFFFFFFFF
    for _ in range(10):
        a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & low, (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _uniform(word):
    return ((word >> np.uint64(9)).astype(np.float64) + 0.5) * 2.0 ** -23


def _exact_mesons(case, seed):
    """M -> gamma V, isotropic in the meson's frame, boosted along its momentum."""
    p4, pid = _meson_beam(case, seed)
    n = len(pid)
    key, mV = int(seed) * 1000003 + 17, float(case["mV"])
    p4 = p4.astype(np.float32).astype(np.float64)
    m = np.where(pid == 111, MESONS[111], MESONS[221])
    words = _philox(np.arange(n, dtype=np.uint64), 12, 7, key)   # the pair's own stream
    u = _philox(words[0] | (words[1] << np.uint64(32)), 0, 3, key)
    ct, phi = 2.0 * _uniform(u[0]) - 1.0, 2.0 * np.pi * _uniform(u[1])
    st = np.sqrt(1.0 - ct * ct)
    E2, pF = (m * m + mV * mV) / (2.0 * m), (m * m - mV * mV) / (2.0 * m)
    v = np.stack([pF * st * np.sin(phi), pF * st * np.cos(phi), pF * ct], 1)
    gam = p4[:, 0] / m
    beta = np.sqrt(1.0 - 1.0 / (gam * gam))
    b = (beta / np.sqrt((p4[:, 1:] ** 2).sum(1)))[:, None] * p4[:, 1:]
    bv = (b * v).sum(1)
    out = np.empty((n, 4))
    out[:, 0] = gam * (E2 + bv)
    out[:, 1:] = v + b * (gam * E2 + (gam - 1.0) / (beta * beta) * bv)[:, None]
    w = np.where(pid == 111, MESON_BR[111], MESON_BR[221]) * 2.0 * (1.0 - (mV / m) ** 2) ** 3
    r = np.zeros((n, 4))
    r[:, 3] = w
    return {"p": out, "r": r, "process": None, "valid": None,
            "yields": [None, None, None, None, float(w.sum())]}


def _exact_detector(case, seed):
    p, r, planes, radius, inner, window = _detector_inputs(case, seed)
    p, r = p.double(), r.double()
    keep = torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
    if window is not None:
        keep = (p[:, 0] > window[0]) & (p[:, 0] < window[1])
    sums = []
    for z in planes:
        T = (z - r[:, 2]) / p[:, 3]
        rt = torch.sqrt((r[:, 0] + T * p[:, 1]) ** 2 + (r[:, 1] + T * p[:, 2]) ** 2)
        sums.append(r[:, 3][keep & (rt > inner) & (rt < radius)].sum())
    sums.append(r[:, 3][keep].sum())
    return {"mask": None, "wsum": torch.stack(sums)}


def exact(case, seed):
    """64-bit results of the passes that are closed forms.  Showers, draws and
    dark vectors are chains of accept/reject decisions: no closed form.  The
    yield rests on the trained tables: no value without them."""
    if case["kind"] == "mesons":
        return _exact_mesons(case, seed)
    if case["kind"] == "detector":
        return _exact_detector(case, seed)
    return None
