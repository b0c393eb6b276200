"""The walk of a run's particles (k_tail) against the sweeps.

Every particle draws from its own Philox stream, so a walk at any point of a
run, with any stack, budget and number of waves, must leave the records of a
run of sweeps alone, bit for bit, and the same counts.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd import Shower
from petite_amd.batch import PRIMARY_DTYPE
from petite_amd.constants import mass_dict


def _primaries(n, e_lo, e_hi, pids, seed):
    rng = np.random.default_rng(seed)
    prim = np.zeros(n, dtype=PRIMARY_DTYPE)
    pid = rng.choice(np.array(pids, dtype=np.int32), size=n)
    m = np.array([mass_dict[int(q)] for q in pid])
    E = np.exp(rng.uniform(np.log(e_lo), np.log(e_hi), n))
    prim["E"], prim["pz"], prim["mass"], prim["weight"], prim["pid"] = E, np.sqrt(E * E - m * m), m, 1.0, pid
    prim["shower"] = np.arange(n)
    prim["sid"] = np.arange(n)
    return prim


def _run(sh, prim, tuning, capacity=None):
    ctx = sh.device_context()
    base = ctx.get_tuning()
    ctx.set_tuning(dict(base, **tuning))
    try:
        b = sh.generate_showers(prim, seed=9, capacity=capacity)
    finally:
        ctx.set_tuning(base)
    a = b.to_numpy()
    order = np.argsort(a["sid"], kind="stable")
    parent = np.where(a["parent"] >= 0, a["sid"][np.maximum(a["parent"], 0)], 0)
    rec = {k: a[k][order] for k in ("sid", "pid", "p0", "r0", "pf", "rf", "meta", "shower")}
    return dict(rec, parent=parent[order]), b.energy.cpu().numpy(), b.stats


# one lane; a wave; more items than lanes of the launch; muons; photons and
# particles below the cutoff
BATCHES = {"one": (1, 5.0, 5.0, [11]), "wave": (65, 0.05, 3.0, [11, -11, 22]), "many": (20011, 0.012, 0.2, [11, -11, 22]),
           "muons": (9, 2.0, 40.0, [13, -13]), "low": (257, 0.002, 0.05, [22, 11])}
# a walk from the start; with every stack limit, budget and width at its
# smallest; after some sweeps, with handed-on particles among its items
WALKS = {"start": {"tail_sweep": 1 << 30}, "smallest": {"tail_sweep": 1 << 30, "tail_depth": 1, "tail_budget": 1,
                                                        "tail_waves": 1},
         "no limit": {"tail_sweep": 1 << 30, "tail_budget": (1 << 30) + 1},
         "handed on": {"yield_steps": 2, "sweep_group": 1, "small_sweep": 1}}


@pytest.fixture(scope="module")
def lead():
    return Shower("100GeV", "lead", 0.010, seed=5)


@pytest.mark.parametrize("batch", BATCHES)
def test_walk_leaves_the_sweeps_records(lead, batch):
    prim = _primaries(*BATCHES[batch], seed=4)
    ref, energy, st = _run(lead, prim, {"tail_sweep": 1})
    assert st["launches_tail"] == 0 and st["launches_transport"] > 0
    for name, tuning in WALKS.items():
        if name == "handed on":  # sweeps until fewer particles wait than there were primaries
            tuning = dict(tuning, tail_sweep=len(prim))
        got, e, s = _run(lead, prim, tuning)
        assert (s["launches_transport"] > 0) == (name == "handed on"), name
        assert s["launches_tail"] > 0 or len(prim) == 1, name
        for k in ref:
            assert np.array_equal(ref[k], got[k]), (batch, name, k)
        assert np.allclose(energy, e, rtol=1e-12, atol=1e-12), (batch, name)
        for k in ("n_particles", "n_steps", "n_draws", "n_trials", "n_dropped", "n_maxf_viol", "n_draws_proc",
                  "n_trials_proc", "n_viol_proc"):
            assert st[k] == s[k], (batch, name, k)


# muons have waves and a list of their own: one muon; one of them and other
# particles in a wave; more than a lane each in every second wave of a launch
MUONS = {"one": (1, 60.0, 60.0, [13]), "mixed": (1500, 0.02, 20.0, [13, -13, 11, 22]), "many": (9001, 0.2, 1.5, [13, -13])}


@pytest.mark.parametrize("batch", MUONS)
def test_muons_walk_apart(lead, batch):
    prim = _primaries(*MUONS[batch], seed=6)
    ref, energy, st = _run(lead, prim, {"tail_sweep": 1})
    for name, tuning in WALKS.items():
        if name == "handed on":
            tuning = dict(tuning, tail_sweep=len(prim) + 1)
        got, e, s = _run(lead, prim, dict(tuning, tail_waves=1))
        for k in ref:
            # the bits: a muon below its rest mass has no momentum
            assert ref[k].tobytes() == got[k].tobytes(), (batch, name, k)
        assert np.allclose(energy, e, rtol=1e-12, atol=1e-12), (batch, name)
        for k in ("n_particles", "n_steps", "n_draws", "n_trials", "n_dropped", "n_maxf_viol"):
            assert st[k] == s[k], (batch, name, k)


# a store with room for 2^26 records: the walk that is held to three waves' registers
@pytest.mark.parametrize("batch", ["one", "wave", "many", "low"])
def test_walk_of_a_large_store(lead, batch):
    prim = _primaries(*BATCHES[batch], seed=8)
    ref, energy, st = _run(lead, prim, {"tail_sweep": 1})
    for name in ("start", "smallest"):
        got, e, s = _run(lead, prim, WALKS[name], capacity=1 << 26)
        for k in ref:
            assert ref[k].tobytes() == got[k].tobytes(), (batch, name, k)
        assert np.allclose(energy, e, rtol=1e-12, atol=1e-12), (batch, name)
        for k in ("n_particles", "n_steps", "n_draws", "n_trials", "n_dropped", "n_maxf_viol"):
            assert st[k] == s[k], (batch, name, k)
