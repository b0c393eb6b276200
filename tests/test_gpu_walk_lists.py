"""The walk's spill lists: bounded in size, complete in content.

A list holds 2^23 particles and 2^20 muons; those past its end are marked
in the store and listed later.  Whatever a launch leaves - unclaimed items,
handed-on particles of the last sweep, stacks - the records are those of a run
of sweeps alone, bit for bit.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd import Shower
from petite_amd.batch import PRIMARY_DTYPE
from petite_amd.constants import mass_dict


def _primaries(parts, seed):
    """parts: (count, pids, lowest and highest kinetic energy)"""
    rng = np.random.default_rng(seed)
    out = []
    for n, pids, lo, hi in parts:
        prim = np.zeros(n, dtype=PRIMARY_DTYPE)
        prim["pid"] = rng.choice(np.array(pids, dtype=np.int32), size=n)
        m = np.select([prim["pid"] == q for q in pids], [mass_dict[q] for q in pids])
        prim["E"] = m + np.exp(rng.uniform(np.log(lo), np.log(hi), n))
        prim["pz"] = np.sqrt(prim["E"] ** 2 - m * m)
        prim["mass"], prim["weight"] = m, 1.0
        out.append(prim)
    prim = rng.permutation(np.concatenate(out))
    prim["sid"] = np.arange(len(prim))
    return prim


def _run(sh, prim, tuning, capacity):
    ctx = sh.device_context()
    base = ctx.get_tuning()
    ctx.set_tuning(dict(base, **tuning))
    try:
        b = sh.generate_showers(prim, seed=9, capacity=capacity)
    finally:
        ctx.set_tuning(base)
    order = torch.argsort(b.sid)
    rec = {k: b.tensor(k)[order] for k in ("sid", "pid", "p0", "r0", "pf", "rf", "meta")}
    parent = b.parent.long()
    rec["parent"] = torch.where(parent >= 0, b.sid[parent.clamp(min=0)], parent)[order]
    return rec, b.stats


def _same(sh, prim, tuning, capacity):
    ref, st = _run(sh, prim, {"tail_sweep": 1}, capacity)
    got, s = _run(sh, prim, tuning, capacity)
    for k in ref:
        assert torch.equal(ref[k], got[k]), k
    for k in ("n_particles", "n_steps", "n_draws", "n_trials", "n_dropped", "n_maxf_viol"):
        assert st[k] == s[k], k
    return st, s


@pytest.fixture(scope="module")
def lead():
    return Shower("100GeV", "lead", 0.010, seed=5)


def _library_bytes():
    """Device memory in use beside torch's."""
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free - torch.cuda.memory_reserved()


def test_a_large_store_needs_no_large_lists(lead):
    prim = _primaries([(100, [11, 22], 0.1, 2.0)], seed=1)
    lead.generate_showers(prim, seed=9, capacity=1 << 23)  # the scratch of every run
    torch.cuda.empty_cache()
    before = _library_bytes()
    lead.generate_showers(prim, seed=9, capacity=1 << 28)
    torch.cuda.empty_cache()
    assert _library_bytes() - before <= 96 << 20


# one iteration's budget: nearly all of the primaries go through the lists
WALK = {"tail_sweep": 1 << 30, "tail_budget": 1}


@pytest.mark.parametrize("name,parts", [
    # fewer than a list's front, more (by less than a block's run of the
    # gathering, and by much), muons more than its back, and both
    ("fits", [(3000001, [11, -11, 22], 0.005, 0.03)]),
    ("just over", [((1 << 23) + 3 * 131072 + 1000, [11, -11, 22], 0.005, 0.03)]),
    ("front", [(10000003, [11, -11, 22], 0.005, 0.03)]),
    ("muons", [(2500001, [13, -13], 0.01, 0.1)]),
    ("both", [(9500000, [11, 22], 0.005, 0.03), (2300007, [13, -13], 0.01, 0.1)])])
def test_particles_past_a_lists_end(lead, name, parts):
    prim = _primaries(parts, seed=3)
    st, s = _same(lead, prim, WALK, 20000000)
    assert s["launches_transport"] == 0 and s["n_iterations"] > 2


def test_marked_particles_beside_empty_lists(lead):
    """Limits double: by the fifth launch, the last of a host check, a launch
    ends a full list's muons, 131,072 lanes' at a time, and the marked ones
    beside it are still to come."""
    n = 6000000
    prim = np.zeros(n, dtype=PRIMARY_DTYPE)
    m = mass_dict[13]
    prim["pid"], prim["mass"], prim["weight"] = 13, m, 1.0
    prim["E"], prim["pz"] = m + 0.001, np.sqrt((m + 0.001) ** 2 - m * m)
    prim["sid"] = np.arange(n)
    st, s = _same(lead, prim, dict(WALK, tail_budget=2), n)
    assert s["n_particles"] == n and s["launches_tail"] > 5


def test_restart_of_handed_on_particles(lead):
    """More handed-on particles than the launch has lanes: those that no wave
    claims go to the list and start over from their records."""
    # (photons below the cutoff end at once: after a sweep fewer particles wait
    # than there were primaries)
    n = 120022
    prim = _primaries([(n // 2, [11, -11], 0.02, 0.05), (n // 2, [22], 0.001, 0.009)], seed=7)
    tuning = {"yield_steps": 2, "sweep_group": 1, "small_sweep": 1, "tail_sweep": n, "tail_waves": 1, "tail_budget": 1}
    st, s = _same(lead, prim, tuning, 8000000)
    rec, _ = _run(lead, prim, tuning, 8000000)
    # one sweep of two substeps, then walks by 16,384 lanes
    assert s["launches_transport"] == 1 and s["n_iterations"] > 3
    assert int(((rec["meta"] == 0) & (rec["rf"][:, 3] > 3)).sum()) > 2 * 16384
