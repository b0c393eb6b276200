"""The walk held to three waves' registers: batches of 2.5e7 cutoffs of energy
and more, whatever their store's size, leave the records of a run of sweeps
alone, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd import Shower
from petite_amd.batch import PRIMARY_DTYPE
from petite_amd.constants import mass_dict


# below the rule's line, above it, and above it with particles that do not shower
@pytest.mark.parametrize("n,e,others", [(230001, 1.0, 0), (270001, 1.0, 0), (9000, 31.0, 500)])
def test_large_batches(n, e, others):
    sh = Shower("100GeV", "graphite", 0.010, seed=5)
    rng = np.random.default_rng(n)
    prim = np.zeros(n, dtype=PRIMARY_DTYPE)
    prim["pid"] = rng.choice(np.array([11, -11, 22], dtype=np.int32), size=n)
    prim["pid"][:others] = 14
    m = np.array([mass_dict.get(int(q), 0.0) for q in prim["pid"]])
    prim["E"], prim["pz"], prim["mass"], prim["weight"] = e, np.sqrt(e * e - m * m), m, 1.0
    prim["shower"] = prim["sid"] = np.arange(n)
    ctx = sh.device_context()
    base = ctx.get_tuning()
    runs = []
    for sweep in (1, 1 << 30):
        ctx.set_tuning(dict(base, tail_sweep=sweep))
        try:
            b = sh.generate_showers(prim, seed=9, capacity=40000000)
        finally:
            ctx.set_tuning(base)
        order = torch.argsort(b.sid)
        parent = b.parent.long()
        rec = {k: b.tensor(k)[order] for k in ("sid", "pid", "p0", "r0", "pf", "rf", "meta", "shower")}
        rec["parent"] = torch.where(parent >= 0, b.sid[parent.clamp(min=0)], parent)[order]
        runs.append((rec, b.energy, b.stats))
    (ref, energy, st), (got, e1, s) = runs
    assert st["launches_tail"] == 0 and s["launches_transport"] == 0
    for k in ref:
        assert torch.equal(ref[k], got[k]), k
    assert torch.allclose(energy, e1, rtol=1e-12, atol=1e-12)
    for k in ("n_particles", "n_steps", "n_draws", "n_trials", "n_dropped", "n_maxf_viol"):
        assert st[k] == s[k], k
