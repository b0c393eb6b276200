"""A walk without a particle budget runs to its end.

tail_budget above 2^30 never stops a wave, one with muons as little as the
others: the first launch walks every muon to its end, and what remains is what
its wave handed on (the muons' other children, a full stack's).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd import Shower
from petite_amd.batch import PRIMARY_DTYPE
from petite_amd.constants import mass_dict


@pytest.mark.parametrize("n", [1, 64, 300])
def test_no_budget_never_stops_a_wave(n):
    sh = Shower("100GeV", "lead", 0.010, seed=5)
    prim = np.zeros(n, dtype=PRIMARY_DTYPE)
    prim["E"], prim["mass"], prim["weight"], prim["pid"] = 60.0, mass_dict[13], 1.0, 13
    prim["pz"] = np.sqrt(prim["E"] ** 2 - prim["mass"] ** 2)
    prim["shower"] = prim["sid"] = np.arange(n)
    ctx = sh.device_context()
    base = ctx.get_tuning()
    runs = {}
    for budget in (16, (1 << 30) + 1):
        ctx.set_tuning(dict(base, tail_sweep=1 << 30, tail_budget=budget))
        try:
            runs[budget] = sh.generate_showers(prim, seed=9)
        finally:
            ctx.set_tuning(base)
    a, b = runs.values()
    assert a.n == b.n and a.stats["n_steps"] == b.stats["n_steps"] and a.stats["n_trials"] == b.stats["n_trials"]
    # n_iterations: the launches that had something to walk.  The muons; the
    # other children of their vertices; stack overflows, if any
    assert a.stats["n_iterations"] > 4
    assert b.stats["n_iterations"] <= 4
