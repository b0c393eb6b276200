"""DarkAnn's draws at the lowest energies: s barely above m_V^2.

There 1 - x2 = 1 - m_V^2 / (x1 s) is left with few digits in float64, so the
integrand (all_processes.py:400-466) is what float64 makes of it, and the draw
the first candidate whose float64 J f exceeds max_F u (draw_dark_sample,
dark_shower.py:649-704).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import philox
from petite_amd import DarkShower
from petite_amd.constants import all_process_code

SEED = 29
CODE = all_process_code["DarkAnn"]


# relative distance from the threshold energy
@pytest.mark.parametrize("lo,hi", [(1e-14, 1e-12), (1e-12, 1e-10), (1e-10, 1e-8), (1e-8, 1e-5)])
@pytest.mark.parametrize("mV", [0.01, 0.1])
def test_first_candidate_above_the_threshold(mV, lo, hi):
    ds = DarkShower("100GeV", "graphite", 0.010, mV, seed=SEED, active_processes=["DarkAnn"])
    ctx = ds.device_context()
    n = 600
    E = ds._resonant_annihilation_energy * (1.0 + np.exp(np.random.default_rng(5).uniform(np.log(lo), np.log(hi), n)))
    x, t, w, _ = ctx.draw(np.full(n, CODE, np.int32), E, np.arange(n), SEED)
    x, t, w = x.cpu().numpy(), t.cpu().numpy(), w.cpu().numpy()
    grid = ctx.tables_grid("DarkAnn")[0]
    checked = 0
    for i in np.nonzero((t > 0) & (t <= 20000))[0][:200]:
        words = philox.words(SEED, np.uint64(i), np.arange(int(t[i]), dtype=np.uint64), philox.PURPOSE_VEGAS_A)
        xe, we = ctx.eval_points(np.full(len(words), CODE, np.int32), np.full(len(words), E[i]), words)
        ie = min(int(np.argmin(np.abs(grid - E[i]))) + 1, len(grid) - 1)
        above = ctx.maxf["DarkAnn"][ie] * philox.to_uniform(words)[:, 3] < we
        assert np.nonzero(above)[0].tolist() == [t[i] - 1], (mV, i, E[i], t[i])
        assert x[i, 0] == np.float32(xe[-1, 0]) and abs(w[i] / we[-1] - 1.0) < 1e-6, (mV, i)
        checked += 1
    assert checked > 50
