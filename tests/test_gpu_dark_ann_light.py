"""DarkAnn's draws close above m_V = 2 m_e.

There the final-state velocity beta_f = sqrt(1 - 4 m_e^2 / m_V^2) is a
difference of nearly equal numbers.  A draw must be that of draw_dark_sample
(dark_shower.py:649-704) with the integrand in float64 (all_processes.py:400-466):
the first candidate whose J f exceeds max_F u.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import philox
from petite_amd import DarkShower
from petite_amd.constants import all_process_code

SEED = 23
CODE = all_process_code["DarkAnn"]


@pytest.mark.parametrize("mV", [0.001021998, 0.001022, 0.00102205, 0.00103, 0.0012])
def test_first_candidate_above_the_threshold(mV):
    ds = DarkShower("100GeV", "graphite", 0.010, mV, mode="approx", seed=SEED, active_processes=["DarkAnn"])
    ctx = ds.device_context()
    n = 4000
    E = np.exp(np.random.default_rng(3).uniform(np.log(0.02), np.log(95.0), n))
    x, t, w, _ = ctx.draw(np.full(n, CODE, np.int32), E, np.arange(n), SEED)
    x, t, w = x.cpu().numpy(), t.cpu().numpy(), w.cpu().numpy()
    grid = ctx.tables_grid("DarkAnn")[0]

    def candidates(i, first, last):
        words = philox.words(SEED, np.uint64(i), np.arange(first, last, dtype=np.uint64), philox.PURPOSE_VEGAS_A)
        xe, we = ctx.eval_points(np.full(len(words), CODE, np.int32), np.full(len(words), E[i]), words)
        ie = min(int(np.argmin(np.abs(grid - E[i]))) + 1, len(grid) - 1)
        return xe, we, ctx.maxf["DarkAnn"][ie] * philox.to_uniform(words)[:, 3] < we

    got = np.nonzero(t > 0)[0]
    assert len(got) > n // 2
    # the accepted candidates are above the threshold: the float64 rule takes them
    for i in got[:400]:
        xe, we, above = candidates(i, int(t[i]) - 1, int(t[i]))
        assert above[0], (mV, i, E[i], t[i])
        assert x[i, 0] == np.float32(xe[0, 0]) and abs(w[i] / we[0] - 1.0) < 1e-6, (mV, i)
    # and none before them is
    few = got[np.argsort(t[got], kind="stable")][:400]
    assert t[few].max() < 100000
    for i in few:
        above = candidates(i, 0, int(t[i]))[2]
        assert np.nonzero(above)[0].tolist() == [t[i] - 1], (mV, i, E[i], t[i])
