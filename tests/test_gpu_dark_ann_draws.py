"""DarkAnn's draws: candidates judged in float32 first, and requests of up to a
million candidates handed to all the waves of a kernel of their own.

Both must leave the draw of draw_dark_sample (dark_shower.py:649-704): the
first candidate whose float64 J f exceeds max_F u.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import philox
from petite_amd import DarkShower
from petite_amd.constants import all_process_code

SEED = 19
CODE = all_process_code["DarkAnn"]


@pytest.fixture(scope="module", params=[0.003, 0.01, 0.1])
def dark(request):
    ds = DarkShower("100GeV", "graphite", 0.010, request.param, seed=SEED, active_processes=["DarkAnn"])
    return ds, ds.device_context()


def _energies(ds, n):
    lo = ds._resonant_annihilation_energy
    return lo * np.exp(np.random.default_rng(2).uniform(1e-5, np.log(95.0 / lo), n))


def test_first_candidate_above_the_threshold(dark):
    ds, ctx = dark
    E = _energies(ds, 300)
    x, t, w, _ = ctx.draw(np.full(len(E), CODE, np.int32), E, np.arange(len(E)), SEED)
    x, t, w = x.cpu().numpy(), t.cpu().numpy(), w.cpu().numpy()
    grid = ctx.tables_grid("DarkAnn")[0]
    checked = 0
    for i in np.nonzero((t > 0) & (t <= 30000))[0][:120]:
        words = philox.words(SEED, np.uint64(i), np.arange(int(t[i]), dtype=np.uint64), philox.PURPOSE_VEGAS_A)
        xe, we = ctx.eval_points(np.full(len(words), CODE, np.int32), np.full(len(words), E[i]), words)
        ie = min(int(np.argmin(np.abs(grid - E[i]))) + 1, len(grid) - 1)
        above = ctx.maxf["DarkAnn"][ie] * philox.to_uniform(words)[:, 3] < we
        assert np.nonzero(above)[0].tolist() == [t[i] - 1], i
        assert x[i, 0] == np.float32(xe[-1, 0]) and abs(w[i] / we[-1] - 1.0) < 1e-6, i
        checked += 1
    assert checked > 60


# fewer requests than lanes, one per lane group, several per group
@pytest.mark.parametrize("n", [1, 67, 2000, 16384])
def test_handed_on_draws(dark, n):
    ds, ctx = dark
    E = _energies(ds, n)
    a = [v.cpu().numpy() for v in ctx.draw(np.full(n, CODE, np.int32), E, np.arange(n), SEED)[:3]]
    b = [v.cpu().numpy() for v in ctx.draw(np.full(n, CODE, np.int32), E, np.arange(n), SEED, noalloc=True)[:3]]
    ok = b[1] > 0
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    assert np.array_equal(a[0][ok, 0], b[0][ok, 0])
    assert n < 2000 or a[1].max() > 20000
