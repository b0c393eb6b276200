"""Draws in large batches against the same requests in small ones.

A request's accepted point, candidate count and J f follow from its process,
energy and stream id alone, so a batch of any size must return bit for bit what
calls of a few requests return (those are compared with the oracle in
test_gpu_draw.py).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd.constants import all_process_code
from petite_amd.device import DeviceContext
from petite_amd.tables import MaterialTables

SEED = 77


@pytest.fixture(scope="module")
def ctx():
    return DeviceContext(MaterialTables("lead"), 0.010)


def _draw(ctx, proc, E, sid, noalloc=False):
    x, t, w, _ = ctx.draw(proc, E, sid, SEED, noalloc=noalloc)
    return x.cpu().numpy(), t.cpu().numpy(), w.cpu().numpy()


def _pieces(ctx, proc, E, sid, size):
    parts = [_draw(ctx, proc[i:i + size], E[i:i + size], sid[i:i + size]) for i in range(0, len(E), size)]
    return [np.concatenate(c) for c in zip(*parts)]


# a block hands out the slots of 2,048 requests: its edges, and codes without a map
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n", [1, 255, 257, 2047, 2048, 2049, 6145])
def test_request_slots(ctx, n, noalloc):
    rng = np.random.default_rng(n)
    proc = rng.choice([0, 0, 0, 1, 2, 2, 3, 4, 5, 9, -1, 12], size=n).astype(np.int32)  # 9: no dark map here
    E = np.exp(rng.uniform(np.log(0.02), np.log(80.0), n))
    sid = rng.integers(0, 2 ** 62, n)
    x, t, w = _draw(ctx, proc, E, sid, noalloc)
    has = (proc >= 0) & (proc <= 5)
    assert np.all(t[has] > 0) and np.all(t[~has] == 0) and np.all(w[~has] == 0.0)
    xs, ts, ws = _pieces(ctx, proc, E, sid, 97)
    assert np.array_equal(t, ts)
    assert np.array_equal(w, ws)
    assert np.array_equal(x[has], xs[has])


# a batch whose groups start at 2 to 32 lanes: once no request waits, a wave's
# idle lanes join the open ones (Ann at 60 MeV takes up to 1,000 candidates)
@pytest.mark.parametrize("P, E", [("Ann", 0.06), ("Ann", 95.0), ("Brem", 50.0), ("PairProd", 10.0), ("MuonBrem", 20.0),
                                  ("Comp", 1.0)])
@pytest.mark.parametrize("n", [9001, 40000, 300001])
def test_groups_that_grow(ctx, P, E, n):
    m = min(n, 6000)
    proc = np.full(n, all_process_code[P], dtype=np.int32)
    e = np.full(n, E)
    sid = np.arange(n)
    x, t, w = _draw(ctx, proc, e, sid)
    assert np.all(t > 0)
    for lo in (0, n - m):
        s = slice(lo, lo + m)
        xs, ts, ws = _pieces(ctx, proc[s], e[s], sid[s], 500)  # 64 lanes per request throughout
        assert np.array_equal(t[s], ts)
        assert np.array_equal(w[s], ws)
        assert np.array_equal(x[s], xs)


# one launch for all processes, its blocks shared by their counts: processes
# that hold almost nothing, one that holds everything, the edges of the rule's
# ranges and of a block per request
@pytest.mark.parametrize("shares", [{"Brem": 1.0}, {"Brem": 0.5, "PairProd": 0.3, "Ann": 0.2},
                                    {"Comp": 0.98, "Brem": 0.01, "Ann": 0.005, "MuonBrem": 0.005}], ids=["one", "three", "few"])
@pytest.mark.parametrize("n", [1, 127, 129, 1 << 16, (1 << 16) + 1, (1 << 19) + 1, (1 << 21) + 1])
def test_processes_in_one_launch(ctx, n, shares):
    rng = np.random.default_rng(n)
    proc = rng.choice([all_process_code[P] for P in shares], size=n, p=list(shares.values())).astype(np.int32)
    E = np.exp(rng.uniform(np.log(0.2), np.log(80.0), n))
    sid = rng.integers(0, 2 ** 62, n)
    x, t, w = _draw(ctx, proc, E, sid)
    assert np.all(t > 0)
    some = np.unique(np.concatenate([np.arange(min(n, 300)), rng.integers(0, n, 1500)]))
    xs, ts, ws = _pieces(ctx, proc[some], E[some], sid[some], 61)
    assert np.array_equal(t[some], ts) and np.array_equal(w[some], ws) and np.array_equal(x[some], xs)
