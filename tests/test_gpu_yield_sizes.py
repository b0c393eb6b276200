"""dark_yield over record sizes and numbers of masses at the edges of its
blocks, groups of masses, passes (32 masses) and parts of a record (2^25
particles), against the oracle (dark_shower.py:595-647 interpolated between
the trained masses); every species, and the processes with and without tables
at each m_V.  Both sides sum float64 values of float32 records: 1e-9."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle.dark import OracleDark, OracleDarkSampler, yield_and_grad
from oracle.tables import SMTables
from petite_amd import DarkShower, _lib
from petite_amd.dark_yield import DarkYield

PROCS = ["DarkBrem", "DarkAnn", "DarkComp", "DarkMuonBrem"]
MASSES = [0.002, 0.003, 0.01, 0.03]
BASE = 509


@pytest.fixture(scope="module")
def model():
    ds = DarkShower("100GeV", "lead", 0.010, 0.01, seed=4)
    m = DarkYield(ds._tables, 0.010, masses=MASSES, active_processes=PROCS, ctx=ds.device_context())
    T = SMTables("lead")
    samplers = [OracleDarkSampler(OracleDark(T, v, with_integrals=False, masses="all"), m.dark[v].W, m.dark[v].D, None)
                for v in m.masses]
    rng = np.random.default_rng(5)
    pid = rng.choice([11, -11, 22, 13, -13, 2112], BASE).astype(np.int32)
    E = np.exp(rng.uniform(np.log(0.008), np.log(60.0), BASE)).astype(np.float32)
    w = rng.uniform(0.1, 2.0, BASE).astype(np.float32)
    return m, samplers, pid, E, w


def _record(pid, E, w, n):
    at = torch.arange(n, device="cuda") % BASE
    p0 = torch.zeros((n, 4), device="cuda")
    r0 = torch.zeros((n, 4), device="cuda")
    p0[:, 0] = torch.from_numpy(E).cuda()[at]
    r0[:, 3] = torch.from_numpy(w).cuda()[at]
    i = torch.from_numpy(pid).cuda()[at]
    return {"p0": p0, "r0": r0, "pf": p0, "rf": r0, "pid": i, "parent": i, "meta": i, "shower": i, "sid": at}, n


def _evaluate(m, record, mv, tables, grad=True):
    m._setup()
    if not tables:  # the trained masses alone: every process interpolated
        _lib.check(m.ctx.lib.petite_yield_setup(m.ctx.ctx, len(m.masses), np.asarray(m.masses).ctypes.data,
                                                _lib.C.cast(m._descs, _lib.C.c_void_p), m._blob.ctypes.data,
                                                m._blob.size), "petite_yield_setup")
    return m.evaluate(record, mv, grad=grad)


def _masses(k):
    # trained masses, the ends of the range and masses between, unordered
    mv = np.concatenate([MASSES, np.geomspace(MASSES[0], MASSES[-1], 80)[1:-1]])[:k]
    return np.random.default_rng(k).permutation(mv)


@pytest.mark.parametrize("n,k", [(0, 3), (1, 1), (63, 8), (256, 9), (257, 32), (4097, 33), (2 ** 25 + 777, 3),
                                 (2 ** 25 + 777, 65)])
def test_interpolated_processes(model, n, k):
    m, samplers, pid, E, w = model
    mv = _masses(k)
    times = np.bincount(np.arange(n % BASE), minlength=BASE) + n // BASE
    Yo, dYo = yield_and_grad(samplers, m.masses, PROCS, pid, E.astype(np.float64), w * times.astype(np.float64), mv)
    rec = _record(pid, E, w, n)
    Y, dY = _evaluate(m, rec, mv, False)
    np.testing.assert_allclose(Y, Yo, rtol=1e-9, atol=0)
    np.testing.assert_allclose(dY, dYo, rtol=1e-9, atol=1e-11 * (np.abs(dYo).max() + 1e-300))
    assert np.abs(_evaluate(m, rec, mv, False, grad=False)[0] - Y).max() <= 1e-12 * np.abs(Y).max()


# the tables at each m_V: the record's yields are those of its repetitions
@pytest.mark.parametrize("n,k", [(257, 4), (4097, 5), (4097, 33), (2 ** 25 + 777, 33)])
def test_tables_at_each_mass(model, n, k):
    m, _, pid, E, w = model
    mv = _masses(k)
    one, rest = (_evaluate(m, _record(pid, E, w, q), mv, True) for q in (BASE, n % BASE))
    Y, dY = _evaluate(m, _record(pid, E, w, n), mv, True)
    for got, a, b in ((Y, one[0], rest[0]), (dY, one[1], rest[1])):
        want = (n // BASE) * a + b
        np.testing.assert_allclose(got, want, rtol=1e-9, atol=1e-11 * np.abs(want).max())
    alone = [float(_evaluate(m, _record(pid, E, w, BASE), [v], True)[0][0]) for v in mv[::7]]
    np.testing.assert_allclose(one[0][::7], alone, rtol=1e-12)
    np.testing.assert_allclose(_evaluate(m, _record(pid, E, w, n), mv, True, grad=False)[0], Y, rtol=1e-12)
