"""Dark entries and yields at the edges of a block: the entries of a record's
first n particles are those of the whole record whose parent is among them
(an entry depends on its particle's stream alone), and the yields are the sums
of the vectors' weights (dark_shower.py:786-804)."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from petite_amd import DarkShower, Particle


@pytest.fixture(scope="module")
def record():
    ds = DarkShower("100GeV", "graphite", 0.010, 0.03, seed=8)
    prims = [Particle([E, 0, 0, math.sqrt(E * E - 2.7e-7)], [0, 0, 0], {"PID": pid})
             for E in np.geomspace(2.0, 60.0, 12) for pid in (11, -11)]
    batch = ds.generate_showers(prims)
    assert batch.n > 1100
    return ds, batch._store, batch.n


def _entries(ds, store, n):
    out, n_e, stats = ds.device_context().dark_reweight(store, n, 8)
    v = {k: out[k][:n_e].cpu().numpy() for k in out}
    o = np.lexsort((v["meta"] & 0xFF, v["parent"]))
    return {k: v[k][o] for k in v}, stats


# less than a wave, than a block; a block; one and four blocks and a particle
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, -1])
def test_entries_of_the_first_records(record, n):
    ds, store, total = record
    n = total if n < 0 else n
    whole = _entries(ds, store, total)[0]
    part, stats = _entries(ds, store, n)
    among = whole["parent"] < n
    for k in whole:
        assert np.array_equal(part[k], whole[k][among]), k
    ok = (part["meta"] & 0x100) != 0
    assert stats["n_vectors"] == ok.sum()
    for code, y in zip(range(8, 12), stats["yield"]):
        w = part["r"][ok & ((part["meta"] & 0xFF) == code), 3].astype(np.float64).sum()
        assert abs(y - w) <= 1.2e-7 * w  # each weight stored rounded to 24 bits
