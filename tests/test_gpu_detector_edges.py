"""detector_cut at the edges of its plane counts (sums in registers up to 8 and
16 planes), of its blocks, and of the radii: masks equal to the oracle's
(shower.py:815-865) bit for bit, also where the transverse radius is a radius
of the cut or a neighbouring double, sums to the rounding of their order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import detector as od
from petite_amd.detector import cut_masks


def _records(n):
    rng = np.random.default_rng(n)
    p = rng.normal(0.0, 0.3, (n, 4)).astype(np.float32)
    p[:, 0] = rng.uniform(0.01, 20.0, n)
    p[:, 3] = 1.0
    r = rng.normal(0.0, 0.2, (n, 4)).astype(np.float32)
    r[:, 3] = rng.uniform(0.0, 2.0, n)
    k = min(n, 64)  # from the origin: the radius at plane z is z |px|, on an edge at z = 1
    p[:k, 1] = np.float32(0.5) * (1.0 + np.arange(-(k // 2), k - k // 2) * 2.0 ** -24)
    p[:k, 2] = 0.0
    r[:k, :3] = 0.0
    return p, r


@pytest.mark.parametrize("radius, inner", [(0.5, 0.0), (0.7, 0.5), (float(np.float32(0.1)), -1.0), (np.inf, 0.25), (0.0, 0.0),
                                           (1e200, 1e-170), (np.sqrt(0.5), np.nextafter(0.5, 0.0))])
@pytest.mark.parametrize("n, planes", [(1, 1), (255, 8), (65537, 9), (300001, 16), (4097, 17), (2100003, 3), (3000, 64)])
def test_masks_and_sums(n, planes, radius, inner):
    p, r = _records(n)
    z = [1.0] + list(np.linspace(0.25, 12.0, planes - 1))
    mask, wsum = cut_masks(torch.from_numpy(p).cuda(), torch.from_numpy(r).cuda(), z, radius, (0.05, 15.0), inner)
    with np.errstate(all="ignore"):
        win, ok = od.pass_matrix(p.astype(np.float64), r.astype(np.float64), z, radius, inner, (0.05, 15.0))
    m = mask.cpu().numpy().view(np.uint64)
    w = r[:, 3].astype(np.float64)
    s = wsum.cpu().numpy()
    for d in range(planes):
        assert np.array_equal(((m >> np.uint64(d)) & np.uint64(1)).astype(bool), ok[d]), d
        assert abs(s[d] - w[ok[d]].sum()) <= 1e-12 * w.sum()
    assert abs(s[planes] - w[win].sum()) <= 1e-12 * w.sum()
