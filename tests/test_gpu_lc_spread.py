"""The FP64 LinkedCells kernels where the particles are spread over the cells in other ways than a liquid's: many empty
cells, few full ones, full ones among many empty, a droplet in vacuum; against the direct sum, or (large) against the
FP64 cluster kernel.  The sizes are chosen so that each way of finding the work is taken, and at its edges."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

# FP64 throughout: the bar of the FP64 kernels against the direct sum
TOL = 1e-10


def _fill(n, lo, hi, seed):
    """n particles on a jittered lattice in [lo, hi), in random order."""
    rng = np.random.default_rng(seed)
    lo, edge = np.asarray(lo, dtype=float), np.asarray(hi, dtype=float) - np.asarray(lo, dtype=float)
    dims = np.ceil(edge / (np.prod(edge) / n) ** (1 / 3) - 1e-9).astype(np.int64)
    while np.prod(dims) < n:
        dims[np.argmax(edge / dims)] += 1
    idx = np.stack(np.unravel_index(rng.permutation(int(np.prod(dims)))[:n], dims))
    return lo[:, None] + (idx + rng.uniform(0.45, 0.55, (3, n))) * (edge / dims)[:, None]


def _run(pos, box, rc, sig, types, kernel=ap.KERNEL_LC_FP64, owned=None):
    t = np.random.default_rng(5).integers(0, types, pos.shape[1]).astype(np.int32)
    eps = np.linspace(0.8, 1.2, types) if types > 1 else np.ones(1)
    sg = sig * (np.linspace(0.95, 1.05, types) if types > 1 else np.ones(1))
    with ap.Engine((0, 0, 0), box, rc, 0.3, cluster_size=8) as e:
        e.set_types(eps, sg, np.ones(types))
        e.upload(*pos, type=t)
        if owned is not None:
            e.set_owned(owned)
        g = e.force(kernel, globals=True)
        return g, e.download(), (t, eps, sg)


def _compare(g, f, ref, pairs, epot, virial):
    num = sum(np.sum((f[k] - ref[k]) ** 2) for k in ("fx", "fy", "fz"))
    den = sum(np.sum(ref[k] ** 2) for k in ("fx", "fy", "fz"))
    assert g.pair_count == pairs
    assert np.sqrt(num) <= TOL * max(np.sqrt(den), 1e-3)
    assert abs(g.potential_energy - epot) <= TOL * max(abs(epot), 1e-3)
    assert abs(g.virial - virial) <= TOL * max(abs(virial), 1e-3)


@pytest.mark.parametrize("types", [1, 3])
@pytest.mark.parametrize("name,n,box,region,rc,sig", [
    ("sparse", 1, (30.0, 30.0, 30.0), None, 2.5, 1.0),
    ("sparse", 63, (30.0, 40.0, 50.0), None, 2.5, 1.0),
    ("sparse", 2049, (60.0, 57.0, 63.0), None, 2.5, 1.0),
    ("sparse, two cells a side", 11, (5.7, 5.7, 30.0), None, 2.5, 1.0),
    ("thin", 8191, (32.0, 33.0, 34.0), None, 2.5, 1.0),
    ("thin", 8200, (34.0, 33.0, 34.0), None, 2.5, 1.0),
    ("cells of 40 and 41", 1100, (8.4, 8.4, 8.4), None, 2.5, 0.5),
    ("one full cell", 900, (3.0, 3.0, 3.0), None, 2.5, 0.2),
    ("eight full cells", 2500, (6.0, 6.0, 6.0), None, 2.5, 0.25),
    ("full cells in a corner", 3001, (25.3, 25.3, 25.3), ((1, 1, 1), (7, 7, 7)), 2.5, 0.25),
    ("full cells in a corner, long cutoff", 3500, (60.0, 60.0, 60.0), ((20, 20, 20), (35, 35, 35)), 6.0, 0.8),
    ("film", 4000, (17.0, 17.0, 120.0), ((0, 0, 50), (17, 17, 70)), 2.5, 0.8),
    ("droplet", 3000, (90.0, 90.0, 90.0), ((40, 40, 40), (56, 56, 56)), 2.5, 0.9),
])
def test_any_spread(oracle, name, n, box, region, rc, sig, types):
    announce(f"LC FP64 kernels, {name}: {n} particles in {box}, cutoff {rc}, {types} types")
    pos = _fill(n, *(region if region else ((0, 0, 0), box)), seed=n)
    g, f, (t, eps, sg) = _run(pos, box, rc, sig, types)
    ref = oracle.direct_sum(*pos, rc, box_len=box, types=t, eps=eps, sig=sg)
    _compare(g, f, ref, ref["pairs"], ref["epot"], ref["virial"])


@pytest.mark.parametrize("n,box,region,types", [
    (30011, (60.0, 60.0, 60.0), None, 1),                          # lanes and slices in one launch
    (150001, (70.0, 81.0, 90.0), None, 3),
    (262144, (106.0, 106.0, 106.0), None, 1),                      # the last of one launch, the first of two
    (262145, (106.0, 106.0, 106.0), None, 3),
    (300000, (300.0, 300.0, 300.0), ((0, 0, 0), (75, 75, 75)), 1),  # a full corner of an empty box
])
def test_many_particles(n, box, region, types):
    announce(f"LC FP64 kernels: {n} particles in {box}, {types} types, against the FP64 cluster kernel")
    pos = _fill(n, *(region if region else ((0, 0, 0), box)), seed=n)
    owned = n // 2 if types > 1 else None
    g, f, _ = _run(pos, box, 2.5, 1.0, types, owned=owned)
    # (the same particles in less empty space, which is all the clusters' towers hold)
    tight = tuple(r + 5.0 for r in region[1]) if region else box
    h, ref, _ = _run(pos, tight, 2.5, 1.0, types, ap.KERNEL_CLUSTER_FP64, owned=owned)
    _compare(g, f, ref, h.pair_count, h.potential_energy, h.virial)
