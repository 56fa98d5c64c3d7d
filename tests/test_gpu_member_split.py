"""The fused force launch of small systems splits a cluster's members over groups of lanes: steps with one and with
several types are those of a context whose launches are too large to be split, to the bit (an ensemble of copies)."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

KEYS = ("x", "y", "z", "vx", "vy", "vz", "fx", "fy", "fz")


@pytest.mark.parametrize("types", [1, 3])
@pytest.mark.parametrize("M,groups,n_side", [(8, 1, 6), (8, 1, 9), (8, 4, 21), (8, 2, 25), (4, 2, 8), (4, 4, 13)])
def test_split_launches_match_unsplit(M, groups, n_side, types):
    # copies enough for more than 384 workgroups (M 8) or 256 (M 4): the largest unsplit limits
    n = n_side ** 3
    copies = (385 * 4 * groups * M) // n + 1
    announce(f"split force M={M} G={groups} {n} particles, {types} types, against {copies} copies")
    a = 0.75 ** (-1.0 / 3.0)
    L = n_side * a
    x, y, z, vx, vy, vz, _ = ap.generate_lattice(3, n, (n_side,) * 3, a, (0, 0, 0), 0.05, 0.9)
    t = np.random.default_rng(1).integers(0, types, n).astype(np.int32)
    eps, sig = [1.0, 0.8, 1.2][:types], [1.0, 0.95, 1.05][:types]
    with ap.Engine((0, 0, 0), (L,) * 3, 2.5, 0.3, cluster_size=M, tile_groups=groups) as e:
        e.set_types(eps, sig, [1.0] * types)
        e.upload(x, y, z, vx, vy, vz, type=t)
        e.step(25, 0.002, ap.KERNEL_CLUSTER_MIXED)
        one = e.download()
    with ap.Engine((0, 0, 0), (L,) * 3, 2.5, 0.3, cluster_size=M, tile_groups=groups) as e:
        e.set_types(eps, sig, [1.0] * types)
        e.set_boxes(np.zeros((copies, 3)), np.full((copies, 3), L), [n] * copies)
        e.upload(*(np.tile(v, copies) for v in (x, y, z, vx, vy, vz)), type=np.tile(t, copies))
        e.step(25, 0.002, ap.KERNEL_CLUSTER_MIXED)
        all_ = e.download()
    for k in KEYS:
        assert np.array_equal(all_[k].reshape(copies, n), np.broadcast_to(one[k], (copies, n))), k
