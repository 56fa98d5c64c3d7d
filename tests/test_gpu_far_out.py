"""j-row builds with particles that a wrap does not bring back into the box: a cluster of such particles lists no
other cluster, and its row is its own members.  The other particles' forces are those without the far ones."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.3


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("dims", [(7, 7, 10), (14, 14, 20)])
@pytest.mark.parametrize("far", ["above", "below", "infinite"])
def test_rows_of_clusters_outside_the_box(oracle, M, dims, far):
    announce(f"j-rows, M={M}: lattice {dims}, 16 particles far out ({far})")
    a = 0.75 ** (-1.0 / 3.0)
    n = int(np.prod(dims))
    x, y, z, _, _, _, _ = ap.generate_lattice(3, n, dims, a, (0.0, 0.0, 0.0), 0.05, 0.9)
    # the lattice fills the middle of a tall box; the far ones stand in one column, whose images in the box are in
    # the empty end, farther than rc from the lattice
    L = (dims[0] * a, dims[1] * a, dims[2] * a + 20.0)
    z = z + 5.0
    k = np.arange(16)
    zf = {"above": 3.0 * L[2], "below": -5.0 * L[2], "infinite": np.inf}[far] + L[2] - 8.0 + 0.05 * k
    xs, ys = np.concatenate([x, np.full(16, 0.4)]), np.concatenate([y, np.full(16, 0.4)])
    zs = np.concatenate([z, zf])
    with ap.Engine((0.0, 0.0, 0.0), L, RC, SKIN, cluster_size=M) as e:
        e.upload(xs, ys, zs)
        for _ in range(2):  # the first build, and one from the cluster layout
            e.rebuild(ap.KERNEL_CLUSTER_JROWS_MIXED)
            e.force(ap.KERNEL_CLUSTER_JROWS_MIXED, globals=False)
            f, g = e.download(), e.clusters()
            sp, off, lj = g["slot_particle"], g["list_offsets"], g["list_j"]
            for c in range(len(off) - 1):
                row = lj[off[c]:off[c + 1]].tolist()
                assert len(row) == len(set(row)), c
                assert {int(p) for p in sp[c * M:(c + 1) * M] if p >= 0} <= set(row), c
            ref = oracle.direct_sum(x, y, z, RC, box_len=L)
            num = sum(np.sum((f[d][:n] - ref[d]) ** 2) for d in ("fx", "fy", "fz"))
            den = sum(np.sum(ref[d] ** 2) for d in ("fx", "fy", "fz"))
            assert np.sqrt(num / den) <= 1e-5
