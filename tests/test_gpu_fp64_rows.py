"""The FP64 cluster kernel on member rows against whole entries (whole_cluster_rows): the same pairs, sums in another
order; and whole entries again once a particle has moved skin/2 without a build."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

TOL = 1e-12  # FP64 sums of a few hundred terms in another order


def _same(a, ga, b, gb):
    for k in ("fx", "fy", "fz"):
        assert np.max(np.abs(a[k] - b[k])) <= TOL * np.max(np.abs(b[k])), k
    assert ga.pair_count == gb.pair_count
    assert abs(ga.potential_energy - gb.potential_energy) <= TOL * abs(gb.potential_energy)
    assert abs(ga.virial - gb.virial) <= TOL * abs(gb.virial)


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("n_side,types", [(4, 1), (7, 3), (14, 1), (23, 3)])
def test_rows_give_the_whole_entries_pairs(M, n_side, types):
    announce(f"FP64 member rows M={M} {n_side}^3, {types} types")
    n = n_side ** 3
    a = 0.7 ** (-1.0 / 3.0)
    L = n_side * a
    x, y, z, vx, vy, vz, _ = ap.generate_lattice(5, n, (n_side,) * 3, a, (0, 0, 0), 0.1, 0.9)
    rng = np.random.default_rng(2)
    t = rng.integers(0, types, n).astype(np.int32)
    near = [v + rng.uniform(-0.05, 0.05, n) for v in (x, y, z)]
    far = [v + rng.uniform(-0.25, 0.25, n) for v in (x, y, z)]
    out = []
    for whole in (0, 1):
        with ap.Engine((0, 0, 0), (L,) * 3, 2.5, 0.3, cluster_size=M, whole_cluster_rows=whole,
                       dynamic_rebuild=False, rebuild_frequency=1000) as e:
            e.set_types([1.0, 0.8, 1.2][:types], [1.0, 0.95, 1.05][:types], [1.0] * types)
            e.upload(x, y, z, vx, vy, vz, type=t)
            res = [(e.force(ap.KERNEL_CLUSTER_FP64, globals=True), e.download())]
            assert not e.update_positions(*near)
            res.append((e.force(ap.KERNEL_CLUSTER_FP64, globals=True), e.download()))
            assert e.update_positions(*far)
            res.append((e.force(ap.KERNEL_CLUSTER_FP64, globals=True), e.download()))
            assert e.update_positions(*far)
            e.rebuild(ap.KERNEL_CLUSTER_FP64)
            res.append((e.force(ap.KERNEL_CLUSTER_FP64, globals=True), e.download()))
            e.step(30, 0.002, ap.KERNEL_CLUSTER_FP64)  # no builds on the way
            out.append(res)
    for (ga, a_), (gb, b_) in zip(*out):
        _same(a_, ga, b_, gb)
