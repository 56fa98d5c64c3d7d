"""Member rows where clusters are long (dilute boxes, films in vacuum), with particles that are not numbers, and after
steps without builds: the FP64 cluster kernel on them against whole entries, the FP32 one on its pairs."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

TOL = 1e-12  # FP64 sums in another order


def _pairs_inside(n, box, M, rc, seed):
    """n particles in pairs whose separations lie just inside rc (or, one in four, just outside), each across the
    border of two towers along x: its particles are of different clusters."""
    rng = np.random.default_rng(seed)
    h = n // 2
    side = np.cbrt(M / (n / np.prod(box)))
    nt = int(np.ceil(box[0] / side))
    a = np.stack([rng.uniform(rc, b - rc, h) for b in box])
    a[0] = rng.integers(1, nt, h) * (box[0] / nt) - 0.2 * rc
    d = rng.standard_normal((3, h))
    d[0] = np.abs(d[0]) + 1.0 * np.linalg.norm(d[1:], axis=0)
    d /= np.linalg.norm(d, axis=0)
    inside = rng.random(h) < 0.75
    r = rc * np.where(inside, 1.0 - 10.0 ** rng.uniform(-8, -5, h), 1.0 + 10.0 ** rng.uniform(-8, -5, h))
    p = np.concatenate([a, a + r * d], axis=1)[:, rng.permutation(2 * h)]
    return [np.ascontiguousarray(v) for v in p]


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("box", [(900.0,) * 3, (3e4,) * 3, (3e5,) * 3, (3e5, 70.0, 5e4)])
@pytest.mark.parametrize("skin", [0.0, 1e-4])
def test_no_pair_is_lost_in_long_clusters(M, box, skin):
    announce(f"member rows M={M} in a dilute box {box}, skin {skin}")
    rc, n = 2.5, 600
    p = _pairs_inside(n, box, M, rc, 7)
    d2 = sum((v[:, None] - v[None, :]) ** 2 for v in p)
    expect = int(np.sum(np.triu(d2 <= rc * rc, 1)))
    assert expect >= n // 3
    out = {}
    for kernel in (ap.KERNEL_CLUSTER_FP64, ap.KERNEL_CLUSTER_MIXED):
        for whole in (False, True):
            with ap.Engine((0, 0, 0), box, rc, skin, cluster_size=M, whole_cluster_rows=whole) as e:
                e.upload(*p)
                g = e.force(kernel, globals=True)
                out[kernel, whole] = g, e.download()
        (ga, fa), (gb, fb) = out[kernel, False], out[kernel, True]
        assert ga.pair_count == gb.pair_count == expect
        for k in ("fx", "fy", "fz"):
            if kernel == ap.KERNEL_CLUSTER_FP64:
                assert np.max(np.abs(fa[k] - fb[k])) <= TOL * np.max(np.abs(fb[k])), k
            assert np.array_equal(fa[k] != 0.0, fb[k] != 0.0), k


@pytest.mark.parametrize("M", [2, 4, 8])
@pytest.mark.parametrize("bad", [(np.nan, 0.0, 0.0), (0.0, 0.0, np.nan), (np.nan, np.nan, np.nan)])
def test_not_a_number_is_not_hidden(M, bad):
    announce(f"FP64 member rows M={M}, one particle displaced by {bad}")
    n_side, a = 8, 0.7 ** (-1.0 / 3.0)
    L = n_side * a
    x, y, z, _, _, _, _ = ap.generate_lattice(5, n_side ** 3, (n_side,) * 3, a, (0, 0, 0), 0.1, 0.9)
    at = 77
    for v, b in zip((x, y, z), bad):
        v[at] += b
    res = []
    for whole in (False, True):
        with ap.Engine((0, 0, 0), (L,) * 3, 2.5, 0.3, cluster_size=M, whole_cluster_rows=whole) as e:
            e.upload(x, y, z)
            g = e.force(ap.KERNEL_CLUSTER_FP64, globals=True)
            res.append((g, e.download()))
    (ga, fa), (gb, fb) = res
    for k in ("fx", "fy", "fz"):
        assert np.array_equal(np.isnan(fa[k]), np.isnan(fb[k])), k
        ok = ~np.isnan(fb[k])
        assert np.max(np.abs(fa[k][ok] - fb[k][ok]), initial=0.0) <= TOL * np.max(np.abs(fb[k][ok]), initial=1.0), k
    if not all(np.isnan(bad)):  # (with no coordinate at all it may stand alone in a cluster without a box)
        assert any(np.isnan(fa[k][at]) for k in ("fx", "fy", "fz"))
    assert ga.pair_count == gb.pair_count
    assert np.isnan(ga.virial) == np.isnan(gb.virial)


@pytest.mark.parametrize("M", [4, 8])
def test_whole_entries_after_steps_without_builds(M):
    # no builds on the way, and particles that move several skin/2: rows of the first build miss pairs by then
    announce(f"FP64 cluster kernel M={M} after steps without builds")
    n_side, a = 9, 0.5 ** (-1.0 / 3.0)
    L = n_side * a
    x, y, z, vx, vy, vz, _ = ap.generate_lattice(5, n_side ** 3, (n_side,) * 3, a, (0, 0, 0), 0.05, 4.0)
    res = []
    for whole in (False, True):
        with ap.Engine((0, 0, 0), (L,) * 3, 2.5, 0.1, cluster_size=M, whole_cluster_rows=whole,
                       dynamic_rebuild=False, rebuild_frequency=1000) as e:
            e.upload(x, y, z, vx, vy, vz)
            e.step(40, 0.002, ap.KERNEL_CLUSTER_FP64)
            res.append((e.force(ap.KERNEL_CLUSTER_FP64, globals=True), e.download()))
    (ga, fa), (gb, fb) = res
    moved = np.sqrt(sum((fb[k] - v) ** 2 for k, v in zip("xyz", (x, y, z))))
    assert np.mean(moved >= 0.05) > 0.5
    # the two runs add the same pairs in the same order, step for step
    assert ga.pair_count == gb.pair_count
    for k in fb:
        assert np.array_equal(fa[k], fb[k]), k
