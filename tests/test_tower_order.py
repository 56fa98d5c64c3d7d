"""The order of a tower's particles under coordinates that are not numbers, infinities and equal ids.

CPU: ljg_order.h gives a total order, and its FP32 word is monotone in it: what the sorts that rank need so that
every place of a tower is taken once.  GPU: cluster builds of every sort (one workgroup, registers, ranked parts,
LDS) on such particles hold each particle once and give the others back unchanged."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

HERE = os.path.dirname(os.path.abspath(__file__))
NAN, INF = float("nan"), float("inf")


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("order") / "tower_order.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-ffp-contract=off", "-shared", "-fPIC",
                    os.path.join(HERE, "cpp", "tower_order.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _towers():
    rng = np.random.default_rng(5)
    yield [0.5, NAN, 0.2, 0.9], np.arange(4)
    yield [NAN] * 5, np.arange(5)[::-1].copy()
    yield [0.0, -0.0, 0.0, -0.0], np.array([3, 1, 1, 3])
    yield [INF, 1e39, NAN, -INF, 1e300, NAN, INF], np.zeros(7)
    for n in (63, 200):
        z = rng.uniform(0.0, 9.0, n)
        z[rng.random(n) < 0.2] = NAN
        z[rng.random(n) < 0.1] = rng.choice([INF, -INF])
        z[rng.random(n) < 0.3] = 4.25  # equal
        z[rng.random(n) < 0.2] += 1e-9  # equal as FP32 words only
        yield z, rng.integers(0, n // 2, n)


def test_order_is_total(order):
    for z, ids in _towers():
        z, ids = np.array(z, dtype=np.float64), np.array(ids, dtype=np.int64)
        n = len(z)
        b = np.zeros((n, n), dtype=np.uint8)
        order.tower_before_matrix(n, _ptr(z), _ptr(ids), _ptr(b))
        off = ~np.eye(n, dtype=bool)
        assert not b.diagonal().any()
        assert np.array_equal((b + b.T)[off], np.ones(n * (n - 1)))  # one of the two is first
        place = b.sum(axis=0)
        assert np.array_equal(np.sort(place), np.arange(n))  # transitive: each place once
        key = [(bool(np.isnan(v)), 0.0 if np.isnan(v) else v, i, k) for k, (v, i) in enumerate(zip(z, ids))]
        assert [int(v) for v in np.argsort(place)] == sorted(range(n), key=lambda k: key[k])
        w = np.zeros(n, dtype=np.float32)
        order.tower_keys32(n, _ptr(z), _ptr(w))
        assert not np.isnan(w).any()
        i, j = np.nonzero(b)
        assert np.all(w[i] <= w[j])
        # counting the smaller z alone is not enough where one of them is not a number
        if np.isnan(z).any():
            assert len(set((z[None, :] < z[:, None]).sum(axis=1))) < n


KERNELS = [ap.KERNEL_CLUSTER_MIXED, ap.KERNEL_CLUSTER_FP64, ap.KERNEL_CLUSTER_JROWS_MIXED]


# particles per tower (one tower column of 2 x 2 towers holds them): the one-workgroup build, registers, ranked parts
# of two and four wavefronts, LDS
@pytest.mark.gpu
@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("n,edge,height", [(300, 6.0, 12.0), (700, 6.0, 24.0), (5000, 20.0, 20.0), (6000, 9.0, 90.0),
                                           (6000, 6.0, 200.0), (9000, 6.0, 300.0), (12000, 6.0, 400.0)])
@pytest.mark.parametrize("bad", [1, 40])
def test_every_particle_is_kept(kernel, n, edge, height, bad):
    announce(f"cluster build, kernel {kernel}: {n} particles in {edge} x {edge} x {height}, {bad} without a z")
    rng = np.random.default_rng(n + bad)
    x, y, z = rng.uniform(0, edge, n), rng.uniform(0, edge, n), rng.uniform(0, height, n)
    lost = rng.choice(n, bad, replace=False)
    z[lost] = NAN
    z[rng.choice(np.setdiff1d(np.arange(n), lost), 20, replace=False)] = height / 3.0  # equal z
    ids = rng.integers(0, n // 3, n)  # ids that are not distinct
    with ap.Engine((0, 0, 0), (edge, edge, height), 2.5, 0.3, cluster_size=8) as e:
        e.upload(x, y, z, id=ids)
        for _ in range(3):  # the first build, and builds from the cluster layout
            e.rebuild(kernel)
            sp = np.asarray(e.clusters()["slot_particle"])
            assert np.array_equal(np.sort(sp[sp >= 0]), np.arange(n))
            f = e.download()
            for k, v in zip("xyz", (x, y, z)):
                assert np.array_equal(f[k], v, equal_nan=True), k


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [ap.KERNEL_LC_FP64, ap.KERNEL_VERLET_MIXED])
@pytest.mark.parametrize("n,L", [(800, 9.0), (5000, 20.0)])
def test_cells_keep_particles_of_equal_ids(kernel, n, L):
    announce(f"cell order, kernel {kernel}: {n} particles whose ids are not distinct")
    rng = np.random.default_rng(n)
    p = [rng.uniform(0, L, n) for _ in range(3)]
    with ap.Engine((0, 0, 0), (L, L, L), 2.5, 0.3) as e:
        e.upload(*p, id=rng.integers(0, 3, n))
        for _ in range(2):
            e.rebuild(kernel)
            f = e.download()
            for k, v in zip("xyz", p):
                assert np.array_equal(f[k], v), k


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 8])
@pytest.mark.parametrize("column", [127, 128, 129])
def test_small_build_where_it_leaves_the_sorts_to_others(oracle, M, column):
    announce(f"small build, M={M}: a column of {column} particles and more in its tower")
    rng = np.random.default_rng(M + column)
    box, n = (9.0, 9.0, 60.0), 700
    x, y, z = (rng.uniform(-0.5 * b, 1.5 * b, n) for b in box)
    z[1::3] = z[::3][:len(z[1::3])]
    x[:column], y[:column] = 0.1, 0.1
    x[column:] = 3.5 + 0.4 * (x[column:] % 9.0) / 9.0 * 10.0  # the others: not in that tower
    ids = rng.permutation(n).astype(np.int64)
    wx, wy, wz = oracle.wrap(x, y, z, (0, 0, 0), box)
    r = oracle.vcl_periodic(wx, wy, wz, ids, (0, 0, 0), box, 2.8, M)
    assert np.max(np.bincount(r["cluster_tower"])) * M >= column
    with ap.Engine((0.0, 0.0, 0.0), box, 2.5, 0.3, cluster_size=M) as e:
        e.upload(x, y, z, id=ids)
        for _ in range(2):
            e.build_pairs()
            g = e.clusters()
            for k in ("slot_particle", "cluster_tower", "list_offsets", "list_j", "list_shift", "bbox"):
                assert np.array_equal(g[k], r[k]), k
