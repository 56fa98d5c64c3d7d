"""The j-row expansion's FP32 member test in boxes that are not cubic and near its frame's limit, and the register
tower sorts at the edges of their ranges, against the oracle's lists (exact)."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.3


def _box(dims, density, seed, jitter):
    n = int(np.prod(dims))
    a = density ** (-1.0 / 3.0)
    x, y, z, _, _, _, _ = ap.generate_lattice(seed, n, dims, a, (0.0, 0.0, 0.0), jitter, 0.9)
    return n, tuple(d * a for d in dims), x, y, z


# units of 1e-20 and 1e9: the test runs in units of rc + skin
@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("dims,density,unit", [((9, 12, 15), 0.75, 1.0), ((6, 7, 6), 0.75, 1.0), ((5, 5, 30), 0.6, 1.0),
                                               ((20, 7, 7), 0.02, 1.0), ((9, 9, 14), 0.75, 1e-20),
                                               ((9, 9, 9), 0.75, 1e9)])
def test_jrows_exact_in_any_box(oracle, M, dims, density, unit):
    # (20, 7, 7) at density 0.02: clusters longer than 1.5 (rc + skin) take the exact test
    _check_jrows(oracle, M, dims, density, unit, 0.2)


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("dims,jitter", [((9, 9, 9), 0.0), ((9, 10, 12), 0.0), ((9, 9, 9), 1e-5), ((12, 9, 9), 1e-6)])
def test_jrows_exact_at_the_edge(oracle, M, dims, jitter):
    # a lattice of spacing (rc + skin) / 3: six neighbours of every particle are at rc + skin, or next to it
    _check_jrows(oracle, M, dims, (3.0 / (RC + SKIN)) ** 3, 1.0, jitter)


def _check_jrows(oracle, M, dims, density, unit, jitter):
    announce(f"j-rows exact M={M}: lattice {dims} density {density} unit {unit} jitter {jitter}")
    n, box, x, y, z = _box(dims, density, 3, jitter)
    box, x, y, z = tuple(b * unit for b in box), x * unit, y * unit, z * unit
    rc, skin = RC * unit, SKIN * unit
    with ap.Engine((0.0, 0.0, 0.0), box, rc, skin, cluster_size=M) as e:
        e.set_types([1.0], [unit], [1.0])
        e.upload(x, y, z, id=np.arange(n, dtype=np.int64))
        e.force(ap.KERNEL_CLUSTER_JROWS_MIXED, globals=False)
        g = e.clusters()
    wx, wy, wz = oracle.wrap(x, y, z, (0, 0, 0), box)
    roff, rnb = oracle.verlet_pairs_fixed(wx, wy, wz, (0, 0, 0), box, rc + skin)
    sp, off, lj = g["slot_particle"], g["list_offsets"], g["list_j"]
    for ci in range(len(off) - 1):
        members = [int(p) for p in sp[ci * M:(ci + 1) * M] if p >= 0]
        expect = set(members)
        for p in members:
            expect.update(int(q) for q in rnb[roff[p]:roff[p + 1]])
        row = lj[off[ci]:off[ci + 1]].tolist()
        assert len(row) == len(set(row)) and set(row) == expect, ci


@pytest.mark.parametrize("longest", [64, 65, 256, 257, 512, 513, 770, 1023, 1024, 1025])
def test_tower_sorts_at_their_edges(oracle, longest):
    # two towers (6 wide each) of `longest` and about a third as many particles; z distinct, some equal in FP32
    announce(f"tower sorts: longest tower {longest}, M=8")
    rng = np.random.default_rng(longest)
    counts = (longest, longest // 3 + 1)
    n = sum(counts)
    box = (12.0, 6.0, n / 1.5)
    x = np.concatenate([rng.uniform(0.1, 5.9, counts[0]), rng.uniform(6.1, 11.9, counts[1])])
    y = rng.uniform(0.0, 6.0, n)
    z = rng.uniform(1.0, box[2] - 1.0, n)
    z[1::2] = z[::2][:len(z[1::2])] * (1.0 + 2.0 ** -45)
    perm = rng.permutation(n)
    x, y, z, ids = x[perm], y[perm], z[perm], rng.permutation(n).astype(np.int64)
    with ap.Engine((0.0, 0.0, 0.0), box, RC, SKIN, cluster_size=8) as e:
        e.upload(x, y, z, id=ids)
        e.build_pairs()
        g = e.clusters()
    assert list(g["towers_per_dim"]) == [2, 1]
    wx, wy, wz = oracle.wrap(x, y, z, (0, 0, 0), box)
    r = oracle.vcl_periodic(wx, wy, wz, ids, (0, 0, 0), box, RC + SKIN, 8)
    for k in ("slot_particle", "cluster_tower", "bbox"):
        assert np.array_equal(g[k], r[k]), k


@pytest.mark.parametrize("M", [1, 4, 8])
@pytest.mark.parametrize("n,box,column", [(5, (6.0, 6.0, 6.0), 0), (700, (10.0, 10.0, 10.0), 0), (1024, (40.0, 40.0, 4.0), 0),
                                          (1025, (40.0, 40.0, 4.0), 0), (2000, (9.0, 9.0, 60.0), 256),
                                          (2000, (9.0, 9.0, 60.0), 257), (4096, (17.0, 17.0, 18.0), 0),
                                          (4097, (17.0, 17.0, 18.0), 0), (4096, (200.0, 200.0, 3.0), 0)])
def test_small_builds(oracle, M, n, box, column):
    # sizes around the limits of the one-workgroup passes: 4096 slots, 1024 towers, towers of 256; ties in z;
    # positions outside the box (wrapped); then a second build from the padded cluster layout
    announce(f"small build n={n} M={M} box {box} column {column}")
    rng = np.random.default_rng(n + M + column)
    x, y, z = (rng.uniform(-0.5 * b, 1.5 * b, n) for b in box)
    z[1::3] = z[::3][:len(z[1::3])]
    if column:
        x[:column], y[:column] = 0.1, 0.1
    ids = rng.permutation(n).astype(np.int64)
    wx, wy, wz = oracle.wrap(x, y, z, (0, 0, 0), box)
    r = oracle.vcl_periodic(wx, wy, wz, ids, (0, 0, 0), box, RC + SKIN, M)
    with ap.Engine((0.0, 0.0, 0.0), box, RC, SKIN, cluster_size=M) as e:
        e.upload(x, y, z, id=ids)
        for _ in range(2):
            e.build_pairs()
            g = e.clusters()
            for k in ("slot_particle", "cluster_tower", "list_offsets", "list_j", "list_shift", "bbox"):
                assert np.array_equal(g[k], r[k]), k
