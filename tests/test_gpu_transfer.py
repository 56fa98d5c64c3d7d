"""Uploads through the staging buffer and downloads through the ring: sizes around their limits, exact values."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

KEYS = ("x", "y", "z", "vx", "vy", "vz", "fx", "fy", "fz")


def _arrays(n, seed, L):
    rng = np.random.default_rng(seed)
    return [rng.uniform(0.0, L, n) for _ in range(3)] + [rng.standard_normal(n) for _ in range(6)]


# one chunk; chunks of 256 KiB; an upload's 4 MiB; the ring wraps above 16 MiB; helpers from 24 MiB
@pytest.mark.parametrize("n", [1, 2, 3640, 3641, 3643, 29129, 87381, 87382, 116508, 116509, 233017, 349525, 349526, 500001])
def test_round_trip(n):
    announce(f"upload and download of {n} particles")
    with ap.Engine((0, 0, 0), (50.0,) * 3, 2.5, 0.3, cluster_size=8) as e:
        e.set_types([1.0, 1.0], [1.0, 1.0], [1.0, 1.0])
        for seed in range(3):  # another upload follows at once: the staging buffer is still being read
            a = _arrays(n, seed, 50.0)
            rng = np.random.default_rng(100 + seed)
            e.upload(*a[:6], type=rng.integers(0, 2, n).astype(np.int32), id=rng.permutation(n).astype(np.int64))
        e.set_forces(*a[6:])
        for _ in range(2):
            f = e.download()
            for k, v in zip(KEYS, a):
                assert np.array_equal(f[k], v), k
        first, count = n // 3, n - n // 3 - n // 5
        f = e.download_range(first, count)
        for k, v in zip(KEYS, a):
            assert np.array_equal(f[k], v[first:first + count]), k
        b = _arrays(n, 9, 50.0)
        assert e.update_positions(*b[:6])
        f = e.download()
        for k, v in zip(KEYS, b[:6] + a[6:]):
            assert np.array_equal(f[k], v), k


@pytest.mark.parametrize("n", [1000, 200000])
@pytest.mark.parametrize("bad", [-2.9, 12.9, float("nan")])
def test_open_region_is_checked_before_anything_changes(n, bad):
    announce(f"open box, {n} particles, one at {bad}")
    a = _arrays(n, 1, 10.0)
    with ap.Engine((0, 0, 0), (10.0,) * 3, 2.5, 0.3, cluster_size=8) as e:
        e.set_open_box((0, 0, 0), (10.0,) * 3)
        e.upload(*a[:6])
        for at in (0, n // 2, n - 1):
            w = a[1].copy()
            w[at] = bad
            with pytest.raises(ap.EngineError):
                e.upload(a[0], w, a[2])
            with pytest.raises(ap.EngineError):
                e.update_positions(a[0], w, a[2])
        f = e.download()
        for k, v in zip(KEYS, a[:6]):
            assert np.array_equal(f[k], v), k


@pytest.mark.parametrize("n", [3000, 40000, 87381, 87382])
def test_uploads_after_a_download(n):
    # the download made the staging buffer large enough for these uploads; the second is queued behind the first
    announce(f"uploads of {n} particles through the staging buffer")
    with ap.Engine((0, 0, 0), (50.0,) * 3, 2.5, 0.3, cluster_size=8) as e:
        e.upload(*_arrays(n, 0, 50.0)[:6])
        e.download()
        for seed in range(1, 6):
            a = _arrays(n, seed, 50.0)
            e.upload(*(a[:6] if seed % 2 else a[:3]))
            if seed % 3 == 0:
                continue
            f = e.download()
            for k, v in zip(KEYS, a[:6] if seed % 2 else a[:3] + [np.zeros(n)] * 3):
                assert np.array_equal(f[k], v), k
