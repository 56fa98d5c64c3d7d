"""What a context pins for its transfers: no more than it needs, since the call that pins pays for it."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
KIB = 1024


@pytest.fixture(scope="module")
def sizes(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stage") / "stage_sizes.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-shared", "-fPIC",
                    os.path.join(HERE, "cpp", "stage_sizes.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    for f in (lib.stage_capacity, lib.download_chunk, lib.ring_bytes):
        f.restype = ctypes.c_size_t
        f.argtypes = [ctypes.c_size_t] * (2 if f is lib.stage_capacity else 1 if f is lib.download_chunk else 0)
    return lib


# 72 bytes per downloaded particle; 30,011 of them need 2.06 MiB
@pytest.mark.parametrize("n", [1, 700, 5000, 9100, 30011, 58254, 116508, 300000, 10**6])
def test_first_buffer_is_the_next_64_kib(sizes, n):
    ring = sizes.ring_bytes()
    wanted = min(72 * n, ring)
    cap = sizes.stage_capacity(wanted, 0)
    assert wanted <= cap <= min(wanted + 64 * KIB, ring)


def test_growth_pins_a_few_times_only(sizes):
    ring, had, pinned = sizes.ring_bytes(), 0, 0
    for wanted in range(64 * KIB, ring + 1, 8 * KIB):
        if had < wanted:
            had, pinned = sizes.stage_capacity(wanted, had), pinned + 1
            assert wanted <= had <= ring
    assert pinned <= 14


@pytest.mark.parametrize("n", [1, 3640, 3641, 29127, 29128, 29129, 116507, 116508, 116509, 10**6, 10**8])
def test_chunks_fit_the_ring(sizes, n):
    total = 9 * n
    chunk = sizes.download_chunk(total)
    chunks = -(-total // chunk)
    need = 8 * (chunks * chunk if chunks > 1 else total)
    cap = sizes.stage_capacity(min(need, sizes.ring_bytes()), 0)
    slots = cap // (8 * chunk)
    assert chunks == 1 or slots >= min(chunks, 8)
