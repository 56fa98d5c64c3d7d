"""The plain FP64 LinkedCells kernel where its staging and queues change shape: neighbourhoods of several stages
and cells of several tiles (a dense system), more hits than a queue holds, hardly any particles per cell,
boxes of one, two and three cells a side (a particle meets several images of another), and mixed types."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.3
# FP64 throughout: the bar of the FP64 kernels against the direct sum
TOL = 1e-10


@pytest.mark.parametrize("n,box,sigma,types", [
    (1, (2.9, 2.9, 2.9), 1.0, 1),          # one cell, a particle and its images
    (37, (2.81, 3.4, 5.7), 1.0, 2),        # 1 x 1 x 2 cells
    (300, (5.7, 8.5, 8.5), 1.0, 1),        # 2 x 3 x 3 cells
    (50, (33.0, 28.5, 40.0), 1.0, 1),      # mostly empty cells
    (1029, (11.3, 11.3, 11.3), 1.0, 2),
    (4096, (8.5, 8.5, 11.5), 0.55, 1),     # ~130 particles a cell, 4096 a neighbourhood, ~325 hits a particle
    (9000, (22.5, 14.1, 16.9), 0.7, 16),   # ~75 a cell, sixteen types
])
def test_lc_fp64_shapes(oracle, n, box, sigma, types):
    announce(f"LC FP64 kernel, n = {n}, box {box}, {types} types")
    rng = np.random.default_rng(n)
    a = (np.prod(box) / n) ** (1 / 3)
    dims = np.ceil(np.array(box) / a).astype(int)
    sites = rng.permutation(int(np.prod(dims)))[:n]
    idx = np.stack(np.unravel_index(sites, dims))
    pos = (idx + 0.5) * (np.array(box) / dims)[:, None] + rng.uniform(-0.03, 0.03, (3, n)) * a
    t = rng.integers(0, types, n).astype(np.int32)
    eps = np.linspace(0.8, 1.2, types) if types > 1 else np.ones(1)
    sig = sigma * (np.linspace(0.95, 1.05, types) if types > 1 else np.ones(1))
    ref = oracle.direct_sum(*pos, RC, box_len=box, types=t, eps=eps, sig=sig)
    with ap.Engine((0, 0, 0), box, RC, SKIN) as e:
        e.set_types(eps, sig, np.ones(types))
        e.upload(*pos, type=t)
        g = e.force(ap.KERNEL_LC_FP64, globals=True)
        f = e.download()
    num = sum(np.sum((f[k] - ref[k]) ** 2) for k in ("fx", "fy", "fz"))
    den = sum(np.sum(ref[k] ** 2) for k in ("fx", "fy", "fz"))
    assert g.pair_count == ref["pairs"]
    assert np.sqrt(num) <= TOL * max(np.sqrt(den), 1e-3)
    assert abs(g.potential_energy - ref["epot"]) <= TOL * max(abs(ref["epot"]), 1e-3)
    assert abs(g.virial - ref["virial"]) <= TOL * max(abs(ref["virial"]), 1e-3)
