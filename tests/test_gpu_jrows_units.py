"""The j-row kernel forms its pair constants in a length unit taken from the particle types: forces in other
length and energy units than sigma and epsilon, with types of very different sizes, in cubic boxes (the first
member's frame) and in others (exact separations), against the direct sum."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

# the FP32-pair kernels' bar on forces, energy and virial
TOL = 1e-5


@pytest.mark.parametrize("length,energy", [(1.0, 1.0), (3.4e-10, 1.65e-21), (250.0, 7.0e3)])
@pytest.mark.parametrize("ratio", [1.0, 0.3, 0.02])
@pytest.mark.parametrize("shape", [(1.0, 1.0, 1.0), (1.0, 1.07, 1.9)])
def test_jrows_units(oracle, length, energy, ratio, shape):
    announce(f"j-row kernel, unit {length} x {energy}, smallest/largest sigma {ratio}, box {shape}")
    rng = np.random.default_rng(7)
    dims = (np.array(shape) * 10).astype(int)
    box = dims * 1.12 * length
    idx = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing="ij")).reshape(3, -1)
    pos = (idx + 0.5 + rng.uniform(-0.06, 0.06, idx.shape)) * 1.12 * length
    n = idx.shape[1]
    types = 1 if ratio == 1.0 else 3
    sig = length * np.array([1.0, np.sqrt(ratio), ratio])[:types]
    eps = energy * np.array([1.0, 1.3, 0.7])[:types]
    t = rng.integers(0, types, n).astype(np.int32)
    rc, skin = 2.5 * length, 0.3 * length
    ref = oracle.direct_sum(*pos, rc, box_len=box, types=t, eps=eps, sig=sig)
    with ap.Engine((0, 0, 0), box, rc, skin, cluster_size=8) as e:
        e.set_types(eps, sig, np.ones(types))
        e.upload(*pos, type=t)
        g = e.force(ap.KERNEL_CLUSTER_JROWS_MIXED, globals=True)
        f = e.download()
        plain = e.force(ap.KERNEL_CLUSTER_JROWS_MIXED, globals=False)
        h = e.download()
    num = sum(np.sum((f[k] - ref[k]) ** 2) for k in ("fx", "fy", "fz"))
    den = sum(np.sum(ref[k] ** 2) for k in ("fx", "fy", "fz"))
    assert np.sqrt(num / den) <= TOL
    assert g.pair_count == ref["pairs"] == plain.pair_count
    assert abs(g.potential_energy / ref["epot"] - 1.0) <= TOL
    assert abs(g.virial / ref["virial"] - 1.0) <= TOL
    num = sum(np.sum((h[k] - ref[k]) ** 2) for k in ("fx", "fy", "fz"))
    assert np.sqrt(num / den) <= TOL
