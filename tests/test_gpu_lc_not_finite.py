"""The FP64 LinkedCells kernel with a particle whose position is not finite: its force, the virial, and the forces of
the particles that meet it are not numbers; all others are those without it."""
import numpy as np
import pytest

import autopas_amd as ap
from conftest import announce

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.3
NAN, INF = float("nan"), float("inf")


def _meets(cells, nh, at):
    """Particles whose 27 cells (periodic, of the box's own cells) hold the cell of particle `at`."""
    no = np.asarray(nh) - 2
    c = np.stack([cells % nh[0] - 1, cells // nh[0] % nh[1] - 1, cells // (nh[0] * nh[1]) - 1])
    near = np.ones(len(cells), dtype=bool)
    for d in range(3):
        if not 0 <= c[d, at] < no[d]:  # a halo cell is no one's neighbour
            return np.zeros(len(cells), dtype=bool)
        k = (c[d] - c[d, at]) % no[d]
        near &= (k <= 1) | (k == no[d] - 1)
    return near


@pytest.mark.parametrize("n,L", [(700, 10.2), (2500, 15.0), (150, 20.0)])
@pytest.mark.parametrize("types", [1, 3])
@pytest.mark.parametrize("bad", [(NAN, 0, 0), (0, NAN, 0), (NAN, NAN, NAN), (0, 0, INF), (-INF, 0, NAN)])
def test_not_finite_is_not_hidden(n, L, types, bad):
    announce(f"LC FP64 kernel, {n} particles, {types} types, one displaced by {bad}")
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    idx = np.stack(np.unravel_index(rng.permutation(side ** 3)[:n], (side,) * 3))
    pos = (idx + 0.5) * (L / side) + rng.uniform(-0.05, 0.05, (3, n))
    t = rng.integers(0, types, n).astype(np.int32)
    at = n // 3
    one = np.arange(n) != at
    args = dict(cutoff=RC, skin=SKIN)
    with ap.Engine((0, 0, 0), (L,) * 3, **args) as e:
        e.set_types([1.0, 0.9, 1.1][:types], [1.0, 0.95, 1.05][:types], [1.0] * types)
        e.upload(*pos[:, one], type=t[one])
        g0 = e.force(ap.KERNEL_LC_FP64, globals=True)
        f0 = e.download()
        moved = pos.copy()
        moved[:, at] += bad
        e.upload(*moved, type=t)
        g = e.force(ap.KERNEL_LC_FP64, globals=True)
        f = e.download()
        cells, nh = e.cells()
    meets = _meets(cells, nh, at)
    scale = max(np.max(np.abs(f0[k])) for k in ("fx", "fy", "fz"))
    for d, k in enumerate(("fx", "fy", "fz")):
        expect = np.zeros(n, dtype=bool)
        if not np.isfinite(bad[d]):
            expect |= meets
            expect[at] = True
        assert np.array_equal(np.isnan(f[k][one]), expect[one]), k
        assert np.isnan(f[k][at]) == expect[at], k
        ok = ~expect[one]
        assert np.max(np.abs(f[k][one] - f0[k])[ok], initial=0.0) <= 1e-11 * scale, k
    assert np.isnan(g.virial) and not np.isnan(g0.virial)
    assert g.pair_count == g0.pair_count
    assert abs(g.potential_energy - g0.potential_energy) <= 1e-11 * abs(g0.potential_energy)
