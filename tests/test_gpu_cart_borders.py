"""GPU: Cartesian walks at the edges of what their dispatch accepts -- borders staged in LDS or read from global
memory (more than 4096 words of them), uneven borders (the guessed bin of a start point is wrong), one bin per
axis -- bit for bit against the oracle in FP64, and mixed against FP64."""
import numpy as np
import pytest

from skirt7_amd import skirt as S
from skirt7_amd.capi import SG_FP64, SG_MIXED
from tests import oracle_lib as O
from tests.test_gpu_paths import assert_paths_equal

pytestmark = pytest.mark.gpu


def _borders(n, lo, hi, uneven):
    t = np.linspace(0.0, 1.0, n + 1)
    if uneven:
        t = np.expm1(6.0 * t) / np.expm1(6.0)
    v = lo + t * (hi - lo)
    v[-1] = hi
    return v


@pytest.mark.parametrize("shape,uneven", [((1, 1, 1), False), ((1, 7, 2), True), ((31, 32, 33), True),
                                          ((2037, 5, 3), False),    # 4096 words in FP64: the most that is staged
                                          ((2038, 5, 3), True),     # one border more; FP32 still staged
                                          ((4200, 2, 2), False)])   # neither staged
def test_paths_bit_for_bit(shape, uneven):
    ext = np.array([-3.0, -2.0, -1.0, 5.0, 4.0, 1.5])
    v = [_borders(n, ext[a], ext[a + 3], uneven) for a, n in enumerate(shape)]
    grid = S.CartesianDustGrid(ext, *v)
    scene = O.Scene().cartesian(ext, *v)
    rng = np.random.default_rng(7)
    n = 300
    k = rng.standard_normal((n, 3))
    k[:20] = np.eye(3)[rng.integers(0, 3, 20)] * rng.choice([-1.0, 1.0], 20)[:, None]   # along an axis
    k /= np.linalg.norm(k, axis=1)[:, None]
    r = ext[:3] + rng.random((n, 3)) * (ext[3:] - ext[:3])
    r[20:60, 0] = v[0][rng.integers(0, len(v[0]), 40)]                                  # on a border
    r[200:] -= 15.0 * k[200:]                                                            # from outside
    rays = np.concatenate([r, k], axis=1)
    assert_paths_equal(grid, scene, rays, 8192)
    # mixed: the same chord, to a rounding of the position (up to 5, 2^-21) per crossing (at most sum(shape) + 3)
    def chords(precision):
        c, _, d = grid.paths(rays, 8192, precision)
        return np.array([d[i, :c[i]].sum() for i in range(n)])   # entries past a ray's count are not written

    np.testing.assert_allclose(chords(SG_MIXED), chords(SG_FP64), rtol=0, atol=2.0**-21 * (sum(shape) + 3) * 4)
