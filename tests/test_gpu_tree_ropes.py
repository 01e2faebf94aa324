"""GPU: the exact tree walk over its ropes against the oracle's own searches, bit for bit, where the ropes do not
simply hit: uniform trees with rays through edges, corners and inside wall planes (points on walls, where the search
methods decide), deep trees (coarser and much finer neighbours), boxes far from the origin, and rays that run beside
planes which FP32 does not hold, so that a descent by the records' FP32 split planes comes to a wrong leaf. Edges and
walls at multiples of 2^-n are exact in FP64 and, for the boxes of the first test, in FP32."""
import numpy as np
import pytest

from skirt7_amd import skirt as S
from skirt7_amd.capi import SG_FP64, SG_NEIGHBOR, SG_TOPDOWN
from tests import oracle_lib as O
from tests.helpers import random_rays, random_tree_flags

pytestmark = pytest.mark.gpu

CUBE = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])


def edge_rays():
    rays = []
    for sx in (-1, 1):
        for sy in (-1, 1):
            for sz in (-1, 1):
                for k in ((sx, 0.0, 0.0), (0.6 * sx, 0.8 * sy, 0.0), (0.48 * sx, 0.64 * sy, 0.6 * sz),
                          (sx / 3 ** 0.5, sy / 3 ** 0.5, sz / 3 ** 0.5)):
                    for r in ((0.25, 0.25, 0.1), (0.25, 0.25, 0.25), (-0.5, 0.125, 0.375), (0.0, 0.0, 0.0), (-1.0, 0.5, 0.25)):
                        rays.append(list(r) + list(k))
    return np.array(rays)


def assert_walks_equal(g, sc, rays):
    counts, m, ds = g.paths(rays, 4096, SG_FP64)
    assert (counts >= 0).all()
    for i, rk in enumerate(rays):
        om, ods = sc.path(rk[:3], rk[3:])
        n = counts[i]
        assert n == len(om), (i, rk.tolist(), n, len(om))
        assert np.array_equal(m[i, :n], om) and np.array_equal(ds[i, :n], ods), (i, rk.tolist())


@pytest.mark.parametrize("arity,search", [(8, SG_TOPDOWN), (8, SG_NEIGHBOR), (2, SG_TOPDOWN), (2, SG_NEIGHBOR)])
@pytest.mark.parametrize("tree", ["root", "uniform", "deep"])
@pytest.mark.parametrize("shift,unit", [(0.0, 1.0), (1.0e3, 1.0), (-3.0, 2.0e18)])
def test_rope_walk_bitexact(arity, search, tree, shift, unit):
    if tree == "root":
        flags = np.zeros(1, np.uint8)
    elif tree == "uniform":
        flags = random_tree_flags(arity, 4 if arity == 8 else 9, 1.0, seed=1, minlevel=1)
    else:
        flags = random_tree_flags(arity, 8 if arity == 8 else 20, 0.2 if arity == 8 else 0.6, seed=5, minlevel=2 if arity == 8 else 6)
    ext = (CUBE + shift) * unit
    g = (S.OctTreeDustGrid if arity == 8 else S.BinTreeDustGrid)(ext, flags, search)
    sc = O.Scene().tree(arity, ext, flags, search)
    rays = np.concatenate([edge_rays(), random_rays(300, 9, CUBE)])
    rays[:, :3] = (rays[:, :3] + shift) * unit
    assert_walks_equal(g, sc, rays)


@pytest.mark.parametrize("arity,search", [(8, SG_TOPDOWN), (8, SG_NEIGHBOR), (2, SG_TOPDOWN), (2, SG_NEIGHBOR)])
def test_rope_walk_beside_inexact_planes(arity, search):
    """A box at 333 with walls at thirds: FP32 holds its planes to 1.5e-5. The rays start within 3e-5 of a plane and
    run along it, about an eighth of them between the plane and its place in FP32, so that a descent into finer cells
    takes the child on the plane's other side."""
    if arity == 8:
        flags = random_tree_flags(8, 7, 0.3, seed=5, minlevel=2)
    else:
        flags = random_tree_flags(2, 18, 0.6, seed=5, minlevel=6)
    ext = (CUBE + 1.0e3) / 3.0
    g = (S.OctTreeDustGrid if arity == 8 else S.BinTreeDustGrid)(ext, flags, search)
    sc = O.Scene().tree(arity, ext, flags, search)
    rng = np.random.default_rng(11)
    rays = []
    for _ in range(600):
        axis = rng.integers(3)
        level = rng.integers(1, 7)
        plane = ext[axis] + (ext[axis + 3] - ext[axis]) * rng.integers(1, 2**level) / 2.0**level
        r = ext[:3] + rng.random(3) * (ext[3:] - ext[:3])
        r[axis] = plane + rng.uniform(-3e-5, 3e-5)
        k = rng.standard_normal(3)
        k[axis] = rng.choice([0.0, 1e-7, -1e-7])
        rays.append(list(r) + list(k / np.linalg.norm(k)))
    rays = np.array(rays)
    wrong = np.abs(rays[:, :3] - rays[:, :3].astype(np.float32)).max()
    assert wrong > 1e-5   # FP32 does not hold positions here to the rays' distance from the planes
    assert_walks_equal(g, sc, rays)
