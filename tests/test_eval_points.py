"""Points that are no numbers, infinite or outside the world give 0, whatever the world's shape, and leave
the other points' values alone."""
import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boxes", [(2, 2, 2), (4, 2, 1), (3, 3, 3), (1, 2, 3)])
def test_points_outside(boxes):
    from mrchem_amd import mrcpp as G
    world = G.BoundingBox(-3, tuple(-(b // 2) for b in boxes), boxes)
    mra = G.MultiResolutionAnalysis(world, G.LegendreBasis(4), 10)
    t = G.project(1e-3, G.FunctionTree(mra), configs.density3(1)[0])
    pts = np.random.default_rng(0).uniform(0.1, 3.0, (8, 3))
    good = t.evalf(pts)
    assert np.isfinite(good).all() and np.abs(good).max() > 0.0
    bad = []
    for v in (np.nan, np.inf, -np.inf, 1e300, -1e300, 100.0):
        for dims in ((0,), (1,), (2,), (0, 1), (0, 1, 2)):
            p = pts[0].copy()
            p[list(dims)] = v
            bad.append(p)
    both = np.concatenate([pts, np.array(bad)])
    out = t.evalf(both)
    assert np.array_equal(out[:8], good)
    assert np.array_equal(out[8:], np.zeros(len(bad)))
