"""GPU: clouds of small extent far from the origin, where a coordinate's own
square overflows but no distance within the cloud does.

3D: the self pair, clamped at 1e-4, is 10^4 q and everything else is below
1e-130 of it, so the potential is 10^4 q to a few ulp and the field next to
nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cloud(dim, n, seed, top, step, width):
    """n points in [2^top, 2^top + 2^width) on a grid of 2^step, exact; unevenly filled."""
    rng = np.random.default_rng(seed)
    k = np.floor(rng.random((n, dim)) ** 2 * 2.0 ** (width - step))
    return 2.0 ** top + k * 2.0 ** step, k, rng.uniform(-1, 1, n)


@pytest.mark.parametrize("n,depth", [(1, 1), (3, 1), (65, 1), (300, 2), (2000, 4)])
def test_3d(lfmm, request, n, depth):
    print("\n[case] %s" % request.node.name, flush=True)
    x, _, q = cloud(3, n, 11 + n, 514, 463, 478)
    pot, field, _ = lfmm.fmm3d(x, q, terms=6, tree_depth=depth)
    assert np.abs(pot - 1e4 * q).max() <= 1e-13 * np.abs(1e4 * q).max()
    assert np.abs(field).max() <= 1e-200


def test_3d_adaptive(lfmm):
    x, _, q = cloud(3, 3000, 12, 514, 463, 478)
    pot, field, _ = lfmm.fmm3d(x, q, terms=6, leaf_max=16, adaptive=True)
    assert np.abs(pot - 1e4 * q).max() <= 1e-13 * np.abs(1e4 * q).max()
    assert np.abs(field).max() <= 1e-200
