"""GPU: clouds of small extent far from the origin, where a coordinate's own
square overflows but no distance within the cloud does.

3D: the self pair, clamped at 1e-4, is 10^4 q and everything else is below
1e-130 of it, so the potential is 10^4 q to a few ulp and the field next to
nothing.  2D: the oracle is the direct sum in long double, every pair near: 1e-8
(single terms are good to a few ulp).  With a far field the results are only
asked to be finite: a box's centre is rounded to the coordinates' grid, a 256th
of a leaf here, and so is its accuracy."""
import numpy as np
import pytest

from conftest import rel_l2

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


# widths: extents of 3e147 and 1e152, whose square is near overflow
@pytest.mark.parametrize("top,step,width", [(531, 480, 490), (545, 494, 505)])
@pytest.mark.parametrize("exclude", [False, True])
@pytest.mark.parametrize("n,depth", [(1, 1), (65, 1), (900, 5)])
def test_2d(lfmm, request, n, depth, exclude, top, step, width):
    print("\n[case] %s" % request.node.name, flush=True)
    x, k, q = cloud(2, n, 13 + n, top, step, width)
    _, first = np.unique(k, axis=0, return_index=True)  # coincident points aside
    x, k, q = x[np.sort(first)], k[np.sort(first)], q[np.sort(first)]
    pot, field, _ = lfmm.fmm2d(x, q, terms=25, tree_depth=depth, exclude_self=exclude)
    d = (k[:, None, :] - k[None, :, :]).astype(np.longdouble)
    r2 = (d ** 2).sum(axis=2)
    np.fill_diagonal(r2, 1)
    logs = np.longdouble(0.5) * np.log(r2) + step * np.log(np.longdouble(2))
    np.fill_diagonal(logs, 0 if exclude else np.log(np.longdouble(1e-4)))
    ref = logs @ q.astype(np.longdouble)
    fx, fy = (d[:, :, 0] / r2) @ q, -(d[:, :, 1] / r2) @ q  # in units of 2^-step
    assert np.isfinite(pot).all() and np.isfinite(field).all()
    if depth > 2:
        return
    assert np.abs(pot - ref).max() <= 1e-8 * max(np.abs(ref).max(), 1e-300)
    ref_field = np.stack([fx, fy], axis=1).astype(np.float64)
    assert rel_l2(field * 2.0 ** step, ref_field) <= 1e-8 if n > 1 else not field.any()
