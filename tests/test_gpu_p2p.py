"""GPU: the near field alone, over the ranges its launch distinguishes.

With one or two tree levels every pair is a near pair, so the solve equals the
FP64 direct sum: two or four targets per lane, one to 64 parts per source
list, ragged leaf ends, separate targets.  Bar 1e-13 rel-L2: the pair kernel's
reciprocal root is good to 4.3e-15 per term.  The orders of the leaves (by
source count, in blocks of 32, 256 or 512) meet the oracle in the parity tests
at 512 and 4,096 leaves and the adaptive tests."""
import pytest

from conftest import rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [1, 2])
@pytest.mark.parametrize("n", [1, 2, 5, 63, 129, 511, 1025, 9001, 40003])
def test_pairs_equal_direct_sum(lfmm, request, n, depth):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = uniform_cube(n, 500 + n)
    p, f, _ = lfmm.fmm3d(x, q, terms=3, tree_depth=depth)
    dp, df = lfmm.direct3d(x, q)
    assert rel_l2(p, dp) <= 1e-13
    if n > 1:
        assert rel_l2(f, df) <= 1e-13


@pytest.mark.parametrize("n,m", [(1, 1), (300, 70), (70, 3001), (9001, 20011)])
def test_pairs_with_targets(lfmm, request, n, m):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = uniform_cube(n, 600 + n)
    t, _ = uniform_cube(m, 700 + m)
    p, f, _ = lfmm.fmm3d(x, q, terms=3, tree_depth=2, targets=t)
    dp, df = lfmm.direct3d(x, q, targets=t)
    assert rel_l2(p, dp) <= 1e-13 and rel_l2(f, df) <= 1e-13
