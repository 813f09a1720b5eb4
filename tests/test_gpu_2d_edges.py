"""GPU: the 2D operators at the edges of their launches, against the oracle.

Expansion sizes at which the M2L changes its row blocks (12, 25), pads a row (odd
sizes) or takes a second coefficient register (17), on clustered particles with
missing children; the pair sums alone (one level: every pair is near) at sizes
around a wave and a workgroup, with coincident points, and with distances whose
square is near overflow.  Bars: 1e-11 as for the other 2D parity tests
(normalised against unnormalised series); pairs 1e-13 (a term is good to a few
ulp, sums of at most 1,025 terms of both signs lose two digits)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0.2, 0.8, (4, 2))
    return c[rng.integers(0, 4, n)] + 0.05 * rng.standard_normal((n, 2)), rng.uniform(-1, 1, n)


@pytest.mark.parametrize("N", [2, 3, 11, 13, 15, 16, 17, 24, 25, 29])
def test_expansion_sizes(lfmm, orc, request, N):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = cloud(3001, 900 + N)
    pot, field, _ = lfmm.fmm2d(x, q, terms=N, tree_depth=6)
    op, of = orc.fmm2d(x, q, N, 6)
    assert rel_l2(pot, op) <= 1e-11 and rel_l2(field, of) <= 1e-11


@pytest.mark.parametrize("scale", [1.0, 1e-3, 1e152])
@pytest.mark.parametrize("n", [2, 63, 65, 257, 1025])
def test_pairs(lfmm, orc, request, n, scale):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = cloud(n, 950 + n)
    x[n // 2] = x[0]
    x *= scale
    pot, field, _ = lfmm.fmm2d(x, q, terms=4, tree_depth=1)
    dp, df = orc.direct2d(x, q, tgt_index=np.arange(n), include_self=True)
    assert rel_l2(pot, dp) <= 1e-13
    assert np.abs(field - df).max() <= 1e-13 * np.abs(df).max()
