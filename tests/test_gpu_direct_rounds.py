"""GPU: direct sums whose targets go in several launches (whole rounds of
workgroups first, the rest in smaller ones): target counts that leave a rest of
one, of a round's half and of several smaller rounds, with enough sources that
the split is worth a launch; separate targets and, where the launch's first
target matters for j == i, one set without its own term.  Bar: the oracle within
1e-13 rel-L2 (sums of at most 20,000 terms of both signs in another order, each to
4e-16)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,ns", [(1025, 20000), (4097, 3000), (5633, 5000), (140001, 300)])
@pytest.mark.parametrize("dim", [3, 2])
def test_targets(lfmm, orc, request, dim, nt, ns):
    print("\n[case] %s" % request.node.name, flush=True)
    rng = np.random.default_rng(dim * 1000003 + nt)
    t, x, q = rng.random((nt, dim)), rng.random((ns, dim)), rng.uniform(-1.0, 1.0, ns)
    p, f = (lfmm.direct3d if dim == 3 else lfmm.direct2d)(x, q, targets=t)
    op, of = orc.direct3d(x, q, tgt_xyz=t) if dim == 3 else orc.direct2d(x, q, tgt_xy=t)
    assert rel_l2(p, op) <= 1e-13 and rel_l2(f, of) <= 1e-13


@pytest.mark.parametrize("n", [4097, 9729])
@pytest.mark.parametrize("dim", [3, 2])
def test_self(lfmm, orc, request, dim, n):
    print("\n[case] %s" % request.node.name, flush=True)
    rng = np.random.default_rng(dim * 1000003 + n)
    x, q = rng.random((n, dim)), rng.uniform(-1.0, 1.0, n)
    p, f = (lfmm.direct3d if dim == 3 else lfmm.direct2d)(x, q, exclude_self=True)
    idx = np.arange(n)
    op, of = (orc.direct3d if dim == 3 else orc.direct2d)(x, q, tgt_index=idx, include_self=False)
    assert rel_l2(p, op) <= 1e-13 and rel_l2(f, of) <= 1e-13
