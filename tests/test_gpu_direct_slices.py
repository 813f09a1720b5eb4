"""GPU: the direct sums over their range of target counts.  The kernel cuts
the sources into 1024 / LT slices, LT from 1 (up to 1,023 targets) to 1024
(from 524,288 targets on); every LT is run with a last workgroup that is not
full, and with fewer sources than slices.  Bar: the oracle within 1e-13
rel-L2 (sums of at most 1,500 terms in another order, each term to 4e-16)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TARGETS = [1, 3, 1023, 1025, 2051, 4099, 8195, 16387, 32771, 65541, 131075, 262147, 524293]


@pytest.mark.parametrize("nt", TARGETS)
@pytest.mark.parametrize("dim", [3, 2])
def test_direct_slices(lfmm, orc, request, dim, nt):
    print("\n[case] %s" % request.node.name, flush=True)
    rng = np.random.default_rng(dim * 1000003 + nt)
    t = rng.random((nt, dim))
    for ns in (1, 7, 1500 if nt < 5000 else 300):
        x, q = rng.random((ns, dim)), rng.uniform(-1.0, 1.0, ns)
        p, f = (lfmm.direct3d if dim == 3 else lfmm.direct2d)(x, q, targets=t)
        op, of = orc.direct3d(x, q, tgt_xyz=t) if dim == 3 else orc.direct2d(x, q, tgt_xy=t)
        assert rel_l2(p, op) <= 1e-13 and rel_l2(f, of) <= 1e-13


@pytest.mark.parametrize("n", [600, 5000, 40000])
def test_direct_slices_self(lfmm, request, n):
    print("\n[case] %s" % request.node.name, flush=True)
    rng = np.random.default_rng(n)
    x, q = rng.random((n, 3)), rng.uniform(-1.0, 1.0, n)
    p, f = lfmm.direct3d(x, q, exclude_self=True)
    pick = rng.choice(n, 50, replace=False)
    d = x[pick, None, :] - x[None, :, :]
    r = np.maximum(np.sqrt((d ** 2).sum(-1)), 1e-4)
    w = q / r
    w[np.arange(50), pick] = 0.0
    assert rel_l2(p[pick], w.sum(1)) <= 1e-13
    assert rel_l2(f[pick], (d * (w / r ** 2)[:, :, None]).sum(1)) <= 1e-12
