"""GPU: the FP64 M2L kernels (vector units up to 13 terms, matrix cores above)
at the edges of their dispatch.

- every number of terms on a full level of 4,096 boxes, which up to 13 terms
  reads class-major packed sources, with the levels above it unpacked and
  their directions split over workgroups;
- a thin shell: missing children and neighbours, tiles that end within the
  parents of a level, steps without any source;
- lists of parents (adaptive tree, 4,096 parents and more) against the same
  solve on the uniform tree.

Bars: the oracle within 1e-11 (potential) and 1e-10 (field) as in
test_gpu_parity.py; list against uniform tree 1e-13: the same operators and
the same order of summation, but the leaf kernel is compiled differently, so
only rounding (2e-16 times the ~500 terms of a target's far field) may differ.
"""
import numpy as np
import pytest

from conftest import rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


def shell(n, seed):
    rng = np.random.default_rng(seed)
    d = rng.standard_normal((n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    return 0.5 + 0.45 * d, rng.uniform(-1.0, 1.0, n)


@pytest.mark.parametrize("kind,n,depth", [("cube", 60000, 5), ("shell", 9000, 5)])
@pytest.mark.parametrize("N", list(range(1, 19)))
def test_m2l_every_order(lfmm, orc, request, kind, n, depth, N):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = uniform_cube(n, 300 + N) if kind == "cube" else shell(n, 300 + N)
    pot, field, rep = lfmm.fmm3d(x, q, terms=N, tree_depth=depth, exclude_self=True)
    if kind == "cube":
        assert rep["num_leaves"] == 4096
    with orc.exact_geometry():
        op, of = orc.fmm3d(x, q, N, depth)
    op -= q * 1e4
    assert rel_l2(pot, op) <= 1e-11
    assert rel_l2(field, of) <= 1e-10


@pytest.mark.parametrize("N", [1, 9, 13, 14, 18])
def test_m2l_parent_lists(lfmm, request, N):
    print("\n[case] %s" % request.node.name, flush=True)
    x, q = uniform_cube(250000, 400 + N)
    pu, fu, ru = lfmm.fmm3d(x, q, terms=N, tree_depth=6, leaf_max=1, exclude_self=True)
    pa, fa, ra = lfmm.fmm3d(x, q, terms=N, tree_depth=6, leaf_max=1, adaptive=True, exclude_self=True)
    assert ra["num_leaves"] == ru["num_leaves"] and ra["xw_pairs"] == 0
    assert rel_l2(pa, pu) <= 1e-13 and rel_l2(fa, fu) <= 1e-13
