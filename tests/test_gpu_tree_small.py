"""GPU: the adaptive octree's arrays for sets so small that it has one level (a
single leaf) or two, where no box has an X list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf_max,depth", [(1, 64, 1), (10, 64, 1), (64, 64, 1), (65, 64, 2), (400, 100, 2)])
def test_one_and_two_levels(lfmm, request, n, leaf_max, depth):
    print("\n[case] %s" % request.node.name, flush=True)
    x = np.random.default_rng(n).random((n, 3))
    t = lfmm.tree3d_adaptive(x, leaf_max=leaf_max)
    assert t["depth"] == depth
    boxes, leaves = len(t["box_key"]), len(t["leaf_box"])
    assert boxes == (1 if depth == 1 else 1 + leaves)
    assert np.array_equal(t["box_range"][0], [0, n])
    # every leaf touches every other
    assert np.array_equal(t["u_off"], leaves * np.arange(leaves + 1))
    assert not t["x_off"].any() and len(t["x_off"]) == boxes + 1 and not t["w_off"].any()
    assert len(t["x_leaf"]) == 0 and len(t["w_box"]) == 0
