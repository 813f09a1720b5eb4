"""GPU: the tree build at the edges of its tiles, exactly against numpy.

Level arrays, maps and depths are whole numbers: they must be equal.  Sizes lie
around 64, 1,024 and 4,096 (a wave, a tile of the levels, a tile of the scans
and the sort); inputs are spread evenly, piled on one point (one leaf over many
tiles), clustered so that the depth comes from sorted keys, and planar."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def points(kind, n, dim):
    rng = np.random.default_rng(n * 10 + dim)
    x = rng.random((n, dim))
    if kind == "pile":
        x[n // 3:] = x[0]
    elif kind == "cluster":
        x = x * 2.0 ** -rng.integers(0, 12, (n, 1))
    return x


def keys_of(x, geom, level):
    dim = x.shape[1]
    shift, scale = geom
    cell = (float(1 << level) * ((x - shift) / scale)).astype(np.uint64)
    key = np.zeros(len(x), np.uint64)
    for b in range(level):
        for a in range(dim):
            key |= ((cell[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(dim * b + dim - 1 - a)
    return key


def want_depth(x, geom, leaf_max, deepest):
    for level in range(deepest + 1):
        if np.unique(keys_of(x, geom, level), return_counts=True)[1].max() <= leaf_max:
            return level + 1
    return deepest + 1


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["even", "cluster", "pile"])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 1023, 1024, 1025, 4096, 4097, 20011])
def test_tree_levels_equal_numpy(lfmm, request, n, kind, dim):
    print("\n[case] %s" % request.node.name, flush=True)
    x = points(kind, n, dim)
    tree = lfmm.tree3d if dim == 3 else lfmm.tree2d
    for leaf_max in ([0] if kind == "pile" else [7, 40]):
        depth = 4 if kind == "pile" else lfmm.FMM_AUTO
        t = tree(x, None, depth, leaf_max=leaf_max)
        geom = (t["shift"], t["scale"])
        if leaf_max:
            assert t["depth"] == want_depth(x, geom, leaf_max, 15 if dim == 3 else 30)
        leaf = t["depth"] - 1
        key = keys_of(x, geom, leaf)
        order = np.argsort(key, kind="stable")
        pos = np.empty(n, np.int64)
        pos[order] = np.arange(n)
        assert np.array_equal(t["pos_map"], pos)
        below = key[order]
        for level in range(leaf, -1, -1):
            k, begin = np.unique(below, return_index=True)
            assert np.array_equal(t["keys"][level], k)
            assert np.array_equal(t["begin"][level], np.append(begin, len(below)))
            below = k >> np.uint64(dim)


def test_scan_of_many_tiles(lfmm):
    """More than 4,096 tiles of 4,096: the scan takes its third launch."""
    n = 4096 * 4096 + 5001
    rng = np.random.default_rng(5)
    x = rng.random((n, 3))
    t = lfmm.tree3d_adaptive(x, leaf_max=2048)
    b = t["box_range"][t["leaf_box"]]
    assert b[0, 0] == 0 and b[-1, 1] == n and np.array_equal(b[1:, 0], b[:-1, 1])
    assert int((b[:, 1] - b[:, 0]).max()) <= 2048
