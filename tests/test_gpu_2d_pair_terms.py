"""GPU: single pair terms of the 2D leaf kernel.

Two particles, self excluded, one level: the potential is q log r and the force
q conj(dz) / r^2 of one pair, as accurate as the library's logarithm and a
correctly rounded quotient give them.

Potential, distances with an exactly representable square: the logarithm is good
to about half an ulp of its value at any distance, next to 1 included, and the
product with q rounds twice (fma, sum): 4 ulp = 8.9e-16 leaves room for that.
Force: q / r^2 correctly rounded, then the same products as direct2d: equal
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NEAR_ONE = [1.0] + [1 + s * 2.0 ** -k for k in (4, 7, 8, 9, 10, 17, 20, 23) for s in (-1, 1)]
OTHER = [2.0 ** -13, 0.0625, 0.25, 0.5, 0.625, 0.7, 0.71, 0.75, 0.84375, 0.845, 1.1875, 1.19, 1.375, 1.5, 2.0, 3.0, 1024.0,
         2.0 ** 120]


def pair(lfmm, d, q):
    x = np.array([[0.0, 0.0], [d, 0.0]])
    pot, field, _ = lfmm.fmm2d(x, np.array(q), terms=4, tree_depth=1, exclude_self=True)
    return np.longdouble(d), pot, field


@pytest.mark.parametrize("d", [float(np.float32(v)) for v in NEAR_ONE + OTHER])  # 24 bits: exact squares
def test_potential_of_one_pair(lfmm, request, d):
    print("\n[case] %s" % request.node.name, flush=True)
    r, pot, _ = pair(lfmm, d, [0.75, -1.25])
    ref = np.array([-1.25, 0.75], dtype=np.longdouble) * np.log(r)
    assert np.abs(pot - ref).max() <= 8.9e-16 * np.abs(ref).max()


def test_force_equals_direct(lfmm):
    rng = np.random.default_rng(77)
    for _ in range(64):
        x = rng.random((2, 2)) * 10.0 ** rng.uniform(-3, 6)
        q = rng.uniform(-1, 1, 2)
        _, field, _ = lfmm.fmm2d(x, q, terms=4, tree_depth=1, exclude_self=True)
        _, direct = lfmm.direct2d(x, q, exclude_self=True)
        assert np.array_equal(field, direct)


@pytest.mark.parametrize("q", [np.inf, -np.inf, 0.0])
def test_charges_without_a_residual(lfmm, request, q):
    """q / r^2 and q log r of an infinite or zero charge."""
    print("\n[case] %s" % request.node.name, flush=True)
    x = np.array([[0.0, 0.0], [0.5, 0.25]])
    pot, field, _ = lfmm.fmm2d(x, np.array([1.0, q]), terms=4, tree_depth=1, exclude_self=True)
    direct_pot, direct = lfmm.direct2d(x, np.array([1.0, q]), exclude_self=True)
    assert np.array_equal(field, direct) and pot[0] == direct_pot[0]
