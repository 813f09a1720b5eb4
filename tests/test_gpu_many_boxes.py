"""GPU: an adaptive solve whose uniform levels together hold more boxes than the
particles of the largest solve (2^28): an even background of 50M particles with
one clump so dense that the tree reaches level 14, so that from level 9 on nearly
every particle has a box of its own on every level.  Sampled against the direct
sum outside the clump (inside, the sum clamps pairs within 1e-4, which boxes of
3e-5 take as far ones); 6 terms on charges of one sign are good to 1e-3."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_background_and_clump(lfmm):
    n, clump = 50_000_000, 4096
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.rand(n, 3, dtype=torch.float64, device="cuda", generator=g)
    x[:clump] = 0.3 + 2e-4 * x[:clump]
    q = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    pot, _, rep = lfmm.fmm3d(x, q, terms=6, leaf_max=64, adaptive=True)
    assert rep["tree_depth"] >= 14
    pick = torch.tensor([0, 17, clump - 1, clump, n // 3, n - 1], device="cuda")
    ref, _ = lfmm.direct3d(x, q, targets=x[pick].contiguous())
    away = pick >= clump
    assert (pot[pick] - ref)[away].norm() <= 1e-3 * ref[away].norm()
