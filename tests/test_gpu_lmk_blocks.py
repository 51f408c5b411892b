"""The landmark fit with slack where its unknowns (k_exp + 7) meet the edges of the 16 x 16 blocks of its
Hessian and the ends of the range: terms to 1e-11 of their largest entry (both sides FP64, sums of at
most 102 products in another order), and whole fits with the same decisions (the bounds of the fits at
other sizes: 1e-6 of the unknowns, which the device returns in FP32)."""
import pytest

from scenes import make_scene
from test_gpu_lmkfit import _check_fit, _check_terms, _start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Kl", [1, 8, 9, 25, 26, 57, 58, 89])
def test_block_edges(Kl):
    sc = make_scene(grid=40, k_exp=89, crops=(96, 200, 300), pose_deg=15.0)
    _check_terms(sc, Kl, 100.0, 31)
    _check_fit(sc, Kl, _start(sc, 32, exp=0.1))
