"""J^T J of one frame whose Jacobian rows pass 2^31 bytes, in a crop of which every row would end below 2^32
(32-bit offsets) and in one beyond it (64-bit ones): the tile kernel against the FP32 kernel, which
addresses every row with 64 bits.  The face fills the crop."""
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


@pytest.mark.parametrize("side", [3300, 3440])
def test_tile_kernel_on_large_crops(side):
    sc = make_scene(grid=100, k_exp=79, fit_light=2, crops=(64,), noise=0.0, pose_deg=5.0)
    fr, theta = sc.frames[0], sc.init().astype(np.float32)
    zoom = 3.0 * side / 64                              # the small crop's view, magnified about its centre
    for f in ("phix", "phiy", "face_size"):
        setattr(fr, f, getattr(fr, f) * zoom)
    fr.cx, fr.cy = side / 2, side / 2
    fr.lmk_x = ((fr.lmk_x - 32) * zoom + side / 2).astype(np.float32)
    fr.lmk_y = ((fr.lmk_y - 32) * zoom + side / 2).astype(np.float32)
    fr.x0 = fr.y0 = 0
    fr.width = fr.height = side
    fr.obs = np.random.default_rng(1).random(side * side, dtype=np.float32)
    ctx = tdi.Context(sc.model, sc.opts)
    b = tdi.Batch(ctx, [fr])
    npix = int(b.render(theta)[2][0])
    assert npix * 96 * 4 > 2 ** 31
    H, g, _ = (t.double() for t in b.normal_equations(theta, mixed=True))
    Hp, gp, _ = (t.double() for t in b.normal_equations(theta, mixed=False))
    b.close()
    ctx.close()
    # BF16 parts and FP32 sums of 10^7 pixels against FP32 products and sums; a wrong row is an error of order 1
    assert float((H - Hp).norm() / Hp.norm()) < 1e-4 and float((g - gp).norm() / gp.norm()) < 1e-4
