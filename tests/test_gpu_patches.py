"""The per-pixel Jacobian through mesh patches against the same frames through gathers.  Batches of seven
frames take the gathers, the whole list the patches (64 frames, or frames times patches of 2048, with 2^18
crop pixels; 128 or 8192 below 40 columns).  Both round every entry alike, so with more than 111 unknowns,
whose J^T J is summed in FP64 in an order of the crop sizes alone, the normal equations are the same bits;
with fewer, the FP32 sums of J^T J are split by the number of frames (1e-5 of the norm)."""
import dataclasses
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


def _normal(sc, frames, theta, mixed):
    ctx = tdi.Context(sc.model, sc.opts)
    b = tdi.Batch(ctx, frames)
    out = [t.clone() for t in b.normal_equations(torch.from_numpy(theta).cuda(), mixed=mixed)]
    torch.cuda.synchronize()
    b.close()
    ctx.close()
    return out


@pytest.mark.parametrize("grid,k_id,k_exp,k_tex,crops,n,mixed", [
    (48, 83, 81, 7, (96, 64, 71, 50, 80, 64, 0), 70, False),    # chunks of 80 + 3 and 80 + 1 columns from 7 and 90, albedo
    (48, 3, 17, 0, (48, 40, 60, 56, 33, 60, 52), 133, True),    # columns from 0 and 3
    (40, 0, 79, 0, (40, 30, 48, 40, 48, 0, 48), 301, True),     # several slices and parts
    (170, 0, 100, 0, (256,), 8, False)])                        # several segments of a frame's positions
def test_patches_give_the_gathers_entries(grid, k_id, k_exp, k_tex, crops, n, mixed):
    sc = make_scene(grid=grid, k_exp=k_exp, k_id=k_id, k_tex=k_tex, fit_id=k_id > 0, fit_tex=k_tex > 0, fit_light=2,
                    crops=tuple(c or 48 for c in crops), noise=0.0, pose_deg=10.0, seed=grid)
    for c, fr in zip(crops, sc.frames):
        if c == 0:
            fr.x0 = 20 * fr.width                               # nothing of the face in the crop
    rng = np.random.default_rng(3)
    m = len(crops)
    theta = np.stack([sc.truths[i % m].theta for i in range(n)])
    theta[:, :sc.lay["pose"]] += rng.uniform(-0.2, 0.2, (n, sc.lay["pose"]))
    theta[:, sc.lay["pose"] + 3:sc.lay["pose"] + 6] += rng.uniform(-0.1, 0.1, (n, 3))
    theta = theta.astype(np.float32)
    frames = [sc.frames[i % m] for i in range(n)]
    H, g, _ = _normal(sc, frames, theta, mixed)
    assert float(H.abs().amax()) > 0
    for i in range(0, n, 7):
        h, q, _ = _normal(sc, frames[i:i + 7], theta[i:i + 7], mixed)
        for a, b in ((H[i:i + 7], h), (g[i:i + 7], q)):
            if sc.K > 111:
                assert torch.equal(a, b), i
            else:
                a, b = a.flatten(1).double(), b.flatten(1).double()
                assert ((a - b).norm(dim=1) <= 1e-5 * b.norm(dim=1)).all(), i


def test_autotune_times_the_patches_once():
    """Without albedo the patches leave nothing to the kernel whose grid is tuned: one timing stands for the
    four areas, and the mean crop stays."""
    sc = make_scene(grid=24, k_exp=79, fit_light=2, crops=(64,), noise=0.0)
    ctx = tdi.Context(sc.model, sc.opts)
    b = tdi.Batch(ctx, sc.frames * 64)
    res = b.autotune(np.tile(sc.init(), (64, 1)).astype(np.float32), reps=1)
    shape = b.launch_shape()
    b.close()
    ctx.close()
    assert len(set(res["dI_ms"].values())) == 1 and min(res["dI_ms"].values()) > 0
    assert shape == (res["jtj_splits"], 64 * 64)
