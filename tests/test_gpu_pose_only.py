"""Fits of the pose alone (6 unknowns: no basis column, the smallest solve) against the FP64 oracle: three
batched Gauss-Newton iterations of one, two and twenty frames.  The Jacobian and J^T J are FP32 to about
1e-6 of themselves (BF16 parts), the 6 x 6 system's condition is below 1e3, so a step is good to 1e-3 of
itself with room to spare."""
import importlib

import numpy as np
import pytest

import pyoracle as O
from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")
abi = importlib.import_module("3di_amd.abi")


@pytest.mark.parametrize("n", [1, 2, 20])
def test_pose_only_fit(n):
    sc = make_scene(grid=40, k_exp=10, crops=(96, 80), noise=0.01)
    pose = sc.lay["pose"]
    opts = abi.default_options(fit_exp=0, max_iters=3, use_landmarks=0)
    frames = [sc.frames[i % 2] for i in range(n)]
    rng = np.random.default_rng(4)
    theta = np.stack([sc.truths[i % 2].theta[pose:pose + 6] for i in range(n)])
    theta[:, :3] += rng.normal(0, 0.5, (n, 3))
    theta[:, 3:] += rng.normal(0, 0.005, (n, 3))
    theta = theta.astype(np.float32)
    ctx = tdi.Context(sc.model, opts)
    b = tdi.Batch(ctx, frames)
    assert b.K == 6
    got, reports = b.fit_batched(torch.from_numpy(theta.copy()).cuda())
    got = got.cpu().numpy()
    b.close()
    ctx.close()
    want, _ = O.Scene(sc.model, frames, opts).fit(theta.astype(np.float64))
    for i in range(n):
        assert reports[i].status == 0
        step = np.abs(want[i] - theta[i])
        assert step.max() > 1e-3
        assert np.abs(got[i] - want[i]).max() <= 1e-3 * step.max(), (i, got[i] - want[i], step)
