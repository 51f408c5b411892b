"""The barrier's FP64 terms against the oracle: the padded column counts around the launch's LDS limit, and
more unknowns than the derivative kernel's 112 without landmarks; a landmark at depth zero."""
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


@pytest.mark.parametrize("k_exp,light,use_landmarks", [
    (49, 2, 1), (53, 2, 1), (58, 2, 1), (97, 2, 1), (97, 2, 0), (98, 2, 0), (200, 0, 0), (1100, 0, 0)])
def test_barrier_terms(k_exp, light, use_landmarks):
    sc = make_scene(grid=24, k_exp=k_exp, fit_light=light, crops=(48, 40), noise=0.0, use_landmarks=use_landmarks)
    th = sc.init()
    ctx = tdi.Context(sc.model, sc.opts)
    b = tdi.Batch(ctx, sc.frames)
    H, g, obj = (t.cpu().numpy() for t in b.barrier_terms(th.astype(np.float32)))
    b.close()
    ctx.close()
    orc = sc.oracle()
    for i in range(2):
        ob, go, Ho = orc.barrier(i, th[i].astype(np.float32).astype(np.float64))
        assert np.isfinite(ob)
        # FP64 on both sides; g is a sum of FP32 terms (the configurations' bounds for the same terms)
        errors = [abs(obj[i] - ob) / abs(ob), np.linalg.norm(H[i] - Ho) / np.linalg.norm(Ho),
                  np.linalg.norm(g[i] - go) / np.linalg.norm(go)]
        assert errors[0] < 1e-12 and errors[1] < 1e-10 and errors[2] < 1e-6, errors


def test_landmark_at_depth_zero():
    """The rotation about z and no expression put a landmark at depth exactly zero: its derivatives are not
    finite, but the light's, which moves no landmark, are zero still."""
    sc = make_scene(grid=24, k_exp=10, fit_light=2, crops=(48,), noise=0.0)
    theta = sc.init().astype(np.float32)
    pose = sc.lay["pose"]
    theta[0, :pose] = 0
    z = sc.model.mean_shape.astype(np.float32).reshape(-1, 3)[sc.model.landmark_ids[20], 2]
    theta[0, pose:pose + 6] = (3.0, 2.0, -z, 0.0, 0.0, 0.25)
    ctx = tdi.Context(sc.model, sc.opts)
    b = tdi.Batch(ctx, sc.frames)
    H, g, _ = b.barrier_terms(theta)
    b.close()
    ctx.close()
    light = slice(pose + 6, None)
    assert not torch.isfinite(g[0, pose]) and (g[0, light] == 0).all() and (H[0, light, light] == 0).all()
