"""Vertex synthesis against FP64 numpy at the edges of its tiles: 16 vertices per workgroup, 16
frames per group, four groups per staging, 80 basis columns at a time."""
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")
synth = importlib.import_module("3di_amd.synth")


@pytest.mark.parametrize("grid,k_id,k_exp,n", [
    (16, 0, 1, 1), (17, 0, 79, 1), (17, 0, 80, 17), (20, 0, 81, 16), (20, 0, 161, 66), (17, 40, 20, 4),
    (19, 81, 80, 65), (16, 1, 83, 3), (17, 80, 7, 33)])
def test_synthesis_matches_fp64(grid, k_id, k_exp, n):
    sc = make_scene(grid=grid, k_exp=k_exp, k_id=k_id, fit_id=k_id > 0, crops=(48,), noise=0.0, seed=grid + k_exp, cfg=61)
    m, lay, fr = sc.model, sc.lay, sc.frames[0]
    rng = np.random.default_rng(5)
    theta = np.tile(sc.truths[0].theta, (n, 1))
    theta[:, :lay["pose"]] = rng.uniform(-1, 1, (n, lay["pose"]))
    theta[:, lay["pose"] + 3:lay["pose"] + 6] += rng.uniform(-0.2, 0.2, (n, 3))
    theta = theta.astype(np.float32)
    ctx = tdi.Context(m, sc.opts)
    b = tdi.Batch(ctx, [fr] * n)
    xyz, xyp = (t.cpu().numpy() for t in b.synthesize(theta))
    b.close()
    ctx.close()
    for i in range(n):
        th = theta[i].astype(np.float64)
        p = m.mean_shape.astype(np.float64).reshape(-1) + m.exp_basis.astype(np.float64) @ th[lay["exp"]:lay["pose"]]
        if k_id:
            p = p + m.id_basis.astype(np.float64) @ th[lay["id"]:lay["exp"]]
        u = th[lay["pose"] + 3:lay["pose"] + 6]
        t = np.linalg.norm(u)
        x, y, z = u / t
        N = np.array([[0, -z, y], [z, 0, -x], [-y, x, 0]])
        R = np.eye(3) + np.sin(t) * N + (1 - np.cos(t)) * N @ N
        q = p.reshape(-1, 3) @ R.T + th[lay["pose"]:lay["pose"] + 3]
        xy = np.stack([fr.phix * q[:, 0] / q[:, 2] + fr.cx, fr.phiy * q[:, 1] / q[:, 2] + fr.cy], 1)
        # FP64 rounded once: half an FP32 ulp, and 1e-12 of the operands for the FP64 roundings
        assert np.all(np.abs(xyz[i] - q) <= 2.0 ** -24 * np.abs(q) + 1e-9), i
        assert np.all(np.abs(xyp[i] - xy) <= 2.0 ** -24 * np.abs(xy) + 1e-8), i


@pytest.mark.parametrize("grid,k_id,k_exp", [(16, 0, 1), (17, 0, 79), (20, 0, 161), (19, 81, 80), (17, 80, 7), (23, 33, 16)])
def test_one_frame_gives_the_bits_of_a_list(grid, k_id, k_exp):
    """A frame alone, in a list of three and in one of twenty: three forms, one order of the sums."""
    sc = make_scene(grid=grid, k_exp=k_exp, k_id=k_id, fit_id=k_id > 0, crops=(48,), noise=0.0, seed=grid, cfg=62)
    rng = np.random.default_rng(6)
    theta = np.tile(sc.truths[0].theta, (20, 1))
    theta[:, :sc.lay["pose"]] = rng.uniform(-1, 1, (20, sc.lay["pose"]))
    theta = theta.astype(np.float32)
    ctx = tdi.Context(sc.model, sc.opts)
    out = {}
    for n in (1, 3, 20):
        b = tdi.Batch(ctx, [sc.frames[0]] * n)
        out[n] = [t[:1].cpu().numpy() for t in b.synthesize(theta[:n])] + [b.fit_buffers(theta[:n])[0][:1].cpu().numpy()]
        b.close()
    ctx.close()
    for n in (3, 20):
        assert all((a == c).all() for a, c in zip(out[1], out[n])), n
