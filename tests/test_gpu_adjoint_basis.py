"""Coefficient gradients of the render loss at the edges of their tiles (16 frames, 80 columns, 16 rows:
grid 40 and 41 leave 0 and 3 rows over): against basis^T times the same call's per-vertex gradient in
FP64.  That gradient is returned in FP32, so the bound is 2^-24 of each product's magnitude, and of the
result's for its own rounding."""
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


@pytest.mark.parametrize("n, k_exp, k_id, grid", [(1, 1, 0, 41), (15, 16, 3, 40), (16, 80, 17, 41), (17, 81, 90, 40)])
def test_coefficient_gradients(n, k_exp, k_id, grid):
    sc = make_scene(grid=grid, k_exp=k_exp, k_id=k_id, fit_id=k_id > 0, crops=(48,) * n, pose_deg=10.0)
    b = tdi.Batch(tdi.Context(sc.model, sc.opts), sc.frames)
    th = torch.from_numpy(sc.init().astype(np.float32)).cuda()
    dv = torch.zeros((n, sc.model.n_vertices, 3), device="cuda")
    _, gth, gv = b.render_loss(th, dv)
    torch.cuda.synchronize()
    gth, gv = gth.cpu().numpy().astype(np.float64), gv.cpu().numpy().astype(np.float64).reshape(n, -1)
    assert np.abs(gv).max() > 0
    parts = [(sc.model.exp_basis, sc.lay["exp"], k_exp)]
    if k_id:
        parts.append((sc.model.id_basis, sc.lay["id"], k_id))
    for basis, o, k in parts:
        B = basis.astype(np.float64)[:, :k]
        want, scale = gv @ B, np.abs(gv) @ np.abs(B)
        assert np.all(np.abs(gth[:, o:o + k] - want) <= 2.0 ** -24 * (scale + np.abs(want)) * 1.01)
