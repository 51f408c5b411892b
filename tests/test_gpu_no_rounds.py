"""Batched fits without a line-search round (max_ls = 0, or a smallest step above 1): nothing is
evaluated, so theta stays and the reported objective is theta's, to the bits of the same evaluation in a
fit that takes no iteration."""
import importlib

import numpy as np
import pytest

from scenes import make_scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")
abi = importlib.import_module("3di_amd.abi")


def _fit(sc, **kw):
    opts = abi.default_options(fit_light=2, **kw)
    ctx = tdi.Context(sc.model, opts)
    b = tdi.Batch(ctx, sc.frames)
    th, reports = b.fit_batched(torch.from_numpy(sc.init().astype(np.float32)).cuda())
    th = th.cpu().numpy()
    b.close()
    ctx.close()
    return th, reports


@pytest.mark.parametrize("kw,iters", [(dict(max_ls=0, max_iters=3), 3), (dict(t_min=2.0, max_iters=3), 1)])
def test_fit_without_rounds(kw, iters):
    sc = make_scene(grid=40, k_exp=10, fit_light=2, crops=(96, 80, 64))
    want, ref = _fit(sc, max_iters=0)
    th, reports = _fit(sc, **kw)
    assert (th == sc.init().astype(np.float32)).all() and (want == th).all()
    for r, q in zip(reports, ref):
        assert r.iters == iters and r.n_pixels == q.n_pixels
        assert r.objective == q.objective
