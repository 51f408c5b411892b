"""The blocked FP64 solve at the edges of its 32-column panels and of the 704 columns that its back
substitution takes at once, condition 1e6: FP64 throughout, so only the solution's rounding to FP32
shows in the residual (2^-24 of each entry; twice that allowed)."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


@pytest.mark.parametrize("n,K", [(2, 113), (1, 127), (3, 128), (1, 129), (1, 704), (1, 735), (2, 736), (1, 737), (1, 1441)])
def test_residual_at_panel_edges(n, K):
    rng = np.random.default_rng(K)
    q, _ = np.linalg.qr(rng.standard_normal((K, K)))
    h = (q * np.geomspace(1.0, 1e6, K)) @ q.T
    H = np.stack([((np.tril(h) + np.tril(h, -1).T) * (1 + i)).astype(np.float32) for i in range(n)])
    g = rng.standard_normal((n, K)).astype(np.float32)
    d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), 0)
    assert (st.cpu().numpy() == 0).all()
    for i in range(n):
        A, x = H[i].astype(np.float64), d[i].cpu().numpy().astype(np.float64)
        assert np.all(np.abs(A @ x + g[i]) <= 2.0 ** -23 * (np.abs(A) @ np.abs(x))), (K, i)
