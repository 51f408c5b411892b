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


def test_break_downs_at_every_panel():
    """A pivot that is not positive in the first, an inner and the last panel, at its first and last column,
    between matrices that are positive definite: only those stop."""
    n, K = 10, 200
    rng = np.random.default_rng(1)
    a = rng.standard_normal((n, K, K)) / np.sqrt(K)
    H = (a @ a.transpose(0, 2, 1) + 0.1 * np.eye(K)).astype(np.float32)
    bad = {1: 0, 2: 31, 4: 32, 5: 100, 7: 192, 8: 199}
    for i, k in bad.items():
        H[i, k, k] = -1.0
    g = rng.standard_normal((n, K)).astype(np.float32)
    d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), 0)
    assert st.cpu().numpy().tolist() == [4 if i in bad else 0 for i in range(n)]
    for i in set(range(n)) - set(bad):
        A, x = H[i].astype(np.float64), d[i].cpu().numpy().astype(np.float64)
        assert np.all(np.abs(A @ x + g[i]) <= 2.0 ** -23 * (np.abs(A) @ np.abs(x))), i
