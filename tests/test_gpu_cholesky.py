"""The per-frame Cholesky solve at the edges of its 16 x 16 blocks and of the two entries a lane
holds, both modes, against FP64 numpy; a matrix that is not positive definite between two that are."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
tdi = importlib.import_module("3di_amd.tdi")


def _systems(n, K, seed, cond):
    rng = np.random.default_rng(seed)
    H = np.empty((n, K, K), np.float32)
    for i in range(n):
        q, _ = np.linalg.qr(rng.standard_normal((K, K)))
        h = (q * np.geomspace(1.0, cond, K)) @ q.T
        s = 10.0 ** rng.uniform(-1, 1, K)
        h = (h * s[:, None] * s[None, :]).astype(np.float32)
        H[i] = np.tril(h) + np.tril(h, -1).T
    return H, rng.standard_normal((n, K)).astype(np.float32)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("K", [1, 2, 15, 16, 17, 48, 63, 64, 65, 80, 81, 94, 96, 97, 111, 112])
def test_solve_at_block_edges(K, mode):
    cond = 1e3
    H, g = _systems(3, K, K, cond)
    d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), mode)
    assert (st.cpu().numpy() == 0).all()
    for i in range(3):
        h = H[i].astype(np.float64)
        want = -np.linalg.solve(h, g[i].astype(np.float64))
        # backward error: the residual against |H||x|, FP32 rounding of the solution (2^-24 per entry);
        # mode 1's refinement leaves (cond 2^-24)^2 of the solution beyond it
        x = d[i].cpu().numpy().astype(np.float64)
        scale = np.abs(h) @ np.abs(want) + np.abs(g[i])
        assert np.all(np.abs(h @ x + g[i]) <= (2.0 ** -23 + (cond * 2.0 ** -22) ** 2) * scale), (K, mode, i)


@pytest.mark.parametrize("mode", [0, 1])
def test_ill_conditioned_and_not_positive_definite(mode):
    # cond 1e7: mode 1's correction is too large (or its FP32 pivot breaks down), FP64 takes over
    H, g = _systems(3, 94, 7, 1e7)
    H[1] = -H[1]
    d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), mode)
    assert st.cpu().numpy().tolist() == [0, 4, 0]
    for i in (0, 2):
        h = H[i].astype(np.float64)
        x = d[i].cpu().numpy().astype(np.float64)
        want = -np.linalg.solve(h, g[i].astype(np.float64))
        scale = np.abs(h) @ np.abs(want) + np.abs(g[i])
        assert np.all(np.abs(h @ x + g[i]) <= 2.0 ** -23 * scale)   # FP32 rounding of the solution
