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


def test_fp32_pivots_that_break_down():
    """Matrices that FP64 factors and FP32 does not: H = S L L^T S, L unit lower bidiagonal with 2 or 3 below
    the diagonal in chains of eleven, S whole numbers; exact in FP32, condition below 2^38.  The pivots of
    L L^T are 1 and an error in one grows by 4 to 9 a column, so FP32's turn negative or leave a correction
    that is refused, and mode 1 ends in the FP64 factorisation: the bits of mode 0.  Every fourth matrix is
    not positive definite in either."""
    rng = np.random.default_rng(11)
    n, K = 256, 94
    c = rng.integers(2, 4, (n, K))
    c[:, ::11] = 0
    L = np.tile(np.eye(K), (n, 1, 1))
    L[:, np.arange(1, K), np.arange(K - 1)] = c[:, 1:]
    S = rng.integers(50, 201, (n, K)).astype(np.float64)
    H = S[:, :, None] * (L @ L.transpose(0, 2, 1)) * S[:, None, :]
    h = H.astype(np.float32)
    assert (h == H).all()
    # the FP32 pivots of the equilibrated matrices (tridiagonal)
    r = np.einsum("nii->ni", h) ** np.float32(-0.5)
    s = h * r[:, :, None] * r[:, None, :]
    d, broke = s[:, 0, 0], np.zeros(n, bool)
    for k in range(1, K):
        d = s[:, k, k] - s[:, k, k - 1] ** 2 / d
        broke |= ~(d > 0)
        d = np.where(d > 0, d, np.float32(1))
    assert broke.sum() > n // 2                  # the break-down is reached, whatever the last bits
    x = rng.integers(-4, 5, (n, K))
    g = -np.einsum("nij,nj->ni", H, x)
    assert (g == g.astype(np.float32)).all()
    bad = np.arange(n) % 4 == 3
    h[bad, 50, 50] = -1.0
    ht, gt = torch.from_numpy(h).cuda(), torch.from_numpy(g.astype(np.float32)).cuda()
    d0, st0 = (t.cpu().numpy() for t in tdi.cholesky_solve(ht, gt, 0))
    d1, st1 = (t.cpu().numpy() for t in tdi.cholesky_solve(ht, gt, 1))
    assert (st0 == np.where(bad, 4, 0)).all() and (st1 == st0).all()
    assert (d0[~bad] == d1[~bad]).all()
    # |x| <= 4; FP64's error is about K 2^-53 times the condition
    assert np.abs(d0[~bad] - x[~bad]).max() < 2.0 ** -8


@pytest.mark.parametrize("K,mode", [(1, 0), (5, 0), (94, 0), (94, 1), (112, 1), (200, 0)])
def test_infinite_diagonal_entries(K, mode):
    """An unknown whose diagonal entry is infinite (an overflowed weight) does not move, and the others are
    solved without it, as by the plain sequence: its column of the factor is zero."""
    H, g = _systems(1, K, K, 1e2)
    held = sorted({0, K // 3, K - 1})
    H[0, held, held] = np.inf
    d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), mode)
    assert st.cpu().numpy().tolist() == [0]
    x = d[0].cpu().numpy().astype(np.float64)
    assert (x[held] == 0).all()
    free = np.setdiff1d(np.arange(K), held)
    h = H[0][np.ix_(free, free)].astype(np.float64)
    scale = np.abs(h) @ np.abs(x[free])
    assert np.all(np.abs(h @ x[free] + g[0, free]) <= 2.0 ** -23 * scale)   # FP32 rounding of the solution


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_few_unknowns(K):
    """A thread per matrix up to 8 unknowns: more than two workgroups of matrices, every fifth not positive
    definite, both modes, and mode 1 no worse than mode 0."""
    n = 130
    H, g = _systems(n, K, 40 + K, 1e4)
    bad = np.arange(n) % 5 == 2
    H[bad, K - 1, K - 1] = -1.0
    for mode in (0, 1):
        d, st = tdi.cholesky_solve(torch.from_numpy(H).cuda(), torch.from_numpy(g).cuda(), mode)
        assert (st.cpu().numpy() == np.where(bad, 4, 0)).all()
        x = d.cpu().numpy().astype(np.float64)
        h = H.astype(np.float64)
        res = np.abs(np.einsum("nij,nj->ni", h, x) + g)
        scale = np.einsum("nij,nj->ni", np.abs(h), np.abs(x))
        # FP32 rounding of the solution; mode 1 above 8 unknowns leaves (cond 2^-24)^2 beyond it
        assert np.all((res <= (2.0 ** -23 + (1e4 * 2.0 ** -22) ** 2 * (mode and K > 8)) * scale)[~bad])
