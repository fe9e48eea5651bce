"""Subspace eigensolver against LAPACK where its Jacobi rounds and its Cholesky pass change shape:
odd and even numbers of columns around the pairs of a round (1, 2, 3, 15 .. 17, 31, 32), n at a
multiple of 16 and next to it, repeated eigenvalues, and matrices scaled by powers of two."""
import numpy as np
import pytest

import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu


def gapped(n, top, seed):
    """Symmetric with eigenvalues `top` over a floor 1e-4 of the smallest; its eigenvectors."""
    rng = np.random.default_rng(seed)
    V, _ = np.linalg.qr(rng.standard_normal((n, n)))
    w = np.concatenate([np.full(n - len(top), 1e-4 * np.min(top)), np.sort(top)])
    G = (V * w) @ V.T
    return 0.5 * (G + G.T), V, w


def solve(G, r):
    import torch
    n = G.shape[0]
    U, w = empty(n * r), torch.empty(r, dtype=torch.float64, device="cuda")
    m = tdx.sym_eig_topr_ex(dev(np.ascontiguousarray(G.ravel(order="F"), np.float64)), n, r, U, w)
    return m, host(U).reshape((n, r), order="F").astype(np.float64), w.cpu().numpy()


@pytest.mark.parametrize("n,r", [(1, 1), (2, 1), (3, 2), (17, 3), (33, 15), (48, 16), (49, 17), (127, 31), (128, 32),
                                 (32, 32), (31, 31)])
@pytest.mark.parametrize("power", [0, -200, 150])
def test_pairs_and_scales(n, r, power):
    top = np.linspace(1.0, 2.0, r)
    G, V, w = gapped(n, top, n + r)
    m, U, got = solve(G * 2.0 ** power, r)
    # the path stops at a residual of 1e-12 ||H||_F; eigenvalues are within it, vectors within it
    # over the gap (1 / 31 of the largest, at 32 columns)
    assert m == 1
    assert np.max(np.abs(got * 2.0 ** -power - w[n - r:])) <= 1e-11 * 2.0
    Vt = V[:, n - r:]
    assert np.max(np.abs(np.abs(np.sum(U * Vt, axis=0)) - 1.0)) <= 1e-6
    assert np.max(np.abs(U.T @ U - np.eye(r))) <= 1e-6


@pytest.mark.parametrize("r", [2, 9, 32])
def test_repeated_eigenvalues_and_diagonal(r):
    """Equal eigenvalues (any basis of their space will do) and a diagonal matrix (no rotation)."""
    n = 40
    G, V, w = gapped(n, np.ones(r), r)
    _, U, got = solve(G, r)
    P = V[:, n - r:] @ V[:, n - r:].T
    assert np.max(np.abs(got - 1.0)) <= 1e-11
    assert np.max(np.abs(U @ U.T - P)) <= 2e-6
    d = np.concatenate([np.full(n - r, 1e-4), np.linspace(1.0, 2.0, r)])
    _, U, got = solve(np.diag(d), r)
    assert np.max(np.abs(got - d[n - r:])) <= 2e-11
    assert np.max(np.abs(U - np.eye(n)[:, n - r:])) <= 1e-6
