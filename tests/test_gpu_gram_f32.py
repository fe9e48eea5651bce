"""Gram of FP32 tensors with whole vectors, from three BF16 parts per element: entry by entry against
FP64 at the edges of its tiles (16-row blocks, 32, 64 and 128 rows, steps of 64 columns), rows of very
different magnitude, and infinities, NaN and values whose squares overflow."""
import numpy as np
import pytest

import tdx
from helpers import dev

pytestmark = pytest.mark.gpu


def gram(X, dims, mode):
    import torch
    n = dims[mode]
    G = torch.full((n * n,), float("nan"), dtype=torch.float64, device="cuda")
    tdx.unfold_gram(dev(X), dims, mode, G)
    return G.cpu().numpy().reshape(n, n)


def unfold(X, dims, mode):
    T = X.astype(np.float64).reshape(dims, order="F")
    return np.moveaxis(T, mode, 0).reshape(dims[mode], -1)


def bound(A):
    # a sum of K FP32 products in any order, (K + 2) 2^-24 of the sum of magnitudes; underflow
    return (A.shape[1] + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(A).T) + A.shape[1] * 2.0 ** -149


@pytest.mark.parametrize("dims,mode", [((4, 1), 0), ((16, 63), 0), ((36, 65), 0), ((64, 64), 0), ((68, 129), 0),
                                       ((128, 200), 0), ((4, 7, 3), 1), ((20, 33, 5), 1), ((8, 64, 9), 1),
                                       ((12, 65, 11), 1), ((4, 97, 50), 1), ((64, 128, 30), 1), ((68, 31, 2), 1),
                                       ((4, 5, 16, 3), 2), ((16, 8, 127), 2)])
def test_edges(dims, mode):
    X = np.random.default_rng(sum(dims) + mode).standard_normal(int(np.prod(dims))).astype(np.float32)
    A = unfold(X, dims, mode)
    assert np.all(np.abs(gram(X, dims, mode) - A @ A.T) <= bound(A))


@pytest.mark.parametrize("dims,mode", [((36, 150), 0), ((8, 40, 30), 1)])
def test_rows_of_different_magnitude(dims, mode):
    """A block of 4 rows near 2^-105 against rows near 2^55."""
    rng = np.random.default_rng(3)
    T = rng.standard_normal(dims).astype(np.float32) * np.float32(2.0 ** 55)
    at = [slice(None)] * len(dims)
    at[mode] = slice(8, 12)
    T[tuple(at)] *= np.float32(2.0 ** -160)
    X = T.ravel(order="F")
    A = unfold(X, dims, mode)
    assert np.all(np.abs(gram(X, dims, mode) - A @ A.T) <= bound(A))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e30])
@pytest.mark.parametrize("dims,mode", [((36, 150), 0), ((8, 40, 30), 1)])
def test_nonfinite_and_overflow(dims, mode, value):
    """One such entry: its row and column become infinite or NaN as products say, the rest stays."""
    X = (np.abs(np.random.default_rng(4).standard_normal(int(np.prod(dims)))) + 0.1).astype(np.float32)
    A = unfold(X, dims, mode)
    B = A.copy()
    B[17, 70] = value
    Y = np.moveaxis(B.reshape([dims[mode]] + [d for m, d in enumerate(dims) if m != mode]), 0, mode)
    got = gram(Y.astype(np.float32).ravel(order="F"), dims, mode)
    rest = np.arange(dims[mode]) != 17
    assert np.all(np.abs(got - A @ A.T)[np.ix_(rest, rest)] <= bound(A)[np.ix_(rest, rest)])
    if np.isnan(value):
        assert np.all(np.isnan(got[17])) and np.all(np.isnan(got[:, 17]))
    elif np.isinf(value):
        assert got[17, 17] == np.inf and np.all(got[17, rest] == value) and np.all(got[rest, 17] == value)
    else:
        assert got[17, 17] == np.inf  # the square overflows FP32
        ref = (B @ B.T)[17, rest]
        assert np.all(np.abs(got[17, rest] - ref) <= (A.shape[1] + 2) * 2.0 ** -24 * ref)


@pytest.mark.parametrize("dims,mode", [((116, 190), 0), ((8, 125, 33), 1), ((128, 65), 0), ((4, 113, 16), 1)])
def test_all_eight_row_blocks(dims, mode):
    """113 to 128 rows, whose waves hold pairs of their own: the edges, and both kinds of tile that are
    multiplied in FP32."""
    test_edges(dims, mode)
    test_rows_of_different_magnitude(dims, mode)
    if int(np.prod(dims)) // dims[mode] > 70:
        for value in (np.inf, np.nan, 1e30):
            test_nonfinite_and_overflow(dims, mode, value)
