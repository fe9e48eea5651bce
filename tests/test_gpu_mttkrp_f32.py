"""FP32 MTTKRP from three BF16 parts per operand: entry by entry against FP64 at the edges of its
tiles (32 rows, 64 fast indices, 16 columns), independence of the scale shared between factors,
and infinities, NaN and values that round to a BF16 infinity."""
import numpy as np
import pytest

import oracle as O
import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu


def run(X, dims, U, mode):
    R = U[0].shape[1]
    out = empty(dims[mode] * R)
    tdx.mttkrp_ex(dev(X), tdx.TDX_F32, None, dims, [dev(u.ravel(order="F")) for u in U], R, mode, out)
    return host(out).reshape((dims[mode], R), order="F")


def data(dims, R, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(int(np.prod(dims))).astype(np.float32),
            [rng.standard_normal((d, R)).astype(np.float32) for d in dims])


def bound(X, dims, U, mode):
    # roundings of a term in units of 2^-24 of its magnitude: the parts left out (1), the sums of 64
    # products (at most 64), w (3), the sums over the slow indices of a split and the partial
    terms = 70 + int(np.prod(dims)) // (dims[mode] * dims[1 if mode == 0 else 0])
    mag = O.mttkrp(np.abs(X), dims, [np.abs(u).astype(np.float64) for u in U], mode)
    return terms * 2.0 ** -24 * mag


@pytest.mark.parametrize("dims,R", [((4, 1, 1), 1), ((32, 64, 5), 16), ((36, 65, 3), 17), ((64, 33, 129), 33),
                                    ((132, 7, 31), 48), ((260, 129, 2), 64), ((8, 5, 3, 7), 5), ((68, 31, 6, 4), 64),
                                    ((4, 128, 200), 20)])
def test_entries_against_fp64(dims, R):
    X, U = data(dims, R, sum(dims) + R)
    U64 = [u.astype(np.float64) for u in U]
    for mode in range(len(dims)):
        got, ref = run(X, dims, U, mode), O.mttkrp(X, dims, U64, mode)
        assert np.all(np.abs(got - ref) <= bound(X, dims, U, mode)), (dims, R, mode)


def test_factor_scale_is_free():
    """2^100 moved from one factor to another changes nothing, bit for bit."""
    dims, R = (64, 70, 9), 24
    X, U = data(dims, R, 1)
    for mode, (up, down) in ((0, (1, 2)), (1, (0, 2)), (2, (0, 1))):
        V = list(U)
        V[up], V[down] = (U[up] * np.float32(2.0 ** 100)), (U[down] * np.float32(2.0 ** -100))
        assert np.array_equal(run(X, dims, U, mode), run(X, dims, V, mode)), mode


@pytest.mark.parametrize("power", [-124, -112, -98, 100, 124])
def test_tiny_and_huge_tensors(power):
    """Entries near the ends of the FP32 range, the results well inside it."""
    dims, R = (64, 70, 9), 40
    X, U = data(dims, R, 3)
    X = X * np.float32(2.0 ** power)
    U = [u * np.float32(2.0 ** (-power // 4)) for u in U]
    for mode in range(3):
        ref = O.mttkrp(X, dims, [u.astype(np.float64) for u in U], mode)
        assert np.all(np.abs(run(X, dims, U, mode) - ref) <= bound(X, dims, U, mode)), mode


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_nonfinite_and_largest_values(value):
    """One such entry in the tensor (a tile of each mode) or in a factor."""
    dims, R = (64, 70, 9), 20
    X, U = data(dims, R, 2)
    U = [np.abs(u) + np.float32(0.1) for u in U]
    if value == 3.4e38:
        U = [u * np.float32(1e-3) for u in U]
    at = (37, 41, 5)
    Y = X.copy()
    Y[at[0] + dims[0] * (at[1] + dims[1] * at[2])] = value
    for mode in range(3):
        got, clean = run(Y, dims, U, mode), run(X, dims, U, mode)
        rest = np.arange(dims[mode]) != at[mode]
        assert np.all(np.abs(got[rest] - clean[rest]) <= 2 * bound(X, dims, U, mode)[rest])
        if np.isnan(value):
            assert np.all(np.isnan(got[at[mode]]))
        elif np.isinf(value):
            assert np.all(got[at[mode]] == value)
        else:
            ref = O.mttkrp(Y, dims, [u.astype(np.float64) for u in U], mode)[at[mode]]
            assert np.all(np.abs(got[at[mode]] - ref) <= 1e-5 * np.abs(ref))
    if np.isinf(value):
        V = [u.copy() for u in U]
        V[0][3, 7] = value
        got = run(np.abs(X) + np.float32(0.1), dims, V, 1)
        assert np.all(got[:, 7] == value) and np.all(np.isfinite(np.delete(got, 7, axis=1)))
