"""FP32 products from three BF16 parts keep their bits where entries far below the ordinary ones stand
beside them: rows of such entries, and a single one that alone makes up a result."""
import numpy as np
import pytest
import torch

import oracle as O
import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

POWERS = [-104, -112, -120, -130]


@pytest.mark.parametrize("power", POWERS)
@pytest.mark.parametrize("dims,R", [((64, 70, 9), 20), ((132, 65, 7), 64), ((36, 33, 6, 5), 40), ((128, 64, 8), 16)])
def test_mttkrp(dims, R, power):
    rng = np.random.default_rng(sum(dims) + R)
    # (the factors lift the results from the bottom of the range)
    U = [(2.0 ** 9 * rng.standard_normal((d, R))).astype(np.float32) for d in dims]
    at = [d // 2 + 1 for d in dims]
    for u, i in zip(U, at):
        u[:, 0] = 0
        u[i, 0] = 2.0 ** 9 * 1.1  # column 0 meets one entry of each row
    for mode in range(len(dims)):
        X = rng.standard_normal(dims).astype(np.float32)
        row = [slice(None)] * len(dims)
        row[mode] = 3
        X[tuple(row)] *= np.float32(2.0 ** power)
        one = list(at)
        one[mode] = 11 if dims[mode] > 11 else 2
        X[tuple(one)] = 1.2345678 * 2.0 ** power
        flat = X.ravel(order="F")
        out = empty(dims[mode] * R)
        tdx.mttkrp_ex(dev(flat), tdx.TDX_F32, None, dims, [dev(u.ravel(order="F")) for u in U], R, mode, out)
        got = host(out).reshape((dims[mode], R), order="F")
        ref = O.mttkrp(flat, dims, [u.astype(np.float64) for u in U], mode)
        mag = O.mttkrp(np.abs(flat), dims, [np.abs(u).astype(np.float64) for u in U], mode)
        # roundings of a term in units of 2^-24: the parts left out, 64 of a sum, the slow factors, the
        # sums over slow indices and the partial
        terms = 70 + X.size // (dims[mode] * dims[1 if mode == 0 else 0])
        assert np.all(np.abs(got - ref) <= terms * 2.0 ** -24 * mag), mode


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("power", POWERS)
@pytest.mark.parametrize("dims,mode", [((128, 128, 8), 0), ((128, 128, 8), 1), ((64, 48, 12), 1), ((32, 20, 64), 2),
                                       ((100, 36, 20), 0)])
def test_gram(dims, mode, power, rows):
    rng = np.random.default_rng(sum(dims) + mode)
    X = np.moveaxis(rng.standard_normal(dims).astype(np.float32), mode, 0).copy()
    n = X.shape[0]
    M = X.reshape(n, -1)
    if rows:
        M[3] *= np.float32(2.0 ** power)
    M[7, 21] = 1.2345678 * 2.0 ** power  # beside ordinary entries of its row; met by row 9 alone
    M[9] = 0
    M[9, 21] = 2.0 ** 30 * 1.1
    flat = np.moveaxis(M.reshape(X.shape), 0, mode).ravel(order="F").astype(np.float32)
    G = torch.empty(n * n, dtype=torch.float64, device="cuda")
    tdx.unfold_gram(dev(flat), dims, mode, G)
    got, M64 = host(G).reshape(n, n), M.astype(np.float64)
    # 64 roundings of a step's sum, one a step, and the partial; products below the range are lost
    terms = 70 + M.shape[1] // 64
    mag = np.abs(M64) @ np.abs(M64).T
    assert np.all(np.abs(got - M64 @ M64.T) <= terms * 2.0 ** -24 * mag + M.shape[1] * 2.0 ** -149)


def test_shared_pass():
    """A row of the second factor that one entry near 2^-120 determines, in an FP32 sweep."""
    dims, R = (256, 16384, 9), 16
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    X = torch.randn(dims[2], dims[1], dims[0], device="cuda", generator=g)
    x = np.float32(1.2345678 * 2.0 ** -120)
    X[:, 77, :] = 0
    X[4, 77, 100] = float(x)
    U = [torch.randn(R, d, device="cuda", generator=g) * s for d, s in zip(dims, (1.0, 2.0 ** -5, 2.0 ** 5))]
    # (A comes out near 2^-9: M1 at 2^-122 and the row at 2^-125 are within FP32's normal range)
    C = U[2].double().cpu().numpy()
    o = tdx.default_cp_options()
    o.init, o.max_sweeps = 1, 1
    st, _, _, _ = tdx.cp_als_ex(X.reshape(-1), dims, R, U, o)
    assert st == tdx.TDX_OK
    A = U[0].double().cpu().numpy()
    ref = np.linalg.solve((A @ A.T) * (C @ C.T), float(x) * A[:, 100] * C[:, 4])
    got = U[1][:, 77].double().cpu().numpy()
    # one product and the roundings of T, the partial and the factor
    assert np.linalg.norm(got - ref) <= 2.0 ** -19 * np.linalg.norm(ref)
