"""The shared pass with FP32 T (modes 1 and 2 of an FP32 or split BF16 sweep from one pass over the
tensor): one sweep against FP64 at the edges of its tiles (32 and 256 rows, chunks of 64 and 128,
pairs of slabs, 16 columns), scale shared between factors, and entries near the ends of the range."""
import numpy as np
import pytest
import torch

import tdx

pytestmark = pytest.mark.gpu

# I0 a multiple of 4 (FP32) and 8 (BF16), at least 2^26 elements; partial chunks, row tiles and pairs
SHAPES = [((512, 512, 256), 64), ((1032, 257, 255), 33), ((2056, 33, 1001), 16), ((264, 1000, 259), 20),
          ((4096, 16, 1027), 48), ((1160, 2048, 29), 5)]


def setup(dims, R, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    F = [torch.randn(R, d, device="cuda", generator=g) for d in dims]
    kr = (F[2].t()[:, None, :] * F[1].t()[None, :, :]).reshape(-1, R)
    X = (kr @ F[0]).reshape(-1)
    X += 0.1 * float(X.std()) * torch.randn(X.shape, device="cuda", generator=g)
    return X, [f + 0.3 * torch.randn(f.shape, device="cuda", generator=g) for f in F]


def sweep64(X, dims, F):
    """one CP-ALS sweep in FP64; also sum |X| |KR| |V^-1| per entry, the scale of its rounding"""
    X3 = X.reshape(dims[2], dims[1], dims[0]).double()
    F = [f.double() for f in F]
    scale = []
    for m in range(3):
        a, b = [F[k] for k in range(3) if k != m]
        V = torch.linalg.inv((a @ a.t()) * (b @ b.t()))

        def mttkrp(X3, F):
            if m == 0:
                T = torch.matmul(F[1], X3)                       # I2 x R x I0
                return (T * F[2].t()[:, :, None]).sum(0)         # R x I0
            T = torch.matmul(X3, F[0].t())                       # I2 x I1 x R
            if m == 1:
                return (T * F[2].t()[:, None, :]).sum(0).t()
            return (T * F[1].t()[None, :, :]).sum(1).t()

        scale.append(V.abs() @ mttkrp(X3.abs(), [f.abs() for f in F]))
        F[m] = V @ mttkrp(X3, F)
        F[m] = F[m].float().double()
    return F, scale


def run(X, dims, R, F, storage, shared=1):
    U = [f.clone() for f in F]
    o = tdx.default_cp_options()
    o.init, o.max_sweeps, o.storage, o.shared_pass = 1, 1, storage, shared
    if storage == tdx.TDX_BF16:
        o.opening_sweeps, o.opening_split, o.refine_sweeps = 1, 1, 0
    st, _, fit, _ = tdx.cp_als_ex(X, dims, R, U, o)
    assert st == tdx.TDX_OK
    return U, fit


@pytest.mark.parametrize("storage", [tdx.TDX_F32, tdx.TDX_BF16])
@pytest.mark.parametrize("dims,R", SHAPES)
def test_one_sweep_against_fp64(dims, R, storage):
    X, F = setup(dims, R, sum(dims) + R)
    U, _ = run(X, dims, R, F, storage)
    ref, scale = sweep64(X if storage == tdx.TDX_F32 else X.bfloat16(), dims, F)
    # FP32: at most 2^-18 of the sum of magnitudes (64 roundings of FP32 in a row) in each mode, and
    # what a mode's error does to the next ones; BF16: coefficients of 17 bits, 2^-17 each, two a term
    unit = 2.0 ** -18 if storage == tdx.TDX_F32 else 2.0 ** -15
    for m in range(3):
        err = (U[m].double() - ref[m]).norm() / scale[m].norm()
        assert float(err) <= (m + 1) * unit, (m, float(err))
        # and no entry away from the others
        assert float(((U[m].double() - ref[m]).abs() / scale[m]).max()) <= 16 * (m + 1) * unit


def test_factor_scale_is_free():
    """Start factors B and C times 2^55 make A 2^-110 times as large, and T with it were its scale not
    taken out."""
    dims, R = (520, 400, 330), 24
    X, F = setup(dims, R, 3)
    U, fit = run(X, dims, R, F, tdx.TDX_F32)
    V, fit2 = run(X, dims, R, [F[0], F[1] * 2.0 ** 55, F[2] * 2.0 ** 55], tdx.TDX_F32)
    for m, s in enumerate((-110, 55, 55)):
        assert float((V[m].double() * 2.0 ** -s - U[m].double()).norm() / U[m].double().norm()) <= 2.0 ** -18, m
    assert abs(fit[0] - fit2[0]) <= 1e-6


def test_tiny_slabs_and_a_huge_entry():
    """Slabs and an entry near the ends of the FP32 range (FP32 products in their tiles) beside ordinary ones,
    against the separate passes."""
    dims, R = (520, 400, 330), 16
    X, F = setup(dims, R, 4)
    X3 = X.view(dims[2], -1)
    X3[:40] *= 2.0 ** -112
    X3[100, 12345] = 2.0 ** 119.5  # (one entry: the sum over a whole slab of such would overflow)
    F[2][:, 100] *= 2.0 ** -116
    U, _ = run(X, dims, R, F, tdx.TDX_F32)
    W, _ = run(X, dims, R, F, tdx.TDX_F32, shared=0)
    for m in range(3):
        u, w = U[m].double(), W[m].double()
        assert bool(torch.isfinite(u).all()), m
        err = (u - w).norm(dim=0) / w.norm(dim=0) if m == 2 else (u - w).norm() / w.norm()
        assert float(err.max()) <= 2.0 ** -14, m
