"""Gram of an unfolding through LDS: FP32 with and without whole vectors, BF16 without, at the
edges of the row blocks (16), pair counts (1, 3, 6, 9 a wave) and column steps (64)."""
import numpy as np
import pytest

import oracle as O
import tdx
from helpers import dev

pytestmark = pytest.mark.gpu

CASES = [(1, 1), (16, 4), (17, 3, 65), (4, 33, 1), (63, 49, 5), (64, 97, 3), (12, 113, 20), (128, 5, 13), (5, 128, 64),
         (125, 7, 3, 2), (96, 2, 33), (81, 80, 79)]


@pytest.mark.parametrize("storage", [tdx.TDX_F32, tdx.TDX_BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("dims", CASES)
def test_gram_any_against_fp64(dims, off, storage):
    import torch
    rng = np.random.default_rng(sum(dims) + off)
    X = rng.standard_normal(int(np.prod(dims))).astype(np.float32)
    Xd = dev(X)
    if storage == tdx.TDX_BF16:
        q = torch.empty(X.size, dtype=torch.int16, device="cuda")
        tdx.quantize_bf16(Xd, q)
        X, Xd = (O.bf16_bits(X).astype(np.uint32) << 16).view(np.float32), q
    buf = torch.full((X.size + off,), 1, dtype=Xd.dtype, device="cuda")
    buf[off:].copy_(Xd)
    T = X.astype(np.float64).reshape(dims, order="F")
    for mode in range(len(dims)):
        n = dims[mode]
        G = torch.full((n * n,), float("nan"), dtype=torch.float64, device="cuda")
        tdx.unfold_gram(buf[off:], dims, mode, G, dtype=storage)
        got = G.cpu().numpy().reshape(n, n)
        A = np.moveaxis(T, mode, 0).reshape(n, -1)
        # a sum of K rounded FP32 products in any order: (K + 2) 2^-24 of the sum of magnitudes
        bound = (A.shape[1] + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(A).T) + 1e-30
        assert np.all(np.abs(got - A @ A.T) <= bound), (dims, mode)
        assert np.array_equal(got, got.T)
