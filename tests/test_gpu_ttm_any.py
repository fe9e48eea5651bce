"""Tensor-times-matrix outside the register kernel's range (modes above 128, ranks above 32, odd
extents, tensors off a 16-byte boundary): both factor layouts and both storages against FP64 at
the edges of the fibre tiles (64, 128), steps (16, 64) and column blocks (16, 64)."""
import numpy as np
import pytest

import oracle as O
import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 1), ((3, 5, 7), 2), ((17, 16, 5), 16), ((129, 3, 5), 17), ((5, 131, 9), 33), ((64, 65, 63), 48),
         ((200, 31, 2), 64), ((33, 2, 257), 65), ((130, 129, 3), 130), ((16, 300, 1), 40), ((1, 77, 1), 5),
         ((127, 61, 43), 20)]


@pytest.mark.parametrize("storage", [tdx.TDX_F32, tdx.TDX_BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("dims,r", CASES)
def test_ttm_any_against_fp64(dims, r, off, storage):
    import torch
    rng = np.random.default_rng(sum(dims) + r)
    X = rng.standard_normal(int(np.prod(dims))).astype(np.float32)
    Xd = dev(X)
    if storage == tdx.TDX_BF16:
        q = torch.empty(X.size, dtype=torch.int16, device="cuda")
        tdx.quantize_bf16(Xd, q)
        X, Xd = (O.bf16_bits(X).astype(np.uint32) << 16).view(np.float32), q
    buf = torch.zeros(X.size + off, dtype=Xd.dtype, device="cuda")
    buf[off:].copy_(Xd)
    X3 = X.astype(np.float64).reshape(dims, order="F")
    for mode in range(3):
        U = rng.standard_normal((dims[mode], r)).astype(np.float32)
        Ue = U if storage == tdx.TDX_F32 else (O.bf16_bits(U.ravel()).astype(np.uint32) << 16).view(np.float32).reshape(U.shape)
        ref, mag = [np.moveaxis(np.tensordot(f(X3), f(Ue.astype(np.float64)), (mode, 0)), -1, mode)
                    for f in (lambda v: v, np.abs)]
        n = X.size // dims[mode] * r
        outs = [empty(n)]
        tdx.ttm_ex(buf[off:], dims, mode, dev(U.ravel(order="F")), r, outs[0], dtype=storage)
        if storage == tdx.TDX_F32:  # the reference's layout: U is r x I, column-major
            outs.append(empty(n))
            tdx.ttm(buf[off:], dev(U.ravel()), outs[1], mode + 1, *dims, r)
        # a sum of I rounded products, in any order: (I + 2) 2^-24 of the sum of magnitudes
        bound = (dims[mode] + 2) * 2.0 ** -24 * mag + 1e-30
        for out in outs:
            got = host(out).reshape(ref.shape, order="F")
            assert np.all(np.abs(got - ref) <= bound), (dims, r, mode, float(np.max(np.abs(got - ref) / bound)))
