"""MTTKRP of shapes and alignments without whole vectors (odd extents, ranks above 64, tensors
off a 16-byte boundary): the FP64-accumulating kernel against the oracle, at the edges of its
row tiles (16, 32, 64, 128), K steps (64) and column blocks (16, 64), every storage and order."""
import numpy as np
import pytest

import oracle as O
import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

CASES = [((1, 1), 1), ((17, 9), 16), ((3, 129), 5), ((13, 16, 5), 17), ((33, 3, 65), 33), ((129, 5, 7), 50),
         ((7, 130, 9), 64), ((65, 64, 3), 20), ((5, 7, 3, 11), 3), ((17, 33, 6, 5), 40), ((32, 16, 8), 65),
         ((16, 20, 9), 130), ((1, 257, 1), 2), ((63, 1, 2, 31), 24), ((255, 31, 17), 16)]


def _check(dims, R, storage, off):
    import torch
    rng = np.random.default_rng(sum(dims) + 7 * R + off)
    n = int(np.prod(dims))
    X = rng.standard_normal(n).astype(np.float32)
    U = [rng.standard_normal((d, R)).astype(np.float32) for d in dims]
    Ud = [dev(u.ravel(order="F")) for u in U]
    U64 = [u.astype(np.float64) for u in U]
    Xd, sc, scales = dev(X), None, None
    if storage == tdx.TDX_BF16:
        q = torch.empty(n, dtype=torch.int16, device="cuda")
        tdx.quantize_bf16(Xd, q)
        X = (O.bf16_bits(X).astype(np.uint32) << 16).view(np.float32)
        Xd = q
    elif storage == tdx.TDX_FP8_E4M3:
        q, sc = torch.empty(n, dtype=torch.uint8, device="cuda"), empty(dims[0])
        tdx.quantize_fp8_mode1(Xd, q, sc, dims[0])
        codes, scales = O.quantize_e4m3_mode1(X, dims[0])
        X, Xd = O.e4m3_decode(codes), q
    buf = torch.zeros(n + off, dtype=Xd.dtype, device="cuda")
    buf[off:].copy_(Xd)
    A64 = [np.abs(u) for u in U64]
    for mode in range(len(dims)):
        out = empty(dims[mode] * R)
        out.fill_(float("nan"))
        tdx.mttkrp_ex(buf[off:], storage, sc, dims, Ud, R, mode, out)
        got = host(out).reshape((dims[mode], R), order="F")
        ref = O.mttkrp(X, dims, U64, mode, scales=scales)
        # FP32 roundings on a term's way: the Khatri-Rao products (2), the slice scale (1), the
        # split's partial (1), the result (1); one more for the slack of the products of them
        bound = 6 * 2.0 ** -24 * O.mttkrp(np.abs(X), dims, A64, mode, scales=scales) + 1e-30
        assert np.all(np.abs(got - ref) <= bound), (dims, R, mode, float(np.max(np.abs(got - ref) / bound)))


@pytest.mark.parametrize("storage", [tdx.TDX_F32, tdx.TDX_BF16, tdx.TDX_FP8_E4M3], ids=["f32", "bf16", "fp8"])
@pytest.mark.parametrize("dims,R", CASES)
def test_any_shape_against_fp64(dims, R, storage):
    _check(dims, R, storage, 0)


@pytest.mark.parametrize("storage", [tdx.TDX_F32, tdx.TDX_BF16, tdx.TDX_FP8_E4M3], ids=["f32", "bf16", "fp8"])
def test_any_alignment_against_fp64(storage):
    _check((64, 32, 48), 16, storage, 1)
