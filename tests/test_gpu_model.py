"""Reconstruction, residual and rse at the edges of the model kernel (64-row blocks, 16-row tiles,
16-fibre blocks, 4 fibre blocks a wave, rank blocks 16/32/48/64 and above) and of the vector loads
(tensors off a 16-byte boundary, lengths that are no multiple of 4), against FP64."""
import numpy as np
import pytest

import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 1), ((16, 3, 5), 4), ((17, 16, 1), 16), ((63, 5, 13), 17), ((65, 1, 67), 33), ((128, 31, 7), 48),
         ((130, 17, 9), 64), ((40, 33, 3), 65), ((7, 20, 11), 200), ((5, 3, 7, 11), 6), ((64, 2, 16, 5), 50),
         ((33, 65, 1, 2), 20)]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("dims,R", CASES)
def test_model_and_errors_against_fp64(dims, R, off):
    import torch
    rng = np.random.default_rng(sum(dims) + R)
    U = [rng.standard_normal((d, R)).astype(np.float32) for d in dims]
    sub = "abcd"[:len(dims)]
    spec = ",".join(c + "r" for c in sub) + "->" + sub
    ref = np.einsum(spec, *[u.astype(np.float64) for u in U]).ravel(order="F")
    mag = np.einsum(spec, *[np.abs(u).astype(np.float64) for u in U]).ravel(order="F")
    Ud = [dev(u.ravel(order="F")) for u in U]
    buf = torch.full((ref.size + off,), float("nan"), device="cuda")
    rec = buf[off:]
    (tdx.gencp if len(dims) == 3 else tdx.gencp4)(rec, *Ud, *dims, R)
    # R terms of (order - 1) products, rounded, and their sum in any order
    assert np.all(np.abs(host(rec) - ref) <= (R + 4) * 2.0 ** -24 * mag + 1e-30)
    X = (ref + 0.1 * rng.standard_normal(ref.size) * max(1e-3, np.std(ref))).astype(np.float32)
    xb = torch.zeros(ref.size + off, device="cuda")
    xb[off:].copy_(dev(X))
    X64, rec64 = X.astype(np.float64), host(rec).astype(np.float64)
    nx = np.linalg.norm(X64)
    # the sums are FP64 of the FP32 values: rse is exact to its FP32 result's rounding
    assert abs(tdx.rse(xb[off:], rec, ref.size) - np.linalg.norm(X64 - rec64) / nx) <= 1e-7 * (
        np.linalg.norm(X64 - rec64) / nx) + 1e-30
    got = tdx.cp_relerr(xb[off:], dims, Ud, R)
    want = np.linalg.norm(X64 - ref) / nx
    # the model entries' FP32 rounding, at most as large as the bound above in norm
    assert abs(got - want) <= np.linalg.norm((R + 4) * 2.0 ** -24 * mag) / nx + 1e-12
