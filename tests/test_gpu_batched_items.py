"""Batched CP-ALS with work items (the default design) at the edges of its row groups (16, 32,
64, 128), column steps (16), slice runs (4) and T widths (4, 8, 16): every sweep's relative error
against the FP64 oracle's, tensor by tensor, and against the one-kernel design."""
import numpy as np
import pytest

import oracle as O
import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

SHAPES = [(1, 17, 5), (3, 5, 4), (4, 4, 4), (15, 16, 1), (16, 1, 33), (17, 15, 3), (31, 33, 6), (32, 16, 16),
          (33, 2, 9), (63, 17, 5), (64, 64, 7), (65, 31, 4), (97, 5, 40), (127, 9, 13), (128, 16, 5), (20, 128, 6),
          (9, 7, 128), (128, 128, 128)]


def test_items_against_fp64_at_the_edges():
    rng = np.random.default_rng(5)
    ranks = [min(r, max(1, sorted(s)[1] - 1)) for s, r in zip(SHAPES, [2, 3, 1, 4, 2, 5, 8, 16, 2, 9, 16, 12, 4, 8, 3,
                                                                     6, 5, 16])]
    b = tdx.Batch(SHAPES, ranks)
    X, U0 = np.empty(b.x_floats, np.float32), np.empty(b.u_floats, np.float32)
    init = []
    for t, (dims, R) in enumerate(zip(SHAPES, ranks)):
        F = [rng.uniform(0.1, 1.0, (d, R)) for d in dims]
        Xt = np.einsum("ar,br,cr->abc", *F).ravel(order="F")
        Xt = Xt + 0.05 * np.linalg.norm(Xt) / np.sqrt(Xt.size) * rng.standard_normal(Xt.size)
        X[b.xoff[t]:b.xoff[t] + Xt.size] = Xt
        init.append([(f * rng.uniform(0.8, 1.25, f.shape)).astype(np.float32) for f in F])
        for m, f in enumerate(init[t]):
            o = int(b.uoff[3 * t + m])
            U0[o:o + f.size] = f.ravel(order="F")
    fits = {}
    for v in (-1, 0):
        U = dev(U0)
        st, fits[v], _ = tdx.cp_als_batched(dev(X), U, b, 4, init=1, variant=v)
        assert st == tdx.TDX_OK
    # relerr is about 0.05: an error of e relative to ||X||^2 in its square moves it by 10 e, and
    # FP32 sums over up to 2^21 products keep e below 2e-6
    assert np.max(np.abs(fits[-1] - fits[0])) < 2e-5
    for t, dims in enumerate(SHAPES):
        n = int(np.prod(dims))
        _, _, dr, _ = O.cp_als(X[b.xoff[t]:b.xoff[t] + n], dims, [u.astype(np.float64) for u in init[t]], 4,
                               direct=True)
        assert np.max(np.abs(fits[-1][t] - dr)) < 2e-5, (t, dims, ranks[t])
