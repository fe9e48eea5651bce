"""Split opening sweeps through the shared pass with FP32 T, with BF16 sweeps behind them: against FP64,
and against the separate passes, whose bits differ where the shared pass was really taken."""
import pytest
import torch

import tdx
from test_gpu_als_wide import setup, sweep64

pytestmark = pytest.mark.gpu

DIMS = (520, 400, 330)  # BF16 sweeps of this shape have no shared pass: their A is not rounded as a whole


def run(X, R, F, opening, sweeps, shared=1):
    U = [f.clone() for f in F]
    o = tdx.default_cp_options()
    o.init, o.max_sweeps, o.storage, o.shared_pass = 1, sweeps, tdx.TDX_BF16, shared
    o.opening_sweeps, o.opening_split, o.refine_sweeps = opening, 1, 0
    st, rep, _, _ = tdx.cp_als_ex(X, DIMS, R, U, o)
    assert st == tdx.TDX_OK and rep.sweeps_done == sweeps
    return U


@pytest.mark.parametrize("R", [64, 24])
def test_opening_and_bf16_sweep(R):
    X, F = setup(DIMS, R, 7 + R)
    opening, both = run(X, R, F, 1, 1), run(X, R, F, 1, 2)
    separate = run(X, R, F, 1, 1, shared=0)
    assert any(not torch.equal(a, b) for a, b in zip(opening, separate))
    ref, scale = sweep64(X.bfloat16(), DIMS, F)
    for m in range(3):  # coefficients of 17 bits, two a term, and what a mode's error does to the next
        assert float((opening[m].double() - ref[m]).norm() / scale[m].norm()) <= (m + 1) * 2.0 ** -15, m
        assert float((separate[m].double() - ref[m]).norm() / scale[m].norm()) <= (m + 1) * 2.0 ** -15, m
    ref, scale = sweep64(X.bfloat16(), DIMS, [r.float() for r in ref])
    for m in range(3):  # a Khatri-Rao entry rounded to 8 bits: 2^-9 of a term
        assert float((both[m].double() - ref[m]).norm() / scale[m].norm()) <= (m + 1) * 2.0 ** -9, m
