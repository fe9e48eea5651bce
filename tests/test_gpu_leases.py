"""Device memory and streams that calls hold: sizes going up and down, a release in between, several
threads at once, and a call that fails leave every result as it is on fresh memory, bit for bit; what
stays idle is bounded and given back."""
import ctypes
import threading

import numpy as np
import pytest

import tdx
from helpers import dev, empty, host

pytestmark = pytest.mark.gpu

SHAPES = [((96, 80, 64), (12, 10, 8)), ((17, 9, 11), (3, 4, 5)), ((40, 30, 20, 12), (6, 5, 4, 3)), ((64, 64, 64), (16, 16, 16))]


def tucker(k, iters=1):
    dims, ranks = SHAPES[k]
    rng = np.random.default_rng(k)
    G = rng.standard_normal(ranks)
    for m, (d, r) in enumerate(zip(dims, ranks)):
        G = np.moveaxis(np.tensordot(rng.standard_normal((d, r)), G, axes=(1, m)), 0, m)
    X = G.astype(np.float32).ravel(order="F")
    core, U = empty(int(np.prod(ranks))), [empty(d * r) for d, r in zip(dims, ranks)]
    tdx.tucker_hooi(dev(X), dims, ranks, iters, core, U)
    return [host(core)] + [host(u) for u in U]


def batched(k):
    rng = np.random.default_rng(100 + k)
    dims = rng.integers(4, 40, (30 + k, 3))
    ranks = rng.integers(1, 9, 30 + k)
    xo = np.concatenate([[0], np.cumsum(dims.prod(1))])
    X = rng.standard_normal(int(xo[-1])).astype(np.float32)
    n = (dims * ranks[:, None]).ravel()
    uo = np.concatenate([[0], np.cumsum(n)])
    U = rng.standard_normal(int(uo[-1])).astype(np.float32)
    Xd, Ud = dev(X), dev(U)
    L = ctypes.c_long
    arr = lambda a: (L * len(a))(*[int(v) for v in a])
    f = tdx.lib().tdx_cp_als_batched
    st = f(ctypes.c_void_p(Xd.data_ptr()), ctypes.c_void_p(Ud.data_ptr()), arr(dims.ravel()), arr(ranks), arr(xo[:-1]),
           arr(uo[:-1]), L(30 + k), 2, 1, ctypes.c_uint64(0), -1, None, None)
    assert st in (0, tdx.TDX_WARN_SINGULAR)
    return [host(Ud)]


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.fixture(scope="module")
def fresh():
    out = {}
    for k in range(4):
        tdx.lib().tdx_release_workspace()
        out[k] = tucker(k)
        tdx.lib().tdx_release_workspace()
        out[10 + k] = batched(k)
    return out


def test_sizes_up_and_down(fresh):
    for k in (0, 1, 2, 3, 1, 0, 3, 2):
        assert same(tucker(k), fresh[k]), k
        assert same(batched(k), fresh[10 + k]), k


def test_threads(fresh):
    bad = []

    def work(i):
        for j in range(6):
            k = (i + j) % 4
            if not same(tucker(k) if i % 2 else batched(k), fresh[k if i % 2 else 10 + k]):
                bad.append((i, k))
            if i == 0 and j == 3:
                tdx.lib().tdx_release_workspace()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_failure_and_release(fresh):
    import torch
    core, U = empty(8), [empty(8)] * 3
    with pytest.raises(Exception):
        tdx.tucker_hooi(dev(np.ones(600 * 4, np.float32)), (600, 2, 2), (2, 2, 2), 1, core, U)
    assert same(tucker(0), fresh[0])
    tdx.lib().tdx_release_workspace()
    free0 = torch.cuda.mem_get_info()[0]
    for k in range(4):
        tucker(k)
        batched(k)
    assert free0 - torch.cuda.mem_get_info()[0] <= 2 << 30
    tdx.lib().tdx_release_workspace()
    assert free0 - torch.cuda.mem_get_info()[0] <= 64 << 20
