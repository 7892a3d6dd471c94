"""K ranges of the direct MFMA tiles: numbers of 16-deep chunks around the loads in flight, over
one and several segments and waves, empty segments, and strides too large for 32-bit offsets.  The
entries are small integers, so every sum is exact and the results have to be equal."""
import ctypes

import numpy as np
import pytest
import torch

from cytnx_amd import _lib
from cytnx_amd.heff import strided_batch_plan

pytestmark = pytest.mark.gpu

DTYPES = {3: torch.float64, 4: torch.float32, 1: torch.complex128, 2: torch.complex64}


def _ints(shape, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-3, 4, shape, generator=g, device="cuda").to(torch.float64)
    if dt.is_complex:
        x = torch.complex(x, torch.randint(-3, 4, shape, generator=g, device="cuda")
                          .to(torch.float64))
    return x.to(dt)


def _exec(handle, a, b, c):
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib().cxa_block_contract_exec(handle, a.data_ptr(), b.data_ptr(),
                                                  c.data_ptr(), None, 0, s))
    torch.cuda.synchronize()


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("kind,split", [(0, 0), (0, 1), (0, 2), (1, 0), (1, 1), (2, 0), (3, 1),
                                        (4, 0)])
def test_segments_and_chunks(ident, kind, split):
    dt, L = DTYPES[ident], _lib.lib()
    M, N = 37, 35
    for ks in ([1], [16], [33], [64], [65], [81], [200], [3, 40], [0, 17, 0, 50], [16, 16, 16, 1],
               [130, 5, 70], [0]):
        nb = len(ks)
        print("kind", kind, split, ident, ks, flush=True)
        # blocks (i | common i) of A and (common i | 0) of B meet in the one output block
        ua = np.array([[0, i] for i in range(nb)], dtype=np.uint64)
        ub = np.array([[i, 0] for i in range(nb)], dtype=np.uint64)
        sa = np.array([[M, k] for k in ks], dtype=np.uint64)
        sb = np.array([[k, N] for k in ks], dtype=np.uint64)
        oa = np.cumsum([0] + [M * k for k in ks])[:nb].astype(np.int64)
        ob = np.cumsum([0] + [N * k for k in ks])[:nb].astype(np.int64)
        uc, sc, oc = np.zeros((1, 2), np.uint64), np.array([[M, N]], np.uint64), np.zeros(1, np.int64)
        u = lambda x: x.ctypes.data_as(_lib.u64p)
        i64 = lambda x: x.ctypes.data_as(_lib.i64p)
        h = ctypes.c_void_p()
        _lib.check(L.cxa_block_contract_plan(ident, 2, nb, u(ua), u(sa), i64(oa), 2, nb, u(ub),
                                             u(sb), i64(ob), 1, _lib.u64_array([1]),
                                             _lib.u64_array([0]), 1, u(uc), u(sc), i64(oc),
                                             ctypes.byref(h)))
        try:
            assert L.cxa_block_contract_set_config(h, -1, kind, split) == 0
            a, b = _ints((sum(ks) * M + 1,), dt, 1), _ints((sum(ks) * N + 1,), dt, 2)
            c = torch.full((M, N), 9, dtype=dt, device="cuda")
            _exec(h, a, b, c)
        finally:
            L.cxa_block_contract_destroy(h)
        wide = torch.complex128 if dt.is_complex else torch.float64
        a, b = a.cpu().to(wide), b.cpu().to(wide)
        want = torch.zeros(M, N, dtype=wide)
        for k, o, q in zip(ks, oa, ob):
            want += a[o:o + M * k].view(M, k) @ b[q:q + N * k].view(k, N)
        assert torch.equal(c.cpu().to(wide), want)


@pytest.mark.parametrize("ident", [3, 2])
@pytest.mark.parametrize("kind,split", [(0, 0), (0, 1), (1, 0)])
def test_wide_strides(ident, kind, split):
    """Rows 2^21 + 1 elements apart: no 32-bit offsets within a tile."""
    dt = DTYPES[ident]
    M, N, K, st = 19, 21, 50, (1 << 21) + 1
    a = torch.zeros(M * st, dtype=dt, device="cuda")
    av = a.view(M, st)[:, :K]
    av.copy_(_ints((M, K), dt, 3))
    b = _ints((K, N), dt, 4)
    c = torch.full((M, N), 9, dtype=dt, device="cuda")
    p = strided_batch_plan(1, M, N, K, (0, st, 1), (0, N, 1), (0, N), ident)
    assert _lib.lib().cxa_block_contract_set_config(p.handle, -1, kind, split) == 0
    _exec(p.handle, a, b, c)
    wide = torch.complex128 if dt.is_complex else torch.float64
    assert torch.equal(c.cpu().to(wide), av.cpu().to(wide) @ b.cpu().to(wide))


@pytest.mark.parametrize("split", [0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_mix_chunks(kind, split):
    """Slices of every number of chunks around the loads in flight, one with wide strides."""
    L, M, N = _lib.lib(), 20, 18
    for ks, st in (([1, 16, 17, 48, 64, 65, 130, 0], 0), ([70], 0), ([5, 90, 3], (1 << 21) + 1)):
        print("mix", kind, split, ks, st, flush=True)
        b = _ints((sum(ks), N), torch.float64, 6)
        a = torch.zeros(M * st if st else M * sum(ks), dtype=torch.float64, device="cuda")
        a.view(M, -1)[:, :sum(ks)].copy_(_ints((M, sum(ks)), torch.float64, 5))
        ld = a.numel() // M
        at = np.cumsum([0] + ks)
        sl = np.array([[at[i], at[i] * N, ld, 1, N, 1, k] for i, k in enumerate(ks)], np.int64)
        coef = np.zeros((2, 8))
        coef[:, :len(ks)] = np.arange(1, 2 * len(ks) + 1).reshape(2, -1)
        items = np.array([[M, N, len(ks), 2]], np.int64)
        outs = np.array([[0, N], [M * N, N]], np.int64)
        i64 = lambda x: x.ctypes.data_as(_lib.i64p)
        h = ctypes.c_void_p()
        _lib.check(L.cxa_mix_contract_plan(3, 1, i64(items), len(ks), i64(sl), 2, i64(outs),
                                           coef.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                           ctypes.byref(h)))
        try:
            assert L.cxa_block_contract_set_config(h, -1, kind, split) == 0
            c = torch.full((2, M, N), 9.0, dtype=torch.float64, device="cuda")
            _exec(h, a, b, c)
        finally:
            L.cxa_block_contract_destroy(h)
        A, B = a.view(M, -1)[:, :sum(ks)].cpu(), b.cpu()
        X = [A[:, at[i]:at[i + 1]] @ B[at[i]:at[i + 1]] for i in range(len(ks))]
        for o in range(2):
            want = sum(coef[o, i] * X[i] for i in range(len(ks)))
            assert torch.equal(c[o].cpu(), want)
