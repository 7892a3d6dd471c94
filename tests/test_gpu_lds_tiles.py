"""Tiles staged through LDS where a plan uses them: blocks of several K segments, k4-packed operands and
the dot-product epilogue of a fused Lanczos iteration."""
import ctypes

import numpy as np
import pytest
import torch

from cytnx_amd import _lib
from cytnx_amd.heff import Heff2
from cytnx_amd.heisenberg import two_site_problem
from cytnx_amd.lanczos import lanczos_gnd_native

pytestmark = pytest.mark.gpu

DTYPES = {3: torch.float64, 4: torch.float32, 1: torch.complex128, 2: torch.complex64}


def _ints(n, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-3, 4, (n,), generator=g, device="cuda").to(torch.float64)
    if dt.is_complex:
        x = torch.complex(x, torch.randint(-3, 4, (n,), generator=g, device="cuda")
                          .to(torch.float64))
    return x.to(dt)


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("kind", [6, 7])
def test_segments(ident, kind):
    """Chunks that end with a segment, empty segments first, between and last, and single values of
    K; integer entries, so that every sum is exact."""
    dt, L = DTYPES[ident], _lib.lib()
    M, N = 70, 67
    for ks in ([1], [64, 64], [65, 63, 1], [0, 17, 0, 50], [16, 0], [0, 0, 128, 3], [130, 5, 70],
               [1] * 9, [33] * 7, [200, 200], [0]):
        nb = len(ks)
        print("segments", ident, kind, ks, flush=True)
        u = lambda x: np.ascontiguousarray(x, dtype=np.uint64).ctypes.data_as(_lib.u64p)
        keep = [np.array([[0, i] for i in range(nb)], np.uint64),
                np.array([[M, k] for k in ks], np.uint64),
                np.array([[i, 0] for i in range(nb)], np.uint64),
                np.array([[k, N] for k in ks], np.uint64),
                np.zeros((1, 2), np.uint64), np.array([[M, N]], np.uint64)]
        at = np.concatenate([[0], np.cumsum(ks)]).astype(np.int64)
        oa, ob, oc = at[:-1] * M, at[:-1] * N, np.zeros(1, np.int64)
        i64 = lambda x: x.ctypes.data_as(_lib.i64p)
        p = [x.ctypes.data_as(_lib.u64p) for x in keep]
        h = ctypes.c_void_p()
        _lib.check(L.cxa_block_contract_plan(
            ident, 2, nb, p[0], p[1], i64(oa), 2, nb, p[2], p[3], i64(ob), 1, u([1]), u([0]), 1, p[4],
            p[5], i64(oc), ctypes.byref(h)))
        try:
            assert L.cxa_block_contract_set_config(h, -1, kind, 0) == 0
            a, b = _ints(sum(ks) * M + 1, dt, 1), _ints(sum(ks) * N + 1, dt, 2)
            c = torch.full((M, N), 9, dtype=dt, device="cuda")
            _lib.check(L.cxa_block_contract_exec(h, a.data_ptr(), b.data_ptr(), c.data_ptr(), None, 0,
                                                 torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
        finally:
            L.cxa_block_contract_destroy(h)
        wide = torch.complex128 if dt.is_complex else torch.float64
        a, b, want = a.cpu().to(wide), b.cpu().to(wide), torch.zeros(M, N, dtype=wide)
        for k, x, y in zip(ks, oa, ob):
            want += a[x:x + M * k].view(M, k) @ b[y:y + N * k].view(k, N)
        assert torch.equal(c.cpu().to(wide), want)


def _operator(chi):
    parts = [t.to(0) for t in two_site_problem(chi, seed=29, hermitian=True)]
    return Heff2(*parts), parts[0].storage()


def _with_last_step(H, kind, split, run):
    H.set_tiles([{"kind": -1, "split": -1}] * (len(H.chain.steps) - 1) + [{"kind": kind, "split": split}])
    try:
        return run()
    finally:
        H.set_tiles([{"kind": -1, "split": -1}] * len(H.chain.steps))


def test_packed_last_step_of_an_fp32_operator():
    """The .R step reads its fixed operand k4-packed: both LDS kinds against FP64, at the level of
    error that the FP32 arithmetic has (5e-6)."""
    H, x = _operator(256)
    want, got = torch.empty_like(x), torch.empty_like(x)
    H.apply_flat(x, want)
    H.set_precision(1)
    try:
        assert H.chain.layout(len(H.chain.steps) - 1) & 1
        for kind in (6, 7):
            print("packed R step", kind, flush=True)
            _with_last_step(H, kind, 0, lambda: H.apply_flat(x, got))
            assert float(torch.linalg.vector_norm(got - want)) <= \
                5e-6 * float(torch.linalg.vector_norm(want))
    finally:
        H.set_precision(0)


def test_dot_epilogue_of_a_fused_fp32_iteration():
    """Alphas and betas of the first iterations with the last step in each LDS kind and in direct
    tiles: both are FP32 matvecs off by at most 5e-6 of the operator's norm, and the Lanczos
    coefficients are off by as much (twice, from two of them)."""
    H, x = _operator(192)
    H.set_precision(1)
    try:
        run = lambda: [np.asarray(v) for v in lanczos_gnd_native(H, x, 1e-30, 6, batch=3)[3:5]]
        a0, b0 = _with_last_step(H, 1, 0, run)
        scale = float(np.abs(a0).max() + np.abs(b0).max())
        for kind in (6, 7):
            print("fused iteration", kind, flush=True)
            a, b = _with_last_step(H, kind, 0, run)
            n = min(len(a), len(a0), 6)
            assert n == 6
            assert np.abs(a[:n] - a0[:n]).max() <= 1e-5 * scale
            assert np.abs(b[:n - 1] - b0[:n - 1]).max() <= 1e-5 * scale
    finally:
        H.set_precision(0)
