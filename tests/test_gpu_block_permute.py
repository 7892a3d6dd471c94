"""Batched block permutes: blocks of one element to more than the batched launch takes, innermost
axis kept or moved, odd extents and unaligned offsets, against torch's permute (bytes equal)."""
import ctypes

import numpy as np
import pytest
import torch

from cytnx_amd import _lib

pytestmark = pytest.mark.gpu

DTYPES = {3: torch.float64, 4: torch.float32, 1: torch.complex128}
BLOCKS = {
    2: [(1, 1), (3, 5), (1, 40), (33, 65), (200, 170), (64, 512), (1100, 1000)],
    3: [(1, 1, 1), (3, 163, 163), (150, 2, 131), (7, 1, 9), (65, 33, 17), (2, 2, 2)],
    4: [(3, 2, 5, 7), (1, 31, 1, 33), (40, 3, 40, 2), (16, 16, 16, 16), (2, 99, 2, 101)],
    6: [(2, 3, 2, 5, 3, 2), (4, 4, 4, 4, 4, 4), (1, 9, 1, 8, 1, 7)],
}


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("rank", sorted(BLOCKS))
def test_blocks(rank, ident):
    L, rng, dt = _lib.lib(), np.random.default_rng(rank), DTYPES[ident]
    orders = [list(range(rank))[::-1], list(range(1, rank)) + [0],
              [1, 0] + list(range(2, rank))] + [list(rng.permutation(rank)) for _ in range(3)]
    shapes = np.array(BLOCKS[rank], dtype=np.uint64)
    sizes = [int(np.prod(s)) for s in BLOCKS[rank]]
    so = np.array([3 + sum(sizes[:i]) + i for i in range(len(sizes))], dtype=np.int64)
    do = np.array([1 + sum(sizes[:i]) + 2 * i for i in range(len(sizes))], dtype=np.int64)
    src = torch.randn(int(so[-1]) + sizes[-1], dtype=dt, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    for order in orders:
        print("block permute", rank, ident, order, flush=True)
        h = ctypes.c_void_p()
        _lib.check(L.cxa_block_permute_plan(
            ident, rank, len(sizes), shapes.ctypes.data_as(_lib.u64p), so.ctypes.data_as(_lib.i64p),
            do.ctypes.data_as(_lib.i64p), _lib.u64_array([int(x) for x in order]),
            ctypes.byref(h)))
        try:
            dst = torch.full((int(do[-1]) + sizes[-1] + 1,), 5, dtype=dt, device="cuda")
            want = dst.clone()
            _lib.check(L.cxa_block_permute_exec(h, src.data_ptr(), dst.data_ptr(), s))
            torch.cuda.synchronize()
        finally:
            L.cxa_block_permute_destroy(h)
        for shp, n, a, b in zip(BLOCKS[rank], sizes, so, do):
            want[b:b + n] = src[a:a + n].view(shp).permute([int(x) for x in order]).reshape(-1)
        assert torch.equal(dst, want)


@pytest.mark.parametrize("ident", sorted(DTYPES))
def test_output_run_cuts(ident):
    """Output runs around the tile heights they are cut at, alone and inside outer axes."""
    from cytnx_amd.tensor import Tensor
    for h in (31, 33, 119, 120, 121, 127, 128, 129, 136, 200, 255, 257, 300):
        for shape, order in (((h, 40), (1, 0)), ((3, h, 2, 17), (3, 0, 2, 1)), ((h, 5, 9), (2, 1, 0))):
            x = torch.randn(shape, dtype=DTYPES[ident], device="cuda")
            got = Tensor.from_storage(x.reshape(-1), shape).permute(*order).contiguous()
            assert torch.equal(got.storage(), x.permute(order).reshape(-1))
