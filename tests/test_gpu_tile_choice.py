"""Tiles chosen by size: skinny, short-K and ragged products of every type against 64-bit products, at
the edges of the choice (numbers of tiles, chunks of K, the area that tiles cover), alone and in
lists.  The entries are small integers, so every sum is exact and the results have to be equal."""
import pytest
import torch

from cytnx_amd import _lib, linalg
from cytnx_amd.heff import strided_batch_plan
from cytnx_amd.tensor import Tensor

pytestmark = pytest.mark.gpu

DTYPES = {3: torch.float64, 4: torch.float32, 1: torch.complex128, 2: torch.complex64}


def _ints(shape, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-3, 4, shape, generator=g, device="cuda").to(torch.float64)
    if dt.is_complex:
        x = torch.complex(x, torch.randint(-3, 4, shape, generator=g, device="cuda")
                          .to(torch.float64))
    return x.to(dt)


def _product(a, b):
    wide = torch.complex128 if a.is_complex() else torch.float64
    return a.to(wide) @ b.to(wide)


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("M,K,N", [(20000, 33, 10), (20000, 112, 10), (20000, 113, 10), (10, 208, 9000),
                                   (10, 209, 9000), (3000, 1, 70), (3000, 17, 66), (1000, 112, 1000),
                                   (1000, 113, 1000), (767, 50, 33), (1500, 300, 66), (260, 200, 520)])
def test_products(ident, M, K, N):
    dt = DTYPES[ident]
    print("product", ident, M, K, N, flush=True)
    a, b = _ints((M, K), dt, 1), _ints((K, N), dt, 2)
    out = linalg.Matmul(Tensor.from_storage(a.reshape(-1), [M, K]),
                        Tensor.from_storage(b.reshape(-1), [K, N]))
    want = _product(a, b)
    assert torch.equal(out.storage().view(M, N).to(want.dtype), want)


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("nb,M,N,K", [(200, 70, 10, 33), (200, 70, 8, 112), (30, 200, 66, 113),
                                      (40, 160, 160, 17), (40, 160, 160, 130), (300, 20, 20, 209),
                                      (3, 500, 500, 48)])
def test_lists(ident, nb, M, N, K):
    dt = DTYPES[ident]
    print("list", ident, nb, M, N, K, flush=True)
    s = torch.cuda.current_stream().cuda_stream
    a, b = _ints((nb, M, K), dt, 3), _ints((nb, K, N), dt, 4)
    want = _product(a, b)
    for a_cols, b_cols in ((False, False), (True, False), (False, True)):
        A = a.transpose(1, 2).contiguous() if a_cols else a
        B = b.transpose(1, 2).contiguous() if b_cols else b
        c = torch.full((nb, M, N), 9, dtype=dt, device="cuda")
        plan = strided_batch_plan(nb, M, N, K, (M * K, 1, M) if a_cols else (M * K, K, 1),
                                  (K * N, 1, K) if b_cols else (K * N, N, 1), (M * N, N), ident)
        _lib.check(_lib.lib().cxa_block_contract_exec(plan.handle, A.data_ptr(), B.data_ptr(),
                                                      c.data_ptr(), None, 0, s))
        assert torch.equal(c.to(want.dtype), want)


@pytest.mark.parametrize("ident", sorted(DTYPES))
def test_values_beside_the_block_are_not_read_into_it(ident):
    """Infinities and NaN next to a block's rows, columns and K, read by no tile: those of the
    direct tiles, with wide loads, and of the tiles staged through LDS."""
    dt, (M, N, K, pad) = DTYPES[ident], (37, 35, 53, 11)
    s = torch.cuda.current_stream().cuda_stream
    a = torch.full((M + pad, K + pad), float("nan"), dtype=dt, device="cuda")
    b = torch.full((K + pad, N + pad), float("inf"), dtype=dt, device="cuda")
    a[:M, :K], b[:K, :N] = _ints((M, K), dt, 5), _ints((K, N), dt, 6)
    want = _product(a[:M, :K], b[:K, :N])
    plan = strided_batch_plan(1, M, N, K, (0, K + pad, 1), (0, N + pad, 1), (0, N), ident)
    for kind, split in ((-1, -1), (0, 0), (0, 1), (1, 0), (1, 1), (6, 0), (7, 0)):
        print("beside", ident, kind, split, flush=True)
        _lib.check(_lib.lib().cxa_block_contract_set_config(plan.handle, -1, kind, split))
        c = torch.full((M, N), 9, dtype=dt, device="cuda")
        _lib.check(_lib.lib().cxa_block_contract_exec(plan.handle, a.data_ptr(), b.data_ptr(),
                                                      c.data_ptr(), None, 0, s))
        assert torch.equal(c.to(want.dtype), want)
