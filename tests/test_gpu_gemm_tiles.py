"""GEMM tile kinds at the edges of their tiles, K chunks and operand orders, against a 64-bit
product: the 64x64 and 32x32 tiles staged through LDS, the 16x16 tiles whose K is split over the
waves of a workgroup, and the tiling the library picks by itself."""
import pytest
import torch

from cytnx_amd import _lib, linalg
from cytnx_amd.heff import strided_batch_plan
from cytnx_amd.tensor import Tensor

pytestmark = pytest.mark.gpu

DTYPES = {3: torch.float64, 4: torch.float32, 1: torch.complex128, 2: torch.complex64}
EPS = {3: 2.0 ** -53, 4: 2.0 ** -24, 1: 2.0 ** -53, 2: 2.0 ** -24}


def _rand(n, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.complex128 if dt.is_complex else torch.float64
    return torch.randn(n, generator=g, dtype=wide, device="cuda").to(dt)


def _check(got, A, B, ident):
    """Each element within its summation bound: K products and K sums, each off by at most eps of
    |A| |B| (complex: four real products), plus the final rounding."""
    wide = torch.complex128 if A.is_complex() else torch.float64
    A, B = A.to(wide), B.to(wide)
    bound = (2 * A.shape[-1] + 4) * EPS[ident] * (A.abs() @ B.abs())
    if A.is_complex():
        bound = 2 * bound
    assert bool(((got.to(wide) - A @ B).abs() <= bound).all())


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("kind,split", [(6, 0), (7, 0), (0, 1), (0, 2), (-1, -1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 17, 15), (31, 33, 16), (32, 32, 64), (33, 65, 17),
                                   (64, 64, 128), (65, 31, 129), (130, 97, 200), (5, 300, 33),
                                   (300, 5, 31), (40, 40, 0)])
def test_tile_kinds(ident, kind, split, M, N, K):
    dt = DTYPES[ident]
    print("tile kind", kind, split, ident, M, N, K, flush=True)
    s = torch.cuda.current_stream().cuda_stream
    for a_cols, b_cols in ((False, False), (True, False), (False, True), (True, True)):
        nb = 2
        a, b = _rand(max(1, nb * M * K), dt, 1), _rand(max(1, nb * K * N), dt, 2)
        c = torch.full((nb * M * N,), 7.0, dtype=dt, device="cuda")
        sa = (M * K, 1, M) if a_cols else (M * K, K, 1)
        sb = (K * N, 1, K) if b_cols else (K * N, N, 1)
        plan = strided_batch_plan(nb, M, N, K, sa, sb, (M * N, N), ident)
        rc = _lib.lib().cxa_block_contract_set_config(plan.handle, -1, kind, split)
        assert rc == 0
        _lib.check(_lib.lib().cxa_block_contract_exec(plan.handle, a.data_ptr(), b.data_ptr(),
                                                      c.data_ptr(), None, 0, s))
        for i in range(nb):
            av, bv = a[i * M * K:(i + 1) * M * K], b[i * K * N:(i + 1) * K * N]
            A = av.view(K, M).t() if a_cols else av.view(M, K)
            B = bv.view(N, K).t() if b_cols else bv.view(K, N)
            _check(c[i * M * N:(i + 1) * M * N].view(M, N), A, B, ident)


@pytest.mark.parametrize("ident", sorted(DTYPES))
@pytest.mark.parametrize("M,K,N", [(16, 4096, 16), (250, 40, 260), (257, 33, 256), (40, 900, 700),
                                   (900, 65, 900), (1000, 32, 40), (1000, 10, 10)])
def test_matmul_of_every_tiling(ident, M, K, N):
    dt = DTYPES[ident]
    print("matmul", ident, M, K, N, flush=True)
    a, b = _rand(M * K, dt, 3), _rand(K * N, dt, 4)
    out = linalg.Matmul(Tensor.from_storage(a, [M, K]), Tensor.from_storage(b, [K, N]))
    _check(out.storage().view(M, N), a.view(M, K), b.view(K, N), ident)


def test_lds_and_direct_tiles_agree_bitwise():
    """FP64 and complex tiles sum K in one order whether they are staged through LDS or not."""
    for ident in (3, 1, 2):
        dt, (M, N, K) = DTYPES[ident], (100, 75, 133)
        a, b = _rand(M * K, dt, 5), _rand(K * N, dt, 6)
        plan = strided_batch_plan(1, M, N, K, (0, K, 1), (0, N, 1), (0, N), ident)
        got = []
        for kind in (0, 6, 7):
            c = torch.empty(M * N, dtype=dt, device="cuda")
            _lib.check(_lib.lib().cxa_block_contract_set_config(plan.handle, -1, kind, 0))
            _lib.check(_lib.lib().cxa_block_contract_exec(
                plan.handle, a.data_ptr(), b.data_ptr(), c.data_ptr(), None, 0,
                torch.cuda.current_stream().cuda_stream))
            got.append(c)
        assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
