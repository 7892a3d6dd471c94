"""How block contractions sum K: lists of few tiles and long K in several partial sums, and narrow
FP32 blocks (N <= 8) in FP64."""
import pytest
import torch

from cytnx_amd import _lib, linalg
from cytnx_amd.heff import strided_batch_plan
from cytnx_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


def _rand(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(n, generator=g, dtype=torch.float32, device="cuda")


def _exec(plan, a, b, c):
    _lib.check(_lib.lib().cxa_block_contract_exec(
        plan.handle, a.data_ptr(), b.data_ptr(), c.data_ptr(), None, 0,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


@pytest.mark.parametrize("ident,nb,M,N,K", [
    (4, 60, 160, 160, 400), (4, 20, 200, 140, 256), (4, 60, 300, 300, 300), (4, 30, 100, 100, 200),
    (3, 60, 160, 160, 400), (3, 20, 200, 140, 256), (3, 40, 300, 40, 500), (3, 30, 100, 100, 200)])
def test_partial_sums_of_long_k(ident, nb, M, N, K):
    """The first and the last product of K are big and -big, the others 1/4: a sum that holds big
    loses every quarter added to it (half its last place is 4, an MFMA adds four of them, 1),
    and one that does not loses none.  Four partial sums, the large products in two of them at most,
    lose at most half of the quarters and a chunk's; a single one loses all."""
    print("partial sums", ident, nb, M, N, K, flush=True)
    dt, big = {3: (torch.float64, 2.0 ** 55), 4: (torch.float32, 2.0 ** 26)}[ident]
    a = torch.full((nb, M, K), 0.25, dtype=dt, device="cuda")
    a[:, :, 0], a[:, :, K - 1] = big, -big
    b = torch.ones((nb, K, N), dtype=dt, device="cuda")
    c = torch.zeros((nb, M, N), dtype=dt, device="cuda")
    _exec(strided_batch_plan(nb, M, N, K, (M * K, K, 1), (K * N, N, 1), (M * N, N), ident), a, b, c)
    want = 0.25 * (K - 2)
    assert float((c - want).abs().max()) <= 0.25 * (K / 2 + 64)


@pytest.mark.parametrize("nb,M,N,K", [(30, 64, 6, 2000), (1, 1, 1, 100000), (4, 16, 8, 10000),
                                      (50, 100, 1, 500), (20, 200, 6, 33)])
def test_narrow_blocks_sum_in_fp64(nb, M, N, K):
    """Products and sums of FP32 inputs in FP64: the result is off by its own rounding, 2^-24 of it,
    and 2 K eps64 of the summed magnitudes."""
    print("narrow", nb, M, N, K, flush=True)
    a, b = _rand(nb * M * K, 1).view(nb, M, K), _rand(nb * K * N, 2).view(nb, K, N)
    want = torch.bmm(a.double(), b.double())
    bound = want.abs() * 2.0 ** -24 + 2 * K * 2.0 ** -53 * torch.bmm(a.double().abs(), b.double().abs())
    c = torch.zeros((nb, M, N), dtype=torch.float32, device="cuda")
    _exec(strided_batch_plan(nb, M, N, K, (M * K, K, 1), (K * N, N, 1), (M * N, N), 4), a, b, c)
    assert bool(((c.double() - want).abs() <= bound).all())
    A = [Tensor.from_storage(x.reshape(-1).clone(), [M, K]) for x in a]
    B = [Tensor.from_storage(x.reshape(-1).clone(), [K, N]) for x in b]
    C = [Tensor([M, N], 4, 0) for _ in range(nb)]
    linalg.Gemm_Batch([1.0], A, B, [0.0], C, [nb])
    got = torch.stack([x.storage().view(M, N) for x in C]).double()
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("nb,M,N,K", [(1, 100, 75, 133), (3, 64, 64, 1000), (2, 33, 17, 16), (1, 40, 70, 65)])
def test_fp32_lds_tiles_sum_as_the_split_does(nb, M, N, K):
    """LDS tiles of both sizes: the bits of 16 x 16 tiles whose K is split over four waves."""
    print("lds and split", nb, M, N, K, flush=True)
    a, b = _rand(nb * M * K, 3), _rand(nb * K * N, 4)
    plan = strided_batch_plan(nb, M, N, K, (M * K, K, 1), (K * N, N, 1), (M * N, N), 4)
    got = []
    for kind, split in ((0, 1), (6, 0), (7, 0)):
        c = torch.zeros(nb * M * N, dtype=torch.float32, device="cuda")
        _lib.check(_lib.lib().cxa_block_contract_set_config(plan.handle, -1, kind, split))
        _exec(plan, a, b, c)
        got.append(c)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
