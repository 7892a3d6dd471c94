"""Row tiles of blocks with N <= 8: one and four rows per lane at the edges of their tiles, K and N, with
rows of C that touch and that do not.  The entries are small integers, so every sum is exact and
the results have to be equal."""
import pytest
import torch

from cytnx_amd import _lib
from cytnx_amd.heff import strided_batch_plan

pytestmark = pytest.mark.gpu


def _ints(shape, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-3, 4, shape, generator=g, device="cuda").to(dt)


@pytest.mark.parametrize("ident", [3, 4])
@pytest.mark.parametrize("nb,M", [(520, 255), (520, 256), (520, 257), (3, 257), (1, 131072), (1, 131071),
                                  (2100, 64)])
def test_rows(ident, nb, M):
    """520 blocks of about 256 rows hold as many rows as four per lane are taken from."""
    dt = {3: torch.float64, 4: torch.float32}[ident]
    s = torch.cuda.current_stream().cuda_stream
    for N, K in ((1, 1), (1, 4), (3, 3), (4, 7), (4, 8), (4, 9), (4, 33), (5, 5), (8, 2), (2, 0)):
        for gap in (0, 3):
            print("rows", ident, nb, M, N, K, gap, flush=True)
            a, b = _ints((nb, M, K), dt, 1), _ints((nb, K, N), dt, 2)
            c = torch.full((nb, M, N + gap), 9, dtype=dt, device="cuda")
            plan = strided_batch_plan(nb, M, N, K, (M * K, K, 1), (K * N, N, 1),
                                      (M * (N + gap), N + gap), ident)
            _lib.check(_lib.lib().cxa_block_contract_exec(
                plan.handle, (a if K else c).data_ptr(), (b if K else c).data_ptr(), c.data_ptr(),
                None, 0, s))
            want = torch.full((nb, M, N + gap), 9, dtype=torch.float64, device="cuda")
            want[:, :, :N] = a.double() @ b.double()
            assert torch.equal(c.double(), want)
