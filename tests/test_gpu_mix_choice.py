"""The tiles that a mix launch takes by itself, at sizes on both sides of its limit of 2400 tiles of
16 x 16."""
import pytest
import torch

from cytnx_amd.heff import Heff2
from cytnx_amd.heisenberg import two_site_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("chi", [1448, 2048])
def test_same_bits_as_the_smallest_tiles(chi, precision):
    """1722 and 3035 tiles: every slice's K is summed front to back by one wave and the slices in a
    fixed order, so the matvec is the same bits in tiles of any size."""
    parts = [t.to(0) for t in two_site_problem(chi, seed=31, hermitian=True)]
    H, x = Heff2(*parts), parts[0].storage()
    assert len(H.chain.steps) == 2
    auto = {"kind": -1, "split": -1}
    got, want = torch.empty_like(x), torch.empty_like(x)
    H.set_precision(precision)
    print("mix choice", chi, precision, flush=True)
    H.apply_flat(x, got)
    H.set_tiles([{"kind": 0, "split": 0}, auto])
    H.apply_flat(x, want)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert float(torch.linalg.vector_norm(want)) > 0
