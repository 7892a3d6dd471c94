"""Operands and outputs of a block contraction that go through its workspace: blocks above the size
that the batched permute takes (2^20 elements), alone and beside smaller ones.  Integer entries, so
every sum is exact."""
import numpy as np
import pytest

pytest.importorskip("torch")
from test_gpu_contract_strides import _DT, _contract, _ints  # noqa: E402

pytestmark = pytest.mark.gpu


def _blocks(rng, last, lead, dt):
    return [_ints(rng, (2,) * lead + (n,), dt) for n in last]


@pytest.mark.parametrize("name", ["f64", "c64"])
@pytest.mark.parametrize("last", [(2100,), (2100, 5, 3)])
def test_operands_above_the_batched_size(name, last):
    """Five contracted axes in reversed order between the free ones: A is copied first."""
    dt, code = _DT[name]
    rng = np.random.default_rng(8)
    a = _blocks(rng, last, 9, dt)
    b = [_ints(rng, (2,) * 5 + (3,), dt) for _ in last]
    assert a[0].numel() > 1 << 20
    assert _contract(a, b, [8, 6, 4, 2, 0], [0, 1, 2, 3, 4], dt, code, None, 0) >= \
        a[0].numel() * a[0].element_size()


@pytest.mark.parametrize("name", ["f64", "c128"])
@pytest.mark.parametrize("last", [(2100,), (2100, 5, 3)])
def test_outputs_above_the_batched_size(name, last):
    """An output stored with its axes reversed falls into more pieces than are written in place."""
    dt, code = _DT[name]
    rng = np.random.default_rng(9)
    a = _blocks(rng, last, 9, dt)
    b = [_ints(rng, (2,) * 5, dt) for _ in last]
    n = 2 ** 7 * last[0] * 2 ** 3
    assert n > 1 << 20
    assert _contract(a, b, [4, 0], [0, 3], dt, code, list(range(10, -1, -1)), 0) >= \
        n * a[0].element_size()
