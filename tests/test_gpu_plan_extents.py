"""Output extents of a block contraction plan that are not those of its operands' legs."""
import ctypes

import numpy as np
import pytest
import torch

from cytnx_amd import _lib

pytestmark = pytest.mark.gpu


def _plan(out_shape, out_axes=None):
    """A (2, 6 | 5) . B (5 | 4), one block each, into a block of extents out_shape."""
    L, keep = _lib.lib(), []

    def u(x):
        keep.append(np.ascontiguousarray(x, dtype=np.uint64))
        return keep[-1].ctypes.data_as(_lib.u64p)

    off = np.zeros(1, dtype=np.int64)
    o = off.ctypes.data_as(_lib.i64p)
    h = ctypes.c_void_p()
    args = (3, 3, 1, u([[0, 0, 0]]), u([[2, 6, 5]]), o, 2, 1, u([[0, 0]]), u([[5, 4]]), o, 1, u([2]),
            u([0]), 1, u([[0, 0, 0]]), u([out_shape]), o)
    rc = L.cxa_block_contract_plan(*args, ctypes.byref(h)) if out_axes is None else \
        L.cxa_block_contract_plan_out(*args, u(out_axes), ctypes.byref(h))
    return rc, h


def test_regrouped_rows_are_the_same_matrix():
    a = torch.randn(12, 5, dtype=torch.float64, device="cuda")
    b = torch.randn(5, 4, dtype=torch.float64, device="cuda")
    for shape in ([2, 6, 4], [3, 4, 4], [12, 1, 4]):
        rc, h = _plan(shape)
        assert rc == 0
        try:
            c = torch.full((12, 4), np.nan, dtype=torch.float64, device="cuda")
            _lib.check(_lib.lib().cxa_block_contract_exec(
                h, a.data_ptr(), b.data_ptr(), c.data_ptr(), None, 0,
                torch.cuda.current_stream().cuda_stream))
            assert float((c - a @ b).abs().max()) <= 1e-14
        finally:
            _lib.lib().cxa_block_contract_destroy(h)


def test_refused_extents():
    for shape, axes in (([2, 5, 4], None), ([2, 6, 3], None), ([3, 4, 4], [2, 0, 1])):
        rc, h = _plan(shape, axes)
        assert rc != 0 and not h.value
