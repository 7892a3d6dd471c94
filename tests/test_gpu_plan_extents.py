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


@pytest.mark.parametrize("order", [(0, 1, 2), (0, 2, 1), (2, 0, 1), (1, 2, 0)])
def test_pairs_of_other_extents_into_one_block(order):
    """(2, 6 | 5) . (5 | 4) + (3, 4 | 7) . (7 | 2, 2) + (1, 12 | 3) . (3 | 4, 1): the same 12 x 4
    matrix, with the left blocks' axes stored in any order; integers, so that the sums are exact."""
    L, keep = _lib.lib(), []

    def u(x):
        keep.append(np.ascontiguousarray(x, dtype=np.uint64))
        return keep[-1].ctypes.data_as(_lib.u64p)

    def at(sizes):
        keep.append(np.concatenate([[0], np.cumsum(sizes)])[:-1].astype(np.int64))
        return keep[-1].ctypes.data_as(_lib.i64p)

    rng = np.random.default_rng(5)
    left, right = [(2, 6, 5), (3, 4, 7), (1, 12, 3)], [(5, 4, 1), (7, 2, 2), (3, 1, 4)]
    A = [rng.integers(-3, 4, s).astype(np.float64) for s in left]
    B = [rng.integers(-3, 4, s).astype(np.float64) for s in right]
    stored = [np.ascontiguousarray(x.transpose(order)) for x in A]
    # rows: the left block's free axes in the order it stores them
    want = sum(np.moveaxis(x, order.index(2), 2).reshape(12, -1) @ y.reshape(-1, 4)
               for x, y in zip(stored, B))
    itoi = np.array([[0, 0, k] for k in range(3)])[:, list(order)]
    h, ws = ctypes.c_void_p(), ctypes.c_int64()
    _lib.check(L.cxa_block_contract_plan(
        3, 3, 3, u(itoi), u([x.shape for x in stored]), at([x.size for x in A]), 3, 3,
        u([[k, 0, 0] for k in range(3)]), u(right), at([x.size for x in B]), 1,
        u([order.index(2)]), u([0]), 1, u([[0, 0, 0, 0]]), u([[2, 6, 4, 1]]), at([48]),
        ctypes.byref(h)))
    try:
        _lib.check(L.cxa_block_contract_info(h, None, ctypes.byref(ws), None))
        a, b = (torch.from_numpy(np.concatenate([x.reshape(-1) for x in t])).cuda()
                for t in (stored, B))
        c = torch.full((12, 4), np.nan, dtype=torch.float64, device="cuda")
        w = torch.empty(max(1, ws.value), dtype=torch.uint8, device="cuda")
        _lib.check(L.cxa_block_contract_exec(h, a.data_ptr(), b.data_ptr(), c.data_ptr(),
                                             w.data_ptr() if ws.value else None, 0,
                                             torch.cuda.current_stream().cuda_stream))
        assert np.array_equal(c.cpu().numpy(), want)
    finally:
        L.cxa_block_contract_destroy(h)
