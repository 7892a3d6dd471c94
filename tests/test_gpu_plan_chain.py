"""A contraction plan that was not made for a chain, used in one: the chain runs what it runs with a
plan made for it, and executions of the plan by itself, captured ones too, stay as they were."""
import ctypes

import pytest
import torch

from cytnx_amd import _lib
from cytnx_amd.heff import _Chain, _Flat, strided_batch_plan

pytestmark = pytest.mark.gpu

M = N = K = 256  # by itself 256 tiles of 16 x 16, as a step of a chain 64 of 32 x 32


def _plan(chain):
    return strided_batch_plan(1, M, N, K, (0, K, 1), (0, N, 1), (0, N), 3, chain=chain)


def _exec(plan, x, b, c, prec=0):
    _lib.check(_lib.lib().cxa_block_contract_exec(plan.handle, x.data_ptr(), b._storage.data_ptr(),
                                                  c.data_ptr(), None, prec,
                                                  torch.cuda.current_stream().cuda_stream))


def _tiles(plan, prec=0):
    n = ctypes.c_int()
    _lib.check(_lib.lib().cxa_block_contract_get_config(plan.handle, prec, None, None,
                                                        ctypes.byref(n)))
    return n.value


def _chain_result(plan, b, x, prec):
    chain = _Chain([(plan, b, False, M * N)], 0)
    chain.prepare(prec)
    y = torch.empty(M * N, dtype=torch.float64, device="cuda")
    chain.apply(x, y)
    torch.cuda.synchronize()
    return y, chain


def _inputs():
    x = torch.randn(M * K, dtype=torch.float64, device="cuda")
    return x, _Flat(torch.randn(K * N, dtype=torch.float64, device="cuda"))


def test_own_executions_are_unchanged():
    x, b = _inputs()
    plan, own = _plan(False), torch.empty(M * N, dtype=torch.float64, device="cuda")
    _exec(plan, x, b, own)
    tiles = _tiles(plan)
    assert tiles == 256
    captured = torch.empty_like(own)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _exec(plan, x, b, captured)
    want, _keep = _chain_result(_plan(True), b, x, 0)
    got, _keep2 = _chain_result(plan, b, x, 0)
    assert torch.equal(got, want)
    assert _tiles(plan) == tiles
    for seed in range(3):
        x.copy_(torch.randn(M * K, dtype=torch.float64, device="cuda"))
        _exec(plan, x, b, own)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, own)


@pytest.mark.parametrize("prec", [0, 1])
def test_chain_results_do_not_depend_on_earlier_executions(prec):
    x, b = _inputs()
    plan, own = _plan(False), torch.empty(M * N, dtype=torch.float64, device="cuda")
    _exec(plan, x, b, own, prec)
    want, _keep = _chain_result(_plan(True), b, x, prec)
    got, _keep2 = _chain_result(plan, b, x, prec)
    assert torch.equal(got, want)
