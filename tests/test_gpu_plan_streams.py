"""One cached plan executed on two streams at once, its operands or its output staged in scratch:
every result equals the one of an execution by itself."""
import pytest
import torch

from cytnx_amd import autograd, unitensor
from cytnx_amd.unitensor import BD_BRA, BD_KET, Bond, Contract, UniTensor

pytestmark = pytest.mark.gpu


def _tensor(kinds, labels, ext, seed):
    T = UniTensor([Bond(k, [[0]], [ext]) for k in kinds], labels, 1, 3, 0)
    g = torch.Generator(device="cuda").manual_seed(seed)
    T.storage().copy_(torch.randn(T.storage().numel(), generator=g, dtype=torch.float64,
                                  device="cuda"))
    return T


def _operands(seed, ext=16):
    # the contracted legs of A lie between its free ones, so the gradient of A falls into more
    # pieces than are written in place
    A = _tensor((BD_KET, BD_KET, BD_KET, BD_KET), ["c1", "f1", "c2", "f2"], ext, seed)
    B = _tensor((BD_BRA, BD_BRA, BD_BRA), ["c1", "c2", "f"], ext, seed + 100)
    return A, B


def _gradients(A, B):
    for T in (A, B):
        T._storage = T.storage().detach().requires_grad_(True)
    C = autograd.contract_ad(A, B)
    (C.storage() * C.storage()).sum().backward()
    return C.storage().detach(), A.storage().grad, B.storage().grad


def test_gradients_on_two_streams():
    autograd._SPECS.clear()
    autograd._OUTS.clear()
    inputs = [_operands(s) for s in (1, 2)]
    want = [_gradients(A, B) for A, B in inputs]
    assert any(sp.ga.ws_bytes > 0 for sp in autograd._SPECS.values())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for _ in range(20):
        for s, (A, B) in zip(streams, inputs):
            with torch.cuda.stream(s):
                got.append(_gradients(A, B))
    torch.cuda.synchronize()
    for i, g in enumerate(got):
        for x, y in zip(g, want[i % 2]):
            assert torch.equal(x, y)


def test_contractions_on_two_streams():
    # axes of extent 2 in reversed order: operands that are permuted into scratch
    labels = ["x%d" % i for i in range(9)]
    inputs = []
    for seed in (3, 4):
        A = _tensor((BD_KET,) * 9, labels, 2, seed)
        B = _tensor((BD_BRA,) * 5 + (BD_KET,) * 4, labels[8::-2] + ["y%d" % i for i in range(4)],
                    2, seed + 100)
        inputs.append((A, B))
    unitensor._PLAN_CACHE.clear()
    want = [Contract(A, B).storage() for A, B in inputs]
    assert any(p.ws_bytes > 0 for p in unitensor._PLAN_CACHE.values())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for _ in range(20):
        for s, (A, B) in zip(streams, inputs):
            with torch.cuda.stream(s):
                got.append(Contract(A, B).storage())
    torch.cuda.synchronize()
    for i, g in enumerate(got):
        assert torch.equal(g, want[i % 2])
