"""Contractions whose operands or output are read and written through strides: axes that do not
merge into one GEMM index are taken apart into blocks and K segments, and an output stored in
another axis order is written in place, or through the workspace where it would fall into too
many pieces.  The entries are small integers, so every sum is exact in every dtype and the results
have to be equal.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

_DT = {"f64": (torch.float64, 3), "f32": (torch.float32, 4), "c128": (torch.complex128, 1),
       "c64": (torch.complex64, 2)}


def _ints(rng, shape, dt):
    x = rng.integers(-3, 4, size=shape).astype(np.float64)
    if dt.is_complex:
        x = x + 1j * rng.integers(-3, 4, size=shape)
    return torch.from_numpy(np.ascontiguousarray(x)).to(dt)


def _contract(blocks_a, blocks_b, c1, c2, dt, code, order, conj):
    """Block list x block list over common axes c1 / c2: block i of A with block i of B into
    output block i, stored in axis order `order` (None: as is)."""
    from cytnx_amd import _lib
    L = _lib.lib()
    ra, rb = blocks_a[0].dim(), blocks_b[0].dim()
    nb = len(blocks_a)
    fa = [i for i in range(ra) if i not in c1]
    fb = [i for i in range(rb) if i not in c2]
    rc = len(fa) + len(fb)
    # the block index is the quantum number of every leg
    itoi = [np.repeat(np.arange(nb, dtype=np.uint64)[:, None], r, axis=1).copy()
            for r in (ra, rb, rc)]
    shp = [np.array([x.shape for x in bl], dtype=np.uint64).reshape(nb, -1)
           for bl in (blocks_a, blocks_b)]
    shp.append(np.array([[a.shape[i] for i in fa] + [b.shape[i] for i in fb]
                         for a, b in zip(blocks_a, blocks_b)], dtype=np.uint64).reshape(nb, rc))

    def offs(shapes):
        n = [int(np.prod(s)) + 3 for s in shapes]  # gaps, at no particular alignment
        return np.array([1 + sum(n[:i]) for i in range(nb)], dtype=np.int64), 1 + sum(n)

    def pack(blocks, off, total):
        flat = torch.zeros(total, dtype=dt)
        for x, o in zip(blocks, off):
            flat[o:o + x.numel()] = x.reshape(-1)
        return flat.cuda()

    (oa, na), (ob, nb_), (oc, nc) = (offs(s) for s in shp)
    A, B = pack(blocks_a, oa, na), pack(blocks_b, ob, nb_)
    C = torch.full((nc,), 77, dtype=dt, device="cuda")
    u = lambda x: np.ascontiguousarray(x).ctypes.data_as(_lib.u64p)
    i64 = lambda x: x.ctypes.data_as(_lib.i64p)
    h = ctypes.c_void_p()
    args = (code, ra, nb, u(itoi[0]), u(shp[0]), i64(oa), rb, nb, u(itoi[1]), u(shp[1]), i64(ob),
            len(c1), _lib.u64_array(c1), _lib.u64_array(c2), nb, u(itoi[2]), u(shp[2]), i64(oc))
    if order is None:
        _lib.check(L.cxa_block_contract_plan(*args, ctypes.byref(h)))
    else:
        _lib.check(L.cxa_block_contract_plan_out(*args, _lib.u64_array(order), ctypes.byref(h)))
    try:
        ws = ctypes.c_int64(0)
        _lib.check(L.cxa_block_contract_info(h, None, ctypes.byref(ws), None))
        W = torch.empty(max(1, ws.value), dtype=torch.uint8, device="cuda")
        s = torch.cuda.current_stream().cuda_stream
        _lib.check(L.cxa_block_contract_exec_ex(h, A.data_ptr(), B.data_ptr(), C.data_ptr(),
                                                W.data_ptr(), 0, conj, s))
        torch.cuda.synchronize()
    finally:
        L.cxa_block_contract_destroy(h)
    wide = torch.complex128 if dt.is_complex else torch.float64
    want = torch.full((nc,), 77, dtype=wide)
    for a, b, o in zip(blocks_a, blocks_b, oc):
        a = (a.conj() if conj & 1 else a).to(wide)
        b = (b.conj() if conj & 2 else b).to(wide)
        t = torch.tensordot(a, b, dims=(list(c1), list(c2)))
        if order is not None:
            t = t.permute(order)
        want[o:o + t.numel()] = t.reshape(-1)
    assert torch.equal(C.cpu().to(wide), want)
    return ws.value


@pytest.mark.parametrize("name", list(_DT))
@pytest.mark.parametrize("seed", range(12))
def test_random_axis_orders(seed, name):
    dt, code = _DT[name]
    rng = np.random.default_rng(100 + seed)
    ra, rb = int(rng.integers(1, 6)), int(rng.integers(1, 6))
    ncomm = int(rng.integers(0, min(ra, rb) + 1))
    c1 = [int(x) for x in rng.permutation(ra)[:ncomm]]
    c2 = [int(x) for x in rng.permutation(rb)[:ncomm]]
    ext = [1, 2, 3, 5, 8, 17]
    ba, bb = [], []
    for _ in range(int(rng.integers(1, 4)) if ncomm else 1):
        sa = [int(rng.choice(ext)) for _ in range(ra)]
        sb = [int(rng.choice(ext)) for _ in range(rb)]
        for i, j in zip(c1, c2):
            sb[j] = sa[i]
        ba.append(_ints(rng, sa, dt))
        bb.append(_ints(rng, sb, dt))
    rc = ra + rb - 2 * ncomm
    conj = int(rng.integers(0, 4)) if dt.is_complex else 0
    _contract(ba, bb, c1, c2, dt, code, None, conj)
    if rc:
        _contract(ba, bb, c1, c2, dt, code, [int(x) for x in rng.permutation(rc)], conj)


@pytest.mark.parametrize("name", ["f64", "c128"])
def test_large_blocks_in_place(name):
    """A middle index contracted, and results in the operands' own axis order: no workspace."""
    dt, code = _DT[name]
    rng = np.random.default_rng(5)
    a, b = _ints(rng, (70, 3, 65), dt), _ints(rng, (3, 70, 2, 33), dt)
    assert _contract([a], [b], [0, 1], [1, 0], dt, code, None, 0) == 0
    assert _contract([a], [b], [0], [1], dt, code, [3, 0, 4, 2, 1], 0) == 0
    w = _ints(rng, (65, 40), dt)
    for order in ([0, 2, 1], [2, 0, 1], [1, 2, 0]):
        assert _contract([a], [w], [2], [0], dt, code, order, 0) == 0


@pytest.mark.parametrize("name", ["f64", "c128"])
def test_many_small_axes_through_the_workspace(name):
    """Axes of extent 2 in reversed order fall into more pieces than a launch should have."""
    dt, code = _DT[name]
    rng = np.random.default_rng(6)
    for nb in (1, 2):
        a = [_ints(rng, (2,) * 9, dt) for _ in range(nb)]
        b = [_ints(rng, (2,) * 9, dt) for _ in range(nb)]
        assert _contract(a, b, [4, 0], [0, 7], dt, code, list(range(13, -1, -1)), 0) > 0


def test_refused_output_axes():
    from cytnx_amd import _lib
    L = _lib.lib()
    one = np.ones((1, 2), dtype=np.uint64)
    off = np.zeros(1, dtype=np.int64)
    u, i64 = one.ctypes.data_as(_lib.u64p), off.ctypes.data_as(_lib.i64p)
    for order in ([0, 0], [0, 2]):
        h = ctypes.c_void_p()
        assert L.cxa_block_contract_plan_out(3, 2, 1, u, u, i64, 2, 1, u, u, i64, 1,
                                             _lib.u64_array([1]), _lib.u64_array([0]), 1, u, u,
                                             i64, _lib.u64_array(order), ctypes.byref(h)) != 0
        assert not h.value
