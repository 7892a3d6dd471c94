"""Timed cases of the contraction path: the calls a tensor-network program makes of this package.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges, ``prepare`` makes
what a program holds before the call (tensors, planned operators), ``run`` is one pass through
the public entry points, ``work`` what that pass cannot do without, and ``exact`` the same result
from plain torch in 64 bits.

Kinds:

* ``permute``       ``Tensor.permute(...).contiguous()``: leg reorderings of dense tensors.
* ``matmul``        ``linalg.Matmul`` of two rank-2 tensors.
* ``dense_chain``   the three dense ``Contract`` calls L.A.W.R of a one-site update.
* ``gemm_batch``    ``linalg.Gemm_Batch``: many small matrices of differing sizes in groups.
* ``env``           ``dmrg.left_env_step``: the environment update of a U(1) DMRG sweep, three
                    block contractions and a block permute.
* ``heff2``         the U(1) two-site effective Hamiltonian applied to a vector (``Heff2``).
* ``lanczos2``      a DMRG bond's eigensolve: 30 Lanczos iterations of that operator.
* ``lanczos1``      the same for a dense one-site operator (``Heff1Dense``).
* ``mps_gradient``  energy of a U(1) MPS and its gradient with respect to every site tensor.

Values are iid normal numbers scaled so that results stay of order one, as random states and
environments are.  Sector sizes follow a Gaussian in the charge, as those of a spin chain's ground
state do.
"""
import math

import numpy as np
import torch

from cytnx_amd import heisenberg, linalg
from cytnx_amd.dmrg import left_env_step
from cytnx_amd.heff import Heff1Dense, Heff2
from cytnx_amd.mps import mps_energy
from cytnx_amd.tensor import Tensor
from cytnx_amd.unitensor import BD_BRA, BD_KET, Bond, Contract, UniTensor

DEV = 0
DTYPES = {"c128": (1, torch.complex128, 16), "c64": (2, torch.complex64, 8),
          "f64": (3, torch.float64, 8), "f32": (4, torch.float32, 4)}
PRECISIONS = {"fp64": 0, "fp32": 1}
ITERATIONS = 30       # Lanczos iterations of one bond update
TUNE_ELEMS = 1 << 17  # operators a DMRG run tunes (dmrg.DMRG.TUNE_MIN_ELEMS)


# ---------------------------------------------------------------------------------- cases
def listed():
    return [
        # legs of a small one-site tensor brought into order: a launch, hardly any data
        {"name": "permute_small", "kind": "permute", "shape": "24,2,5,24", "perm": "2,0,3,1",
         "dtype": "f64"},
        # one permutation of the rank-6 sweep of the benchmark (16 MiB)
        {"name": "permute_rank6", "kind": "permute", "shape": "16,8,16,8,16,8",
         "perm": "4,1,5,0,3,2", "dtype": "f64"},
        # legs of a large dense environment reversed, ragged extents (84 MB)
        {"name": "permute_large", "kind": "permute", "shape": "1021,5,1027", "perm": "2,1,0",
         "dtype": "c128"},
        # a large dense product, no dimension a multiple of a tile
        {"name": "matmul_large", "kind": "matmul", "m": 2000, "k": 1801, "n": 2107,
         "dtype": "f64"},
        # a dense one-site update in complex arithmetic (time evolution)
        {"name": "dense_chain", "kind": "dense_chain", "chi": 192, "dtype": "c128"},
        # sector matrices of a large two-site state (up to 458 rows) multiplied in one call
        {"name": "gemm_batch", "kind": "gemm_batch", "groups": 12, "per_group": 5, "top": 458,
         "dtype": "f32"},
        # the environment update of a DMRG sweep at the bond dimension of the large DMRG runs
        {"name": "env_update", "kind": "env", "chi": 2048, "dtype": "f64"},
        # a small operator: two launches and little work
        {"name": "heff2_small", "kind": "heff2", "chi": 128, "precision": "fp64"},
        # the bond dimension of the large DMRG runs, contractions in FP32
        {"name": "heff2_large", "kind": "heff2", "chi": 2048, "precision": "fp32"},
        # one bond update's eigensolve at the bond dimension of the headline
        {"name": "lanczos_two_site", "kind": "lanczos2", "chi": 1024},
        # the dense one-site eigensolve at chi=128
        {"name": "lanczos_one_site", "kind": "lanczos1", "chi": 128},
        # differentiable energy of a 32-site MPS: forward and backward
        {"name": "mps_gradient", "kind": "mps_gradient", "sites": 32, "chi": 512,
         "dtype": "c128"},
    ]


def _spread(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["permute", "matmul", "dense_chain", "gemm_batch", "env", "heff2",
                       "lanczos2", "lanczos1", "mps_gradient"])
    if kind == "permute":
        rank = rng.randint(3, 6)
        total = _spread(rng, 1 << 12, 5 << 20)
        shape, left = [], total
        for axis in range(rank):
            mean = left ** (1.0 / (rank - axis))
            e = max(2, int(mean * rng.uniform(0.4, 1.6)))
            shape.append(e)
            left = max(1.0, left / e)
        perm = list(range(rank))
        while perm == sorted(perm):
            rng.shuffle(perm)
        return {"kind": kind, "shape": ",".join(map(str, shape)),
                "perm": ",".join(map(str, perm)), "dtype": rng.choice(["f32", "f64", "c128"])}
    if kind == "matmul":
        return {"kind": kind, "m": _spread(rng, 40, 1600), "k": _spread(rng, 40, 1600),
                "n": _spread(rng, 40, 1600), "dtype": rng.choice(["f64", "f32", "c64", "c128"])}
    if kind == "dense_chain":
        return {"kind": kind, "chi": _spread(rng, 24, 192), "dtype": rng.choice(["f64", "c128"])}
    if kind == "gemm_batch":
        return {"kind": kind, "groups": rng.randint(1, 16), "per_group": rng.randint(1, 6),
                "top": _spread(rng, 20, 458), "dtype": rng.choice(["f32", "f64", "c128"])}
    if kind == "env":
        return {"kind": kind, "chi": _spread(rng, 48, 2048), "dtype": rng.choice(["f64", "c128"])}
    if kind == "heff2":
        return {"kind": kind, "chi": _spread(rng, 64, 2048),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "lanczos2":
        return {"kind": kind, "chi": _spread(rng, 64, 1024)}
    if kind == "lanczos1":
        return {"kind": kind, "chi": _spread(rng, 24, 160)}
    return {"kind": kind, "sites": 2 * rng.randint(4, 16), "chi": _spread(rng, 32, 512),
            "dtype": rng.choice(["c128", "c64", "f64"])}


# ---------------------------------------------------------------------------------- inputs
class _Values:
    """Normal numbers on the device, from the seed alone, in the order they are asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda:%d" % DEV)
        self.gen.manual_seed(int(seed))

    def __call__(self, n, dtype, scale=1.0):
        real = torch.float64 if dtype in (torch.float64, torch.complex128) else torch.float32
        k = 2 if dtype.is_complex else 1
        x = torch.randn(n * k, generator=self.gen, dtype=real, device=self.gen.device) * scale
        return torch.view_as_complex(x.view(-1, 2)) if k == 2 else x


def _ints(text):
    return [int(x) for x in text.split(",")]


def _gaussian(chi, parity=None, most=20):
    """Charges and sector sizes of a bond of chi states, Gaussian in the charge."""
    qs = [q for q in range(-most, most + 1) if parity is None or (q - parity) % 2 == 0]
    w = [math.exp(-q * q / 50.0) for q in qs]
    ideal = [chi * x / sum(w) for x in w]
    size = [int(x) for x in ideal]
    for i in sorted(range(len(qs)), key=lambda i: size[i] - ideal[i])[:chi - sum(size)]:
        size[i] += 1
    return ([q for q, d in zip(qs, size) if d > 0], [d for d in size if d > 0])


# a leg is (sign, charges, sizes): sign -1 for a KET, +1 for a BRA; a block is stored when the
# signed charges of its sectors add up to zero, the last leg's sector running fastest
PHYS = ([1, -1], [1, 1])
MPO_Q = ([0, 2, -2], [3, 1, 1])


def _bond(leg):
    return Bond(BD_KET if leg[0] < 0 else BD_BRA, leg[1], leg[2])


def _blocks(legs):
    """(slices into the dense tensor, extents, offset) of every stored block, and the total."""
    found, at = [], 0
    starts = [np.concatenate([[0], np.cumsum(l[2])]).astype(int) for l in legs]
    last = {q: i for i, q in enumerate(legs[-1][1])}
    stack = [[]]
    for leg in legs[:-1]:
        stack = [t + [i] for t in stack for i in range(len(leg[1]))]
    for t in stack:
        q = sum(leg[0] * leg[1][i] for leg, i in zip(legs, t))
        i = last.get(-q * legs[-1][0])
        if i is None:
            continue
        idx = t + [i]
        shape = [int(leg[2][j]) for leg, j in zip(legs, idx)]
        found.append((tuple(slice(int(s[j]), int(s[j + 1])) for s, j in zip(starts, idx)),
                      shape, at))
        at += int(np.prod(shape))
    return found, at


def _dense(flat, legs):
    out = torch.zeros([int(sum(l[2])) for l in legs], dtype=flat.dtype, device=flat.device)
    for sl, shape, at in _blocks(legs)[0]:
        out[sl] = flat[at:at + int(np.prod(shape))].view(shape)
    return out


def _flat(dense, legs):
    return torch.cat([dense[sl].reshape(-1) for sl, _, _ in _blocks(legs)[0]])


def _unitensor(flat, legs, labels, rowrank, dtype):
    T = UniTensor([_bond(l) for l in legs], labels, rowrank, DTYPES[dtype][0], DEV)
    T.storage().copy_(flat)
    return T


def _mpo_dense():
    """The Heisenberg MPO W[w, w', s, s'] with its bond states in charge groups (0, +2, -2)."""
    eye, sz = np.eye(2), np.diag([0.5, -0.5])
    sp = np.array([[0.0, 1.0], [0.0, 0.0]])
    W = np.zeros((5, 5, 2, 2))
    for (a, b), o in {(0, 0): eye, (1, 0): sp, (2, 0): sp.T, (3, 0): sz, (4, 1): 0.5 * sp.T,
                      (4, 2): 0.5 * sp, (4, 3): sz, (4, 4): eye}.items():
        W[a, b] = o.T
    order = [0, 3, 4, 1, 2]
    return torch.from_numpy(W[np.ix_(order, order, [0, 1], [0, 1])].copy()).to("cuda:%d" % DEV)


def _legs_two_site(chi):
    vq, vd = _gaussian(chi)
    psi = [(-1, vq, vd), (1,) + PHYS, (1,) + PHYS, (1, vq, vd)]
    left = [(1,) + MPO_Q, (1, vq, vd), (-1, vq, vd)]
    right = [(-1,) + MPO_Q, (-1, vq, vd), (1, vq, vd)]
    return psi, left, right


def _two_site_values(case, seed, symmetric):
    """(psi, L, R) flat, with the environments symmetrised when the operator must be."""
    rnd, legs = _Values(seed), _legs_two_site(case["chi"])
    psi, left, right = (rnd(_blocks(l)[1], torch.float64, case["chi"] ** -0.5) for l in legs)
    if symmetric:  # E[w, a, b] + E[w', b, a], w' the MPO state of the adjoint operator
        for l, e in ((legs[1], left), (legs[2], right)):
            d = _dense(e, l)
            e.copy_(_flat(d + d[[0, 1, 2, 4, 3]].transpose(1, 2), l))
        psi /= torch.linalg.vector_norm(psi)
    return legs, psi, left, right


def _legs_env(chi):
    vq, vd = _gaussian(chi)
    return ([(1,) + MPO_Q, (1, vq, vd), (-1, vq, vd)],           # L (w, a, a')
            [(-1, vq, vd), (1,) + PHYS, (1, vq, vd)])            # A (a, s, b)


def _mps_legs(sites, chi):
    """Site legs (a, s, b) of an MPS of total charge 0 with bonds of at most about chi states."""
    bonds = []
    for k in range(sites + 1):
        qs = [q for q in range(-k, k + 1, 2) if abs(q) <= sites - k]
        most = [min(math.comb(k, (k + q) // 2), math.comb(sites - k, (sites - k - q) // 2))
                for q in qs]
        if sum(most) > chi:
            gq, gd = _gaussian(chi, parity=k % 2)
            have = dict(zip(gq, gd))
            most = [min(m, have.get(q, 0)) for q, m in zip(qs, most)]
        bonds.append(([q for q, d in zip(qs, most) if d], [d for d in most if d]))
    return [[(1,) + bonds[k], (1,) + PHYS, (-1,) + bonds[k + 1]] for k in range(sites)]


def _mps_values(case, seed):
    rnd, legs = _Values(seed), _mps_legs(case["sites"], case["chi"])
    return legs, [rnd(_blocks(l)[1], DTYPES[case["dtype"]][1], (2.0 * sum(l[0][2])) ** -0.5)
                  for l in legs]


def _one_site_values(chi, seed, dtype, symmetric):
    rnd = _Values(seed)
    L = rnd(chi * 5 * chi, dtype, chi ** -0.5).view(chi, 5, chi)
    A = rnd(chi * 2 * chi, dtype, chi ** -0.5).view(chi, 2, chi)
    R = rnd(chi * 5 * chi, dtype, chi ** -0.5).view(chi, 5, chi)
    if symmetric:
        adj = [0, 1, 2, 4, 3]
        L, R = (e + e[:, adj].permute(2, 1, 0) for e in (L, R))
        A = A / torch.linalg.vector_norm(A)
    return L.contiguous(), A.contiguous(), R.contiguous()


def _batch_shapes(case):
    """(M, K, N) of every group: sizes of ragged sectors up to `top`."""
    g, top = case["groups"], case["top"]
    return [(max(3, top - (7 * i) % top), max(3, top - (11 * i + 3) % top),
             max(3, top - (5 * i + 1) % top)) for i in range(g)]


# ---------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    torch.cuda.set_device(DEV)
    kind = case["kind"]
    if kind == "permute":
        shape = _ints(case["shape"])
        x = _Values(seed)(int(np.prod(shape)), DTYPES[case["dtype"]][1])
        return {"kind": kind, "x": Tensor.from_storage(x, shape), "perm": _ints(case["perm"])}
    if kind == "matmul":
        rnd, dt = _Values(seed), DTYPES[case["dtype"]][1]
        m, k, n = case["m"], case["k"], case["n"]
        return {"kind": kind, "a": Tensor.from_storage(rnd(m * k, dt, k ** -0.5), [m, k]),
                "b": Tensor.from_storage(rnd(k * n, dt), [k, n])}
    if kind == "dense_chain":
        chi, (ident, dt, _) = case["chi"], DTYPES[case["dtype"]]
        L, A, R = _one_site_values(chi, seed, dt, False)
        W = _mpo_dense().to(dt)

        def dense(t, labels):
            T = UniTensor([Bond(int(d)) for d in t.shape], labels, 1, ident, DEV)
            T.storage().copy_(t.reshape(-1))
            return T
        return {"kind": kind, "L": dense(L, ["l", "w", "l'"]), "A": dense(A, ["l", "s", "r"]),
                "W": dense(W, ["w", "w'", "s", "s'"]), "R": dense(R, ["r", "w'", "r'"])}
    if kind == "gemm_batch":
        rnd, (ident, dt, _) = _Values(seed), DTYPES[case["dtype"]]
        a, b, c = [], [], []
        for m, k, n in _batch_shapes(case):
            for _ in range(case["per_group"]):
                a.append(Tensor.from_storage(rnd(m * k, dt, k ** -0.5), [m, k]))
                b.append(Tensor.from_storage(rnd(k * n, dt), [k, n]))
                c.append(Tensor([m, n], ident, DEV))
        g = case["groups"]
        return {"kind": kind, "a": a, "b": b, "c": c, "one": [1.0] * g, "zero": [0.0] * g,
                "sizes": [case["per_group"]] * g}
    if kind == "env":
        rnd, (ident, dt, _) = _Values(seed), DTYPES[case["dtype"]]
        lleg, aleg = _legs_env(case["chi"])
        L = rnd(_blocks(lleg)[1], dt, case["chi"] ** -0.5)
        A = rnd(_blocks(aleg)[1], dt, case["chi"] ** -0.5)
        return {"kind": kind, "L": _unitensor(L, lleg, ["w", "a", "b"], 1, case["dtype"]),
                "A": _unitensor(A, aleg, ["a", "s", "c"], 2, case["dtype"]),
                "M": heisenberg.xxz_mpo_block(device=DEV).astype(ident)}
    if kind in ("heff2", "lanczos2"):
        legs, psi, left, right = _two_site_values(case, seed, kind == "lanczos2")
        M = heisenberg.xxz_mpo_block(device=DEV)
        H = Heff2(_unitensor(psi, legs[0], ["-1", "-2", "-3", "-4"], 1, "f64"),
                  _unitensor(left, legs[1], ["-5", "-1", "0"], 1, "f64"),
                  M.relabel(["-5", "-6", "-2", "1"]), M.relabel(["-6", "-7", "-3", "2"]),
                  _unitensor(right, legs[2], ["-7", "-4", "3"], 2, "f64"))
        H.set_precision(PRECISIONS[case.get("precision", "fp64")])
        if kind == "lanczos2" and H.nx() >= TUNE_ELEMS:
            H.tune(5)
        return {"kind": kind, "H": H, "x": psi, "y": torch.empty_like(psi),
                "single": case.get("precision") == "fp32"}
    if kind == "lanczos1":
        L, A, R = _one_site_values(case["chi"], seed, torch.float64, True)
        return {"kind": kind, "H": Heff1Dense(L, _mpo_dense(), R, A.shape), "x": A.reshape(-1)}
    legs, flats = _mps_values(case, seed)
    sites = [_unitensor(f, l, ["a%d" % k, "s%d" % k, "a%d" % (k + 1)], 2, case["dtype"])
             for k, (f, l) in enumerate(zip(flats, legs))]
    for A in sites:
        A.storage().requires_grad_(True)
    return {"kind": kind, "sites": sites}


# ---------------------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "permute":
        return state["x"].permute(state["perm"]).contiguous().storage()
    if kind == "matmul":
        return linalg.Matmul(state["a"], state["b"]).storage()
    if kind == "dense_chain":
        return Contract(Contract(Contract(state["L"], state["A"]), state["W"]),
                        state["R"]).storage()
    if kind == "gemm_batch":
        linalg.Gemm_Batch(state["one"], state["a"], state["b"], state["zero"], state["c"],
                          state["sizes"])
        return torch.cat([c.storage() for c in state["c"]])
    if kind == "env":
        return left_env_step(state["L"], state["A"], state["M"]).storage()
    if kind == "heff2":
        state["H"].apply_flat(state["x"], state["y"])
        # a program that contracts in FP32 keeps the result as precise as it is
        return state["y"].float() if state["single"] else state["y"]
    if kind in ("lanczos2", "lanczos1"):
        E, vec, _, alphas, betas = state["H"].ground_state(state["x"], 1e-14, ITERATIONS)
        return {"E": E, "vec": vec, "alphas": alphas, "betas": betas[:-1]}
    for A in state["sites"]:
        A.storage().grad = None
    E, _, _ = mps_energy(state["sites"])
    E.backward()
    return {"E": E.detach(), "grad": [A.storage().grad for A in state["sites"]]}


# ---------------------------------------------------------------------------------- work
def _pair_flops(legs_a, legs_b, axes_a, axes_b):
    """2 M N K summed over the block pairs of the contraction over the legs axes_a / axes_b."""
    blocks_b = {}
    for sl, shape, _ in _blocks(legs_b)[0]:
        key = tuple((sl[j].start, sl[j].stop) for j in axes_b)
        n = int(np.prod([d for j, d in enumerate(shape) if j not in axes_b]))
        blocks_b[key] = blocks_b.get(key, 0) + n
    total = 0
    for sl, shape, _ in _blocks(legs_a)[0]:
        key = tuple((sl[j].start, sl[j].stop) for j in axes_a)
        total += 2 * int(np.prod(shape)) * blocks_b.get(key, 0)
    return total


def _two_site_flops(chi):
    """The two contractions whose work grows with the cube of the bond dimension: L with psi, and
    R with a tensor of psi's blocks."""
    psi, left, right = _legs_two_site(chi)
    return _pair_flops(left, psi, [1], [0]) + _pair_flops(right, psi, [1], [3])


def work(case):
    kind = case["kind"]
    size = DTYPES[case.get("dtype", "f64")][2]
    cx = 4 if case.get("dtype") in ("c128", "c64") else 1
    if kind == "permute":
        return {"bytes": 2 * size * int(np.prod(_ints(case["shape"]))), "flops": 0}
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": size * (m * k + k * n + m * n), "flops": 2 * cx * m * k * n}
    if kind == "dense_chain":
        chi = case["chi"]
        return {"bytes": size * (2 * 5 + 2 * 2) * chi * chi,
                "flops": cx * (4 * 10 * chi ** 3 + 2 * 100 * chi * chi)}
    if kind == "gemm_batch":
        each = case["per_group"]
        return {"bytes": size * each * sum(m * k + k * n + m * n
                                           for m, k, n in _batch_shapes(case)),
                "flops": 2 * cx * each * sum(m * k * n for m, k, n in _batch_shapes(case))}
    if kind == "env":
        lleg, aleg = _legs_env(case["chi"])
        n_l, n_a = _blocks(lleg)[1], _blocks(aleg)[1]
        return {"bytes": size * (2 * n_l + n_a),
                "flops": 2 * cx * _pair_flops(lleg, aleg, [1], [0])}
    if kind in ("heff2", "lanczos2"):
        legs = _legs_two_site(case["chi"])
        n_psi, n_l, n_r = (_blocks(l)[1] for l in legs)
        env = 4 if case.get("precision") == "fp32" else 8
        flops, nbytes = _two_site_flops(case["chi"]), 16 * n_psi + env * (n_l + n_r)
        if kind == "heff2":
            return {"bytes": nbytes, "flops": flops}
        return {"bytes": ITERATIONS * (nbytes + 4 * 8 * n_psi), "flops": ITERATIONS * flops}
    if kind == "lanczos1":
        chi = case["chi"]
        return {"bytes": ITERATIONS * 8 * chi * chi * (10 + 4 + 8),
                "flops": ITERATIONS * (4 * 10 * chi ** 3 + 2 * 100 * chi * chi)}
    legs = _mps_legs(case["sites"], case["chi"])
    n = sum(_blocks(l)[1] for l in legs)
    flops = 0
    for l in legs:
        da, db = sum(l[0][2]), sum(l[2][2])
        # E.A, .conj(A) with and without the MPO, over about half of the charge pairs
        pairs = len(l[0][1])
        flops += 2 * cx * (5 + 1) * 2 * (da * da * db + da * db * db) // max(1, pairs * pairs)
    return {"bytes": 3 * size * n, "flops": 3 * flops}


# ---------------------------------------------------------------------------------- exact
def _wide(t):
    return t.to(torch.complex128) if t.is_complex() else t.to(torch.float64)


def _dot(a, b, axes_a, axes_b):
    return torch.tensordot(a, b, dims=(axes_a, axes_b))


def _lanczos(apply, x):
    """alphas, betas and the lowest Ritz value after ITERATIONS steps of the plain recurrence."""
    alphas, betas = [], []
    v, prev, beta = x / torch.linalg.vector_norm(x), None, 0.0
    for _ in range(ITERATIONS):
        w = apply(v)
        alphas.append(float(torch.dot(w, v)))
        w = w - alphas[-1] * v - (beta * prev if prev is not None else 0.0)
        beta = float(torch.linalg.vector_norm(w))
        betas.append(beta)
        prev, v = v, w / beta
    T = np.diag(alphas) + np.diag(betas[:-1], 1) + np.diag(betas[:-1], -1)
    return {"E": float(np.linalg.eigvalsh(T)[0]), "vec": None, "alphas": np.array(alphas),
            "betas": np.array(betas[:-1])}  # the Ritz vector's sign is free


def exact(case, seed):
    torch.cuda.set_device(DEV)
    kind = case["kind"]
    dt = DTYPES[case.get("dtype", "f64")][1]
    if kind == "permute":
        shape = _ints(case["shape"])
        x = _wide(_Values(seed)(int(np.prod(shape)), dt))
        return x.view(shape).permute(_ints(case["perm"])).reshape(-1)
    if kind == "matmul":
        rnd = _Values(seed)
        m, k, n = case["m"], case["k"], case["n"]
        a = _wide(rnd(m * k, dt, k ** -0.5)).view(m, k)
        return (a @ _wide(rnd(k * n, dt)).view(k, n)).reshape(-1)
    if kind == "dense_chain":
        L, A, R = (_wide(t) for t in _one_site_values(case["chi"], seed, dt, False))
        X = _dot(L, A, [0], [0])                                  # (w, l', s, r)
        Y = _dot(X, _wide(_mpo_dense().to(dt)), [0, 2], [0, 2])   # (l', r, w', s')
        return _dot(Y, R, [1, 2], [0, 1]).reshape(-1)             # (l', s', r')
    if kind == "gemm_batch":
        rnd, out = _Values(seed), []
        for m, k, n in _batch_shapes(case):
            for _ in range(case["per_group"]):
                a = _wide(rnd(m * k, dt, k ** -0.5)).view(m, k)
                out.append((a @ _wide(rnd(k * n, dt)).view(k, n)).reshape(-1))
        return torch.cat(out)
    if kind == "env":
        rnd = _Values(seed)
        lleg, aleg = _legs_env(case["chi"])
        L = _dense(_wide(rnd(_blocks(lleg)[1], dt, case["chi"] ** -0.5)), lleg)
        A = _dense(_wide(rnd(_blocks(aleg)[1], dt, case["chi"] ** -0.5)), aleg)
        X = _dot(L, A, [1], [0])                                  # (w, a', s, b)
        Y = _dot(X, _mpo_dense().to(X.dtype), [0, 2], [0, 2])     # (a', b, w', t)
        Z = _dot(Y, A.conj(), [0, 3], [0, 1])                     # (b, w', b')
        # the blocks in Z's order, each with its legs as (w', b, b')
        return torch.cat([Z[sl].permute(1, 0, 2).reshape(-1)
                          for sl, _, _ in _blocks([lleg[1], lleg[0], lleg[2]])[0]])
    if kind in ("heff2", "lanczos2"):
        legs, psi, left, right = _two_site_values(case, seed, kind == "lanczos2")
        L, R, W = _dense(left, legs[1]), _dense(right, legs[2]), _mpo_dense()

        def apply(x):
            X = _dot(L, _dense(x, legs[0]), [1], [0])             # (w, l', s1, s2, r)
            Y = _dot(X, W, [0, 2], [0, 2])                        # (l', s2, r, w', s1')
            Z = _dot(Y, W, [3, 1], [0, 2])                        # (l', r, s1', w'', s2')
            return _flat(_dot(Z, R, [3, 1], [0, 1]), legs[0])     # (l', s1', s2', r')
        return apply(psi) if kind == "heff2" else _lanczos(apply, psi)
    if kind == "lanczos1":
        L, A, R = _one_site_values(case["chi"], seed, torch.float64, True)
        W = _mpo_dense()

        def apply1(x):
            Y = _dot(_dot(L, x.view(A.shape), [0], [0]), W, [0, 2], [0, 2])
            return _dot(Y, R, [1, 2], [0, 1]).reshape(-1)
        return _lanczos(apply1, A.reshape(-1))
    legs, flats = _mps_values(case, seed)
    flats = [_wide(f).requires_grad_(True) for f in flats]
    W = _mpo_dense().to(flats[0].dtype)
    E = F = None
    for l, f in zip(legs, flats):
        A = _dense(f, l)
        if E is None:
            E = torch.zeros((1, 5, 1), dtype=A.dtype, device=A.device)
            E[0, 2, 0] = 1.0
            F = torch.ones((1, 1), dtype=A.dtype, device=A.device)
        Y = _dot(_dot(E, A, [0], [0]), W, [0, 2], [0, 2])         # (b, a', w', t)
        E = _dot(Y, A.conj(), [0, 3], [0, 1])                     # (a', w', b')
        F = _dot(_dot(F, A, [0], [0]), A.conj(), [0, 1], [0, 1])
    num, den = E[0, 0, 0], F[0, 0]
    e = num.real / den.real if num.is_complex() else num / den
    e.backward()
    return {"E": e.detach(), "grad": [f.grad for f in flats]}
