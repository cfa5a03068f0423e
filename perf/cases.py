"""Performance cases of the framework: the work its users have it do, through
its public entry points.

Six kinds of work, each with its own ranges (``draw`` samples them):

apply   y = A x, Y = A X or A^H X (``VBCSR.mult`` / ``mult_adjoint``) on
        variable-block matrices, real and complex, one to 128 columns.
loop    the Chebyshev moment loop of a user's script: ``mult``, ``scale``,
        ``axpy`` and ``bdot`` on device multivectors, one moment per product.
kpm     native KPM moments of one Hamiltonian (``kpm.kpm_moments``).
batch   native KPM moments of many Hamiltonians (``kpm.kpm_moments_batched``).
prop    Chebyshev time propagation (``autograd.propagate``), forward only or
        with the gradient of the block values.
spgemm  thresholded products of density-matrix purification (``VBCSR.spmm``,
        ``spmm_hermitian``) in FP64, FP32 or BF16.

Matrices are Hermitian tight-binding Hamiltonians (a periodic honeycomb
lattice, or a periodic cubic lattice with all neighbours up to a radius and
the sites numbered at random), scaled so that their spectrum lies inside
[-1, 1], or non-symmetric matrices with uniformly drawn block columns.
"""
import math

import numpy as np
import torch

DEV = "cuda"


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one matrix-vector product of a small matrix (500 block rows of 4-8,
        # about 40 blocks a row): the latency of a single call
        {"name": "spmv_small", "kind": "apply", "pattern": "random", "nb": 500, "per_row": 40, "blocks": "4-8",
         "complex": False, "K": 1, "adjoint": False},
        # one matrix-vector product of a matrix far beyond every cache (0.7 GB
        # of values): the inner step of an eigensolver
        {"name": "spmv_large", "kind": "apply", "pattern": "random", "nb": 60000, "per_row": 40, "blocks": "4-8",
         "complex": False, "K": 1, "adjoint": False},
        # a block of 96 columns (filtered subspace iteration) on an atomic
        # basis of 1, 4, 9 and 13 functions a site
        {"name": "spmm_wide", "kind": "apply", "pattern": "cubic", "side": 20, "radius2": 2, "blocks": "1,4,9,13",
         "complex": False, "K": 96, "adjoint": False},
        # the adjoint product of a complex matrix with a few columns
        # (biorthogonal Krylov methods)
        {"name": "adjoint_c128", "kind": "apply", "pattern": "random", "nb": 6000, "per_row": 20, "blocks": "4-8",
         "complex": True, "K": 6, "adjoint": True},
        # a user's own moment loop on a graphene-like lattice, 10 random vectors
        {"name": "moment_loop", "kind": "loop", "nx": 96, "ny": 90, "orbitals": 4, "K": 10, "M": 24},
        # density of states of graphene, 200 x 200 cells with 4 orbitals, 200
        # moments, 10 random vectors, FP32 recursion: the benchmark's workload
        {"name": "kpm_graphene_fp32", "kind": "kpm", "nx": 200, "ny": 200, "orbitals": 4, "K": 10, "M": 200,
         "mode": "two", "precision": "fp32"},
        # the same question for a small sample in FP64: many short steps
        {"name": "kpm_small_fp64", "kind": "kpm", "nx": 21, "ny": 20, "orbitals": 4, "K": 4, "M": 128, "mode": "two",
         "precision": "fp64"},
        # spectra of many independent molecules at once, FP32 values and FP64
        # vectors
        {"name": "kpm_batch_mixed", "kind": "batch", "count": 16, "side_lo": 5, "side_hi": 14, "radius2": 2,
         "blocks": "1,4,9,13", "K": 32, "M": 128, "precision": "mixed"},
        # training through a time propagation: the gradient of an overlap with
        # respect to every block value, complex128, one wave packet
        {"name": "propagate_grad_c128", "kind": "prop", "nx": 100, "ny": 100, "orbitals": 4, "K": 1, "nsteps": 10,
         "nterms": 64, "checkpoint": 5, "precision": "fp64", "grad": True},
        # propagation of four states in complex64
        {"name": "propagate_c64", "kind": "prop", "nx": 77, "ny": 65, "orbitals": 4, "K": 4, "nsteps": 20,
         "nterms": 48, "checkpoint": 10, "precision": "fp32", "grad": False},
        # the first product of a purification: about 30 neighbours a row,
        # blocks of 4-8, threshold 1e-5, FP64
        {"name": "spgemm_fp64", "kind": "spgemm", "side": 17, "radius2": 4, "blocks": "4-8", "numeric": "fp64",
         "hermitian": False, "threshold": 1e-5},
        # a later product, whose factors have filled up, in BF16
        {"name": "spgemm_filled_bf16", "kind": "spgemm", "side": 12, "radius2": 14, "blocks": "4-8",
         "numeric": "bf16", "hermitian": False, "threshold": 1e-7},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= 5e10 and w["bytes"] <= 1.5e9:
            return case


def _draw(rng):
    kind = rng.choice(["apply", "apply", "loop", "kpm", "kpm", "batch", "prop", "prop", "spgemm", "spgemm"])
    blocks = rng.choice(["4-8", "1,4,9,13", "1-6", "3", "4", "2-13"])
    if kind == "apply":
        K = 1 if rng.random() < 0.4 else _log_int(rng, 2, 128)
        cplx = rng.random() < 0.35
        # bounded by 6e7 stored values and by 6e8 products of values and columns
        cap = min(6e7, 6e8 / K) / (36 * (2 if cplx else 1))
        if rng.random() < 0.5:
            per_row = rng.randint(8, 60)
            return {"kind": kind, "pattern": "random", "nb": _log_int(rng, 200, max(400, min(40000, cap / per_row))),
                    "per_row": per_row, "blocks": blocks, "complex": cplx, "K": K, "adjoint": rng.random() < 0.35}
        r2 = rng.randint(1, 5)
        side = int(max(7, min(30, (cap / _stencil_count(r2)) ** (1.0 / 3.0))))
        return {"kind": kind, "pattern": "cubic", "side": _log_int(rng, 6, side), "radius2": r2, "blocks": blocks,
                "complex": cplx, "K": K, "adjoint": rng.random() < 0.35}
    if kind == "loop":
        return {"kind": kind, "nx": _log_int(rng, 10, 140), "ny": _log_int(rng, 10, 140), "orbitals": rng.randint(2, 6),
                "K": _log_int(rng, 1, 24), "M": rng.randint(10, 40)}
    if kind == "kpm":
        prec = rng.choice(["fp64", "fp32", "mixed"])
        return {"kind": kind, "nx": _log_int(rng, 8, 160), "ny": _log_int(rng, 8, 160),
                "orbitals": rng.choice([2, 4, 4, 5]), "K": _log_int(rng, 1, 12), "M": _log_int(rng, 32, 200),
                "mode": rng.choice(["two", "two", "one"]), "precision": prec}
    if kind == "batch":
        lo = rng.randint(4, 6)
        return {"kind": kind, "count": rng.randint(3, 16), "side_lo": lo, "side_hi": rng.randint(lo + 1, 13),
                "radius2": rng.randint(1, 3), "blocks": blocks, "K": rng.choice([8, 10, 16, 17, 32]),
                "M": _log_int(rng, 32, 200), "precision": rng.choice(["fp64", "fp32", "mixed", "mixed"])}
    if kind == "prop":
        grad = rng.random() < 0.6
        return {"kind": kind, "nx": _log_int(rng, 12, 90), "ny": _log_int(rng, 12, 90), "orbitals": rng.choice([2, 4, 4, 5]),
                "K": rng.choice([1, 1, 1, 2, 4]), "nsteps": rng.randint(3, 8 if grad else 20),
                "nterms": rng.randint(24, 64), "checkpoint": rng.randint(2, 6),
                "precision": rng.choice(["fp64", "fp32"]), "grad": grad}
    numeric = rng.choice(["fp64", "fp64", "fp32", "bf16"])
    r2 = rng.randint(1, 8)
    top = {1: 20, 2: 18, 3: 17, 4: 16}.get(r2, 12)
    return {"kind": kind, "side": _log_int(rng, 6, top), "radius2": r2, "blocks": rng.choice(["4-8", "1-6", "3", "4"]),
            "numeric": numeric, "hermitian": numeric == "fp64" and rng.random() < 0.3,
            # (reduced precision: far below every block, so that rounding decides on none)
            "threshold": rng.choice([0.0, 1e-5, 1e-4] if numeric == "fp64" else [0.0, 1e-9])}


# ---------------------------------------------------------------- matrices
def _sizes(spec):
    if "-" in spec:
        lo, hi = (int(t) for t in spec.split("-"))
        return np.arange(lo, hi + 1, dtype=np.int32)
    return np.array([int(t) for t in spec.split(",")], np.int32)


def _block_sizes(spec, nb, rng):
    """Every size equally often, in random order: the row count does not
    depend on the seed."""
    return rng.permutation(np.resize(_sizes(spec), nb))


def _stencil(radius2):
    """Half of the non-zero cubic offsets of squared length <= radius2."""
    m = int(math.isqrt(radius2))
    r = range(-m, m + 1)
    return [(x, y, z) for x in r for y in r for z in r
            if 0 < x * x + y * y + z * z <= radius2 and (x, y, z) > (0, 0, 0)]


def _stencil_count(radius2):
    return 2 * len(_stencil(radius2)) + 1


def _cubic_pairs(side, radius2, rng):
    """Pairs (i, j) of a periodic cubic lattice, sites numbered at random,
    each pair once, and the weights exp(-distance / cutoff)."""
    n = side ** 3
    label = rng.permutation(n)
    x, y, z = np.unravel_index(np.arange(n), (side, side, side))
    iu, ju, w = [label], [label], [np.ones(n)]
    cut = math.sqrt(radius2)
    for dx, dy, dz in _stencil(radius2):
        other = np.ravel_multi_index(((x + dx) % side, (y + dy) % side, (z + dz) % side), (side, side, side))
        iu.append(label)
        ju.append(label[other])
        w.append(np.full(n, math.exp(-math.sqrt(dx * dx + dy * dy + dz * dz) / cut)))
    iu, ju, w = np.concatenate(iu), np.concatenate(ju), np.concatenate(w)
    lo, hi = np.minimum(iu, ju), np.maximum(iu, ju)
    _, first = np.unique(lo * n + hi, return_index=True)  # short sides meet themselves
    return n, lo[first], hi[first], w[first]


def _honeycomb_pairs(nx, ny):
    """On-site, 3 nearest and 6 next-nearest pairs of a periodic honeycomb
    lattice, each pair once, and the weights 1 / distance."""
    ix, iy = (g.ravel() for g in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))

    def site(x, y, s):
        return 2 * ((x % nx) * ny + y % ny) + s

    a = site(ix, iy, 0)
    b = site(ix, iy, 1)
    iu, ju, w = [a, b], [a, b], [1.0, 1.0]
    for dx, dy in ((0, 0), (-1, 0), (0, -1)):
        iu.append(a)
        ju.append(site(ix + dx, iy + dy, 1))
        w.append(1.0)
    for s in (0, 1):
        for dx, dy in ((1, 0), (0, 1), (1, -1)):
            iu.append(site(ix, iy, s))
            ju.append(site(ix + dx, iy + dy, s))
            w.append(1.0 / math.sqrt(3.0))
    w = np.repeat(w, nx * ny)
    iu, ju = np.concatenate(iu), np.concatenate(ju)
    lo, hi = np.minimum(iu, ju), np.maximum(iu, ju)
    _, first = np.unique(lo * (2 * nx * ny) + hi, return_index=True)
    return 2 * nx * ny, lo[first], hi[first], w[first]


class _Matrix:
    """Block-row CSR arrays on the host (bs, row_ptr, col_ind, vals)."""

    def __init__(self, bs, row_ptr, col_ind):
        self.bs, self.row_ptr, self.col_ind = bs, row_ptr.astype(np.int64), col_ind.astype(np.int32)
        self.nb, self.nnzb, self.n = len(bs), len(col_ind), int(bs.sum())
        self.rows = np.repeat(np.arange(self.nb), np.diff(self.row_ptr))
        self.off = np.concatenate([[0], np.cumsum(bs, dtype=np.int64)])
        self.r = bs[self.rows].astype(np.int64)
        self.c = bs[self.col_ind].astype(np.int64)
        self.voff = np.concatenate([[0], np.cumsum(self.r * self.c)])
        self.nnz = int(self.voff[-1])

    def elements(self):
        """Slot, row in the block and column in the block of every value."""
        sz = torch.as_tensor(self.r * self.c, device=DEV)
        slot = torch.repeat_interleave(torch.arange(self.nnzb, device=DEV), sz)
        e = torch.arange(self.nnz, device=DEV) - torch.as_tensor(self.voff, device=DEV)[slot]
        c = torch.as_tensor(self.c, device=DEV)[slot]
        a = torch.div(e, c, rounding_mode="floor")
        return slot, a, e - a * c


def _hermitian(bs, iu, ju, w, cplx, rng):
    """Hermitian matrix with blocks of uniform entries of unit variance times w
    on the pairs (iu <= ju), divided by a little more than its spectral radius:
    2.4 times the root of the largest row sum of the entries' variances."""
    nb = len(bs)
    p = np.arange(len(iu))
    off = iu != ju
    rows, cols = np.concatenate([iu, ju[off]]), np.concatenate([ju, iu[off]])
    pair = np.concatenate([p, p[off]])
    mirror = np.concatenate([np.zeros(len(iu), bool), np.ones(int(off.sum()), bool)])
    order = np.lexsort((cols, rows))
    rows, cols, pair, mirror = rows[order], cols[order], pair[order], mirror[order]
    row_ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nb))])
    m = _Matrix(bs, row_ptr, cols)
    usz = bs[iu].astype(np.int64) * bs[ju]
    uoff = np.concatenate([[0], np.cumsum(usz)])
    u = math.sqrt(12.0) * (rng.random(int(uoff[-1])) - 0.5)
    if cplx:
        u = (u + 1j * math.sqrt(12.0) * (rng.random(len(u)) - 0.5)) * math.sqrt(0.5)
    var = np.bincount(rows, weights=w[pair] ** 2 * bs[cols], minlength=nb)
    scale = w / (2.4 * math.sqrt(var.max()))
    ud = torch.as_tensor(u, device=DEV) * torch.repeat_interleave(torch.as_tensor(scale, device=DEV),
                                                                 torch.as_tensor(usz, device=DEV))
    slot, a, b = m.elements()
    first = torch.as_tensor(uoff[pair], device=DEV)[slot]
    r, c = torch.as_tensor(m.r, device=DEV)[slot], torch.as_tensor(m.c, device=DEV)[slot]
    direct, turned = ud[first + a * c + b], ud[first + b * r + a].conj().resolve_conj()
    mi = torch.as_tensor(mirror, device=DEV)[slot]
    diag = torch.as_tensor(rows == cols, device=DEV)[slot]
    m.vals = torch.where(diag, 0.5 * (direct + turned), torch.where(mi, turned, direct)).cpu().numpy()
    return m


def _honeycomb(case, seed, cplx):
    rng = np.random.default_rng(seed)
    nb, iu, ju, w = _honeycomb_pairs(case["nx"], case["ny"])
    return _hermitian(np.full(nb, case["orbitals"], np.int32), iu, ju, w, cplx, rng), rng


def _cubic(side, radius2, blocks, cplx, rng):
    nb, iu, ju, w = _cubic_pairs(side, radius2, rng)
    return _hermitian(_block_sizes(blocks, nb, rng), iu, ju, w, cplx, rng)


def _random(case, rng):
    """The diagonal block and per_row uniformly drawn block columns a row,
    entries uniform in [-1, 1]."""
    nb, per = case["nb"], case["per_row"]
    bs = _block_sizes(case["blocks"], nb, rng)
    cols = rng.integers(0, nb, size=(nb, per + 1))
    cols[:, 0] = np.arange(nb)
    cols.sort(axis=1)
    keep = np.ones(cols.shape, bool)
    keep[:, 1:] = cols[:, 1:] != cols[:, :-1]
    m = _Matrix(bs, np.concatenate([[0], np.cumsum(keep.sum(1))]), cols[keep])
    m.vals = rng.random(m.nnz) * 2.0 - 1.0
    if case["complex"]:
        m.vals = m.vals + 1j * (rng.random(m.nnz) * 2.0 - 1.0)
    return m


def _vbcsr(m):
    from vbcsr_amd import VBCSR

    return VBCSR.from_block_csr(m.bs, m.row_ptr, m.col_ind, m.vals)


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Host inputs of a case, from the seed alone."""
    kind = case["kind"]
    if kind == "apply":
        rng = np.random.default_rng(seed)
        if case["pattern"] == "random":
            m = _random(case, rng)
        else:
            m = _cubic(case["side"], case["radius2"], case["blocks"], case["complex"], rng)
        x = rng.standard_normal((m.n, case["K"]))
        if case["complex"]:
            x = x + 1j * rng.standard_normal(x.shape)
        return m, x
    if kind in ("loop", "kpm"):
        m, rng = _honeycomb(case, seed, False)
        return m, 2.0 * rng.integers(0, 2, size=(m.n, case["K"])) - 1.0
    if kind == "batch":
        rng = np.random.default_rng(seed)
        # sides spread evenly over the range, so that the work does not
        # depend on the seed
        sides = np.linspace(case["side_lo"], case["side_hi"], case["count"]).round().astype(int)
        ms = [_cubic(int(s), case["radius2"], case["blocks"], False, rng) for s in sides]
        return ms, [2.0 * rng.integers(0, 2, size=(m.n, case["K"])) - 1.0 for m in ms]
    if kind == "prop":
        m, rng = _honeycomb(case, seed, True)
        cells = case["nx"] * case["ny"]
        ix, iy = np.unravel_index(np.arange(cells), (case["nx"], case["ny"]))
        # Gaussian packets around the middle of the sample, a random phase an orbital
        env = np.exp(-(((ix - case["nx"] / 2) / (0.2 * case["nx"])) ** 2 + ((iy - case["ny"] / 2) / (0.2 * case["ny"])) ** 2))
        env = np.repeat(env, 2 * case["orbitals"])[:, None]
        psi = env * np.exp(2j * np.pi * rng.random((m.n, case["K"])))
        psi /= np.linalg.norm(psi, axis=0)
        target = rng.standard_normal(psi.shape) + 1j * rng.standard_normal(psi.shape)
        target /= np.linalg.norm(target, axis=0)
        if case["precision"] == "fp32":
            psi, target = psi.astype(np.complex64), target.astype(np.complex64)
        return m, psi, target
    # one Hamiltonian a case, in a local basis of the seed's: the functions of
    # every site reordered and their signs changed, which leaves the norms of
    # the blocks, and with them the pattern of the product, as they are
    m = _cubic(case["side"], case["radius2"], case["blocks"], False, np.random.default_rng(case["side"]))
    rng = np.random.default_rng(seed)
    site = np.repeat(np.arange(m.nb), m.bs)
    order = torch.as_tensor(np.lexsort((rng.random(m.n), site)) - m.off[site], device=DEV)
    sign = torch.as_tensor(2.0 * rng.integers(0, 2, size=m.n) - 1.0, device=DEV)
    slot, a, b = m.elements()
    off = torch.as_tensor(m.off, device=DEV)
    row = off[torch.as_tensor(m.rows, device=DEV)[slot]] + a
    col = off[torch.as_tensor(m.col_ind.astype(np.int64), device=DEV)[slot]] + b
    place = torch.as_tensor(m.voff, device=DEV)[slot] + order[row] * torch.as_tensor(m.c, device=DEV)[slot] + order[col]
    # the start of a purification: 0.1 H + 0.5
    m.vals = (0.1 * sign[row] * sign[col] * torch.as_tensor(m.vals, device=DEV)[place]).cpu().numpy()
    d = np.nonzero(m.rows == m.col_ind)[0]
    for b in np.unique(m.bs):
        s = m.voff[d[m.r[d] == b]]
        m.vals[(s[:, None] + np.arange(b) * (b + 1)).ravel()] += 0.5
    return (m,)


class _Device:
    """Device memory that ``owner`` keeps alive, for torch."""

    def __init__(self, owner, ptr, shape, strides, dtype):
        self.owner = owner
        item = np.dtype(dtype).itemsize
        self.__cuda_array_interface__ = {"shape": shape, "strides": tuple(s * item for s in strides),
                                         "typestr": np.dtype(dtype).str, "data": (ptr, False), "version": 2}


def _view(v):
    """A device vector or multivector as a torch tensor over its own memory."""
    if v.ndim == 1:
        return torch.as_tensor(_Device(v, v._core.device_ptr, (v.local_size,), (1,), v.dtype), device=DEV)
    return torch.as_tensor(_Device(v, v._core.device_ptr, v.shape, (v._core.ld, 1), v.dtype), device=DEV)


def _fill(v, x):
    v.from_numpy(x)
    v._core.device_ptr  # moves the host copy to the device
    return v


def prepare(case, seed):
    kind = case["kind"]
    if kind == "apply":
        m, x = _inputs(case, seed)
        H = _vbcsr(m)
        if case["K"] == 1:
            x, y = _fill(H.create_vector(), x[:, 0]), H.create_vector()
        else:
            x, y = _fill(H.create_multivector(case["K"]), x), H.create_multivector(case["K"])
        H._core.handle  # moves the values to the device
        return {"kind": kind, "call": H.mult_adjoint if case["adjoint"] else H.mult, "x": x, "y": y, "out": _view(y)}
    if kind == "loop":
        m, v0 = _inputs(case, seed)
        H = _vbcsr(m)
        H._core.handle
        work = [H.create_multivector(case["K"]) for _ in range(3)]
        return {"kind": kind, "H": H, "v0": _fill(H.create_multivector(case["K"]), v0), "work": work,
                "views": [_view(t) for t in work], "M": case["M"]}
    if kind == "kpm":
        m, v0 = _inputs(case, seed)
        H = _vbcsr(m)
        H._core.handle
        return {"kind": kind, "H": H, "v0": _fill(H.create_multivector(case["K"]), v0), "M": case["M"],
                "mode": case["mode"], "precision": case["precision"]}
    if kind == "batch":
        ms, v0s = _inputs(case, seed)
        Hs = [_vbcsr(m) for m in ms]
        for H in Hs:
            H._core.handle
        return {"kind": kind, "Hs": Hs, "v0s": [_fill(H.create_multivector(case["K"]), v) for H, v in zip(Hs, v0s)],
                "M": case["M"], "precision": case["precision"]}
    if kind == "prop":
        m, psi, target = _inputs(case, seed)
        H = _vbcsr(m)
        H._core.handle
        return {"kind": kind, "H": H, "values": torch.as_tensor(m.vals, device=DEV),
                "psi": torch.as_tensor(psi, device=DEV), "target": torch.as_tensor(target, device=DEV), "case": case}
    (m,) = _inputs(case, seed)
    P = _vbcsr(m)
    P._core.handle
    return {"kind": kind, "P": P, "case": case}


# ---------------------------------------------------------------- one pass
DT = 0.5  # time step of the propagations


def run(state):
    kind = state["kind"]
    if kind == "apply":
        state["call"](state["x"], state["y"])
        return state["out"]
    if kind == "loop":
        H, v0 = state["H"], state["v0"]
        prev, cur, nxt = state["work"]
        a, b, c = state["views"]
        prev._core.copy_from(v0._core)
        H.mult(prev, cur)
        mu = [v0.bdot(prev), v0.bdot(cur)]
        for _ in range(2, state["M"]):  # t_n = 2 H t_n-1 - t_n-2
            H.mult(cur, nxt)
            nxt.scale(2.0)
            nxt.axpy(-1.0, prev)
            mu.append(v0.bdot(nxt))
            prev, cur, nxt = cur, nxt, prev
            a, b, c = b, c, a
        return {"moments": np.array(mu), "last": b}
    if kind == "kpm":
        from vbcsr_amd import kpm

        return kpm.kpm_moments(state["H"], state["v0"], state["M"], mode=state["mode"], precision=state["precision"])
    if kind == "batch":
        from vbcsr_amd import kpm

        return kpm.kpm_moments_batched(state["Hs"], state["v0s"], state["M"], precision=state["precision"])
    case = state["case"]
    if kind == "prop":
        from vbcsr_amd import autograd

        args = (DT, case["nsteps"], case["nterms"])
        if not case["grad"]:
            with torch.no_grad():
                return {"psi": autograd.propagate(state["H"], state["values"], state["psi"], *args,
                                                  precision=case["precision"])}
        values = state["values"].detach().requires_grad_(True)
        psi0 = state["psi"].detach().requires_grad_(True)
        psi = autograd.propagate(state["H"], values, psi0, *args, checkpoint=case["checkpoint"],
                                 precision=case["precision"])
        loss = _overlap(state["target"], psi)
        loss.backward()
        return {"psi": psi.detach(), "loss": loss.detach(), "grad_values": values.grad, "grad_psi0": psi0.grad}
    P = state["P"]
    product = P.spmm_hermitian if case["hermitian"] else P.spmm
    C = product(P, case["threshold"], numeric=case["numeric"])
    values = torch.as_tensor(_Device(C, C._core.values_ptr, (C.local_nnz,), (1,), C.dtype), device=DEV)
    return {"row_ptr": C.row_ptr, "col_ind": C.col_ind, "values": values}


def _overlap(target, psi):
    o = (target.conj() * psi).sum(0)
    return (o.real ** 2 + o.imag ** 2).sum()


# ---------------------------------------------------------------- work
def work(case):
    """Inputs read once, outputs written once, and the products of the stored
    values with the columns (a complex product counts 8 operations)."""
    kind = case["kind"]

    def stored(nb, per, bs):  # bytes of the pattern, values, rows
        return 4.0 * nb * (per + 1), nb * per * bs * bs, nb * bs

    if kind == "apply":
        nb = case["nb"] if case["pattern"] == "random" else case["side"] ** 3
        per = case["per_row"] + 1 if case["pattern"] == "random" else _stencil_count(case["radius2"])
        idx, nnz, n = stored(nb, per, float(_sizes(case["blocks"]).mean()))
        p, f = (16, 8) if case["complex"] else (8, 2)
        return {"bytes": idx + p * nnz + 2 * p * n * case["K"], "flops": f * nnz * case["K"]}
    if kind == "batch":
        sides = np.linspace(case["side_lo"], case["side_hi"], case["count"]).round()
        idx, nnz, n = stored(float((sides ** 3).sum()), _stencil_count(case["radius2"]), float(_sizes(case["blocks"]).mean()))
        pv = 8 if case["precision"] == "fp64" else 4
        px = 4 if case["precision"] == "fp32" else 8
        return {"bytes": idx + pv * nnz + px * n * case["K"] + 8 * case["count"] * case["M"],
                "flops": 2 * nnz * case["K"] * (case["M"] // 2)}
    if kind == "spgemm":
        nb, per, bs = case["side"] ** 3, _stencil_count(case["radius2"]), float(_sizes(case["blocks"]).mean())
        idx, nnz, _ = stored(nb, min(per, nb), bs)
        perc = min(_stencil_count(4 * case["radius2"]), nb)  # neighbours within twice the radius
        idxc, nnzc, _ = stored(nb, perc, bs)
        share = 0.5 if case["hermitian"] else 1.0
        return {"bytes": idx + 8 * nnz + idxc + 8 * nnzc, "flops": share * 2 * nb * min(per, nb) ** 2 * bs ** 3}
    bs = case["orbitals"]
    idx, nnz, n = stored(2 * case["nx"] * case["ny"], 10, bs)
    if kind == "loop":
        return {"bytes": idx + 8 * nnz + 2 * 8 * n * case["K"], "flops": (2 * nnz + 5 * n) * case["K"] * (case["M"] - 1)}
    if kind == "kpm":
        pv = 8 if case["precision"] == "fp64" else 4
        px = 4 if case["precision"] == "fp32" else 8
        steps = case["M"] // 2 if case["mode"] == "two" else case["M"] - 1
        return {"bytes": idx + pv * nnz + px * n * case["K"] + 8 * case["M"],
                "flops": (2 * nnz + 7 * n) * case["K"] * steps}
    p = 16 if case["precision"] == "fp64" else 8
    applies = case["nsteps"] * (case["nterms"] - 1)
    # the gradient: the states again, the adjoint recurrence and an outer product a term
    times = 4 if case["grad"] else 1
    return {"bytes": idx + p * nnz + 2 * p * n * case["K"] + (16 * nnz + p * n * case["K"] if case["grad"] else 0),
            "flops": 8.0 * nnz * case["K"] * applies * times}


# ---------------------------------------------------------------- 64-bit values
class _Rows:
    """The scalar rows of a block matrix, each padded to the longest: the
    index of every value and its column.  Products in plain torch."""

    def __init__(self, m, adjoint=False):
        slot, a, b = m.elements()
        off = torch.as_tensor(m.off, device=DEV)
        row = off[torch.as_tensor(m.rows, device=DEV)[slot]] + a
        col = off[torch.as_tensor(m.col_ind.astype(np.int64), device=DEV)[slot]] + b
        if adjoint:
            row, col = col, row
        order = torch.argsort(row, stable=True)
        row, col = row[order], col[order]
        count = torch.bincount(row, minlength=m.n)
        start = torch.cumsum(count, 0) - count
        place = torch.arange(m.nnz, device=DEV) - start[row]
        width = max(int(count.max()), 1)
        self.index = torch.full((m.n, width), m.nnz, device=DEV)  # the value past the end is a zero
        self.index[row, place] = order
        self.col = torch.zeros((m.n, width), dtype=torch.int64, device=DEV)
        self.col[row, place] = col

    def padded(self, vals):
        return torch.cat([vals, vals.new_zeros(1)])[self.index]

    def product(self, padded, X):
        step = max(1, (1 << 26) // (self.index.shape[1] * X.shape[1]))
        if step >= self.index.shape[0]:
            return (padded[:, :, None] * X[self.col]).sum(1)
        return torch.cat([(padded[i:i + step, :, None] * X[self.col[i:i + step]]).sum(1)
                          for i in range(0, self.index.shape[0], step)])


def _moments(m, v0, M):
    rows = _Rows(m)
    A, t0 = rows.padded(torch.as_tensor(m.vals, device=DEV)), torch.as_tensor(v0, device=DEV)
    prev, cur = t0, rows.product(A, t0)
    mu = [(t0 * t0).sum(0), (t0 * cur).sum(0)]
    for _ in range(2, M):
        prev, cur = cur, 2.0 * rows.product(A, cur) - prev
        mu.append((t0 * cur).sum(0))
    return torch.stack(mu).cpu().numpy(), cur


def _bessel(n, x):
    """J_0(x) .. J_n-1(x): the trapezoidal rule of their integral over a period."""
    t = np.arange(4096) * (2.0 * np.pi / 4096)
    return np.cos(np.arange(n)[:, None] * t - x * np.sin(t)).mean(1)


def _propagation(m, values, psi, case):
    rows = _Rows(m)
    A = rows.padded(values)
    coef = (-1j) ** np.arange(case["nterms"]) * _bessel(case["nterms"], DT) * np.where(np.arange(case["nterms"]) > 0, 2.0, 1.0)
    for _ in range(case["nsteps"]):
        prev, cur = psi, rows.product(A, psi)
        out = complex(coef[0]) * prev + complex(coef[1]) * cur
        for n in range(2, case["nterms"]):
            prev, cur = cur, 2.0 * rows.product(A, cur) - prev
            out = out + complex(coef[n]) * cur
        psi = out
    return psi


def _product_blocks(m, case):
    """The kept blocks of the thresholded square of m: values in slot order."""
    thr, nb, w = case["threshold"], m.nb, int(m.bs.max())
    vals = torch.as_tensor(m.vals, device=DEV)
    slot, a, b = m.elements()
    blocks = torch.zeros((m.nnzb, w, w), dtype=torch.float64, device=DEV)
    blocks[slot, a, b] = vals
    del slot, a, b
    rows, cols = torch.as_tensor(m.rows, device=DEV), torch.as_tensor(m.col_ind.astype(np.int64), device=DEV)
    ptr = torch.as_tensor(m.row_ptr, device=DEV)
    norm = blocks.square().sum((1, 2)).sqrt()
    dense = torch.zeros((nb, nb), dtype=torch.float64, device=DEV)
    dense[rows, cols] = norm
    keep = dense @ dense > thr
    if case["hermitian"]:
        keep &= torch.arange(nb, device=DEV)[None, :] >= torch.arange(nb, device=DEV)[:, None]
    del dense
    place = torch.full((nb, nb), -1, dtype=torch.int64, device=DEV)
    ci, cj = keep.nonzero(as_tuple=True)
    place[ci, cj] = torch.arange(len(ci), device=DEV)
    C = torch.zeros((len(ci), w, w), dtype=torch.float64, device=DEV)
    count = ptr[1:] - ptr[:-1]
    eps = thr / count.clamp(min=1).to(torch.float64)
    per = count[cols]  # partners of every left block
    first = torch.cumsum(per, 0) - per
    total = int(per.sum())
    for p0 in range(0, total, 1 << 20):
        p = torch.arange(p0, min(total, p0 + (1 << 20)), device=DEV)
        left = torch.searchsorted(first, p, right=True) - 1
        right = ptr[cols[left]] + (p - first[left])
        at = place[rows[left], cols[right]]
        # pairs below the row's share of the threshold are left out
        ok = at >= 0
        ok &= ~(norm[left] * norm[right] < eps[rows[left]])
        left, right, at = left[ok], right[ok], at[ok]
        C.index_add_(0, at, torch.bmm(blocks[left], blocks[right]))
    cn = C.square().sum((1, 2)).sqrt()
    if case["numeric"] != "fp64" and thr > 0.0 and bool(((cn - thr).abs() < 0.1 * thr).any()):
        return None  # which blocks stay depends on the rounding
    if thr > 0.0:
        stay = cn >= thr
        ci, cj, C = ci[stay], cj[stay], C[stay]
    if case["hermitian"]:
        up = ci < cj
        diag = ci == cj
        C[diag] = 0.5 * (C[diag] + C[diag].transpose(1, 2))
        C = torch.cat([C, C[up].transpose(1, 2)])
        ci, cj = torch.cat([ci, cj[up]]), torch.cat([cj, ci[up]])
        order = torch.argsort(ci * nb + cj)
        C, ci, cj = C[order], ci[order], cj[order]
    bs = torch.as_tensor(m.bs.astype(np.int64), device=DEV)
    k = torch.arange(w, device=DEV)
    inside = (k[None, :, None] < bs[ci][:, None, None]) & (k[None, None, :] < bs[cj][:, None, None])
    return C[inside].cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "apply":
        m, x = _inputs(case, seed)
        rows = _Rows(m, case["adjoint"])
        vals = torch.as_tensor(m.vals, device=DEV)
        y = rows.product(rows.padded(vals.conj().resolve_conj() if case["adjoint"] else vals), torch.as_tensor(x, device=DEV))
        return (y[:, 0] if case["K"] == 1 else y).cpu().numpy()
    if kind == "loop":
        m, v0 = _inputs(case, seed)
        mu, last = _moments(m, v0, case["M"])
        return {"moments": mu, "last": last.cpu().numpy()}
    if kind == "kpm":
        m, v0 = _inputs(case, seed)
        return _moments(m, v0, case["M"])[0].sum(1)
    if kind == "batch":
        return np.stack([_moments(m, v0, case["M"])[0].sum(1) for m, v0 in zip(*_inputs(case, seed))])
    if kind == "prop":
        m, psi, target = _inputs(case, seed)
        values = torch.as_tensor(m.vals, device=DEV)
        psi, target = (torch.as_tensor(t, device=DEV).to(torch.complex128) for t in (psi, target))
        if not case["grad"]:
            with torch.no_grad():
                return {"psi": _propagation(m, values, psi, case).cpu().numpy()}
        values.requires_grad_(True)
        psi.requires_grad_(True)
        out = _propagation(m, values, psi, case)
        loss = _overlap(target, out)
        loss.backward()
        return {"psi": out.detach().cpu().numpy(), "loss": loss.detach().cpu().numpy(), "grad_values": values.grad.cpu().numpy(),
                "grad_psi0": psi.grad.cpu().numpy()}
    values = _product_blocks(*_inputs(case, seed), case)
    return None if values is None else {"row_ptr": None, "col_ind": None, "values": values}
