"""The work that programs have this framework do, as measurable cases.

Every case is one call (or the short chain of calls that belong together)
through the package's public entry points: sparse matrix-vector products,
the Krylov solvers with their preconditioners, ILU(0) set-up, mixed
precision, batches of systems and the training of the learned approximate
inverse.  A case is a dict of plain values; `kind` names the path.

Matrices come from the package's own generators where these take sizes only
(Poisson, convection-diffusion) and are made here from the seed where their
values vary (diffusion, power-law rows).  Right-hand sides come from the
seed; where no closed form of the solution exists the right-hand side is
A x for an x drawn from the seed, so that x is the exact answer.
"""
import math

import numpy as np
import torch

import sparkit_amd as spk

_TYPESTR = {np.dtype(np.float64): "<f8", np.dtype(np.float32): "<f4"}


class _View:
    """A DeviceVector's memory as torch.as_tensor reads it (no copy)."""

    def __init__(self, vec):
        self.vec = vec
        self.__cuda_array_interface__ = {
            "shape": (vec.n,), "typestr": _TYPESTR[vec.dtype],
            "data": (vec.ptr.value, False), "version": 2}


def _tensor(vec):
    return torch.as_tensor(_View(vec), device="cuda")


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # latency of the smallest product: y = multiply(A, x) returns a new
        # vector, as an explicit time step or a user's own iteration calls it
        {"name": "spmv_poisson2d_64", "kind": "multiply", "matrix": "poisson2d",
         "nx": 64, "ny": 64, "dtype": "f64"},
        # the largest product: 7.1M rows, streaming, into a kept vector
        {"name": "spmv_poisson3d_192", "kind": "spmv", "matrix": "poisson3d",
         "nx": 192, "ny": 192, "nz": 192, "dtype": "f64"},
        # irregular rows in single precision: a scale-free graph's matrix
        {"name": "spmv_powerlaw_f32", "kind": "spmv", "matrix": "powerlaw",
         "n": 262144, "dtype": "f32"},
        # Jacobi-PCG on a small 2D problem: many short iterations
        {"name": "cg_poisson2d_256", "kind": "cg", "matrix": "poisson2d",
         "nx": 256, "ny": 256, "shift": 0.01, "tol": 1e-8},
        # Jacobi-PCG at full size: the solver's streaming rate
        {"name": "cg_poisson3d_192", "kind": "cg", "matrix": "poisson3d",
         "nx": 192, "ny": 192, "nz": 192, "tol": 1e-8},
        # FP32 PCG with FP64 reliable updates, coefficients that vary from
        # cell to cell, a 9-point stencil on a ragged grid
        {"name": "ir_cg_diffusion", "kind": "ir_cg", "nx": 500, "ny": 387,
         "tol": 1e-10},
        # restarted GMRES with exact ILU(0) on an upwind operator, the
        # defaults (modified Gram-Schmidt)
        {"name": "gmres_ilu0_64", "kind": "gmres", "nx": 64, "ny": 64, "nz": 64,
         "peclet": 63.3, "restart": 50, "precond": "ilu0", "tol": 1e-10},
        # flexible GMRES with Jacobi on a small operator
        {"name": "fgmres_jacobi_24", "kind": "fgmres", "nx": 24, "ny": 21,
         "nz": 29, "peclet": 40.0, "restart": 30, "precond": "jacobi",
         "tol": 1e-10},
        # BiCGSTAB on the full-size upwind operator
        {"name": "bicgstab_128", "kind": "bicgstab", "nx": 128, "ny": 128,
         "nz": 128, "peclet": 63.3, "precond": "jacobi", "tol": 1e-10},
        # a new matrix every time step: ILU(0) of it, then its first use
        {"name": "ilu0_setup_96", "kind": "ilu0_setup", "nx": 96, "ny": 90,
         "nz": 85, "peclet": 30.0},
        # many small independent SPD systems at once
        {"name": "batched_256", "kind": "batched", "count": 256, "side_min": 32,
         "side_max": 96, "tol": 1e-8},
        # training of the learned inverse, its prediction and first use
        {"name": "spai_train_256", "kind": "spai", "side": 256, "count": 8,
         "batch": 4, "epochs": 2},
    ]


def _span(rng, lo, hi):
    """A whole number, spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["multiply", "spmv", "spmv", "cg", "cg", "ir_cg", "gmres",
                       "gmres", "fgmres", "bicgstab", "ilu0_setup", "batched",
                       "spai"])
    if kind in ("multiply", "spmv"):
        dtype = rng.choice(["f64", "f32"])
        m = rng.choice(["poisson2d", "poisson3d", "powerlaw", "diffusion"])
        c = {"kind": kind, "matrix": m, "dtype": dtype}
        if m == "poisson2d":
            c.update(nx=_span(rng, 24, 2000), ny=_span(rng, 24, 2000))
        elif m == "poisson3d":
            c.update(nx=_span(rng, 8, 192), ny=_span(rng, 8, 192),
                     nz=_span(rng, 8, 192))
        elif m == "powerlaw":
            c.update(n=_span(rng, 2000, 262144))
        else:
            c.update(nx=_span(rng, 24, 1000), ny=_span(rng, 24, 1000))
        return c
    if kind == "cg":
        if rng.random() < 0.5:
            return {"kind": "cg", "matrix": "poisson2d",
                    "nx": _span(rng, 24, 600), "ny": _span(rng, 24, 600),
                    "shift": rng.choice([0.01, 0.03, 0.1]), "tol": 1e-8}
        return {"kind": "cg", "matrix": "poisson3d", "nx": _span(rng, 12, 160),
                "ny": _span(rng, 12, 160), "nz": _span(rng, 12, 160), "tol": 1e-8}
    if kind == "ir_cg":
        return {"kind": "ir_cg", "nx": _span(rng, 40, 500),
                "ny": _span(rng, 40, 500), "tol": 1e-10}
    if kind in ("gmres", "fgmres", "bicgstab"):
        hi = {"gmres": 64, "fgmres": 64, "bicgstab": 110}[kind]
        c = {"kind": kind, "nx": _span(rng, 12, hi), "ny": _span(rng, 12, hi),
             "nz": _span(rng, 12, hi), "peclet": round(rng.uniform(10, 100), 1),
             "tol": 1e-10}
        c["precond"] = rng.choice(["ilu0", "jacobi"]) if kind == "gmres" else "jacobi"
        if kind != "bicgstab":
            c["restart"] = rng.choice([20, 30, 50])
        return c
    if kind == "ilu0_setup":
        return {"kind": kind, "nx": _span(rng, 16, 96), "ny": _span(rng, 16, 96),
                "nz": _span(rng, 16, 85), "peclet": round(rng.uniform(10, 100), 1)}
    if kind == "batched":
        lo = _span(rng, 12, 40)
        return {"kind": kind, "count": _span(rng, 16, 256), "side_min": lo,
                "side_max": lo + rng.randint(1, 50), "tol": 1e-8}
    return {"kind": "spai", "side": _span(rng, 32, 256), "count": 8,
            "batch": rng.choice([2, 4, 8]), "epochs": 2}


# ------------------------------------------------------------------ matrices

def _rng(seed, what):
    return np.random.default_rng([seed, what])


def _diffusion(ny, nx, rng, nine):
    """CSR arrays of a cell-centred diffusion operator with lognormal
    conductivities and Dirichlet walls, natural order: 5-point, or 9-point
    with the diagonal neighbours coupled at a quarter of the weight."""
    k = np.exp(rng.normal(0.0, 1.0, (ny, nx)))

    def link(a, b):
        return 2.0 * a * b / (a + b)

    w = np.zeros((9, ny, nx))  # (dy, dx) in column order, weights >= 0
    we = link(k[:, :-1], k[:, 1:])
    wn = link(k[:-1, :], k[1:, :])
    w[5][:, :-1] = we
    w[3][:, 1:] = we
    w[7][:-1, :] = wn
    w[1][1:, :] = wn
    if nine:
        ne = 0.25 * link(k[:-1, :-1], k[1:, 1:])
        nw = 0.25 * link(k[:-1, 1:], k[1:, :-1])
        w[8][:-1, :-1] = ne
        w[0][1:, 1:] = ne
        w[6][:-1, 1:] = nw
        w[2][1:, :-1] = nw
    wall = np.zeros((ny, nx))
    for edge in (np.s_[0, :], np.s_[-1, :], np.s_[:, 0], np.s_[:, -1]):
        wall[edge] += 2.0 * k[edge]
    diag = w.sum(0) + wall
    off = np.array([dy * nx + dx for dy in (-1, 0, 1) for dx in (-1, 0, 1)])
    vals = -w
    vals[4] = diag
    keep = (vals != 0.0).reshape(9, -1).T  # rows x 9, columns ascending
    cols = np.arange(ny * nx)[:, None] + off[None, :]
    rp = np.zeros(ny * nx + 1, np.int64)
    np.cumsum(keep.sum(1), out=rp[1:])
    return rp, cols[keep], vals.reshape(9, -1).T[keep]


def _csr_apply(rp, ci, v, x):
    """A x for a CSR matrix without empty rows, in 64 bits."""
    return np.add.reduceat(v * x[ci], rp[:-1])


def _powerlaw(n, seed):
    """Row and column numbers and values (on the GPU) of a matrix whose row
    lengths follow a power law between 4 and 4096 (mean about 44), columns
    uniform, the diagonal present; sorted, no duplicates."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    length = (4.0 / (1.0 - u) ** (1.0 / 0.9)).clamp(max=min(4096, n // 2)).long()
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), length)
    cols = torch.randint(0, n, rows.shape, generator=g, device="cuda")
    eye = torch.arange(n, device="cuda") * (n + 1)
    key = torch.unique(torch.cat([rows * n + cols, eye]))
    rows, cols = key // n, key % n
    vals = torch.rand(key.shape, generator=g, device="cuda",
                      dtype=torch.float64) * 2.0 - 1.0
    return rows, cols, vals


def _powerlaw_store(n, seed):
    rows, cols, vals = _powerlaw(n, seed)
    rp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return spk.CsrMatrix.from_host(n, n, rp.cpu().numpy(), cols.cpu().numpy(),
                                   vals.cpu().numpy())


def _velocity(c):
    """Upwind face terms of the velocity (1, 1/2, 1/4) at the case's Peclet
    number, as `spk.convdiff_3d` takes them."""
    v = np.array([1.0, 0.5, 0.25])
    v = c["peclet"] * v / np.linalg.norm(v)
    return tuple(float(a / (c[k] + 1)) for a, k in zip(v, ("nx", "ny", "nz")))


def _convdiff_apply(c, x):
    """The upwind operator (7-point, Dirichlet, unit diffusion) applied to x
    in 64 bits."""
    u = x.reshape(c["nz"], c["ny"], c["nx"])
    vel = _velocity(c)
    y = (6.0 + sum(vel)) * u
    for axis, a in zip((2, 1, 0), vel):
        lo = [slice(None)] * 3
        hi = [slice(None)] * 3
        lo[axis], hi[axis] = slice(None, -1), slice(1, None)
        lo, hi = tuple(lo), tuple(hi)
        y[hi] -= (1.0 + a) * u[lo]
        y[lo] -= u[hi]
    return y.reshape(-1)


def _matrix(c, seed):
    m = c["matrix"]
    if m == "poisson2d":
        return spk.poisson_2d(c["nx"], c["ny"], c.get("shift", 0.0))
    if m == "poisson3d":
        return spk.poisson_3d(c["nx"], c["ny"], c["nz"])
    if m == "powerlaw":
        return _powerlaw_store(c["n"], seed)
    rp, ci, v = _diffusion(c["ny"], c["nx"], _rng(seed, 1), True)
    return spk.CsrMatrix.from_host(c["nx"] * c["ny"], c["nx"] * c["ny"], rp, ci, v)


def _rows(c):
    if c.get("matrix") == "powerlaw":
        return c["n"]
    return c["nx"] * c["ny"] * c.get("nz", 1)


def _batch(c, seed):
    """The systems' sides, CSR arrays of the block diagonal and row offsets."""
    lo, hi, count = c["side_min"], c["side_max"], c["count"]
    sides = np.random.default_rng([lo, hi]).integers(lo, hi + 1, count)
    rng = _rng(seed, 2)
    rps, cis, vs, at, nnz = [np.zeros(1, np.int64)], [], [], 0, 0
    offsets = [0]
    for s in sides:
        rp, ci, v = _diffusion(int(s), int(s), rng, False)
        rps.append(rp[1:] + nnz)
        cis.append(ci + at)
        vs.append(v)
        at += int(s) ** 2
        nnz += len(ci)
        offsets.append(at)
    return (np.concatenate(rps), np.concatenate(cis), np.concatenate(vs),
            np.array(offsets, np.int64))


def _uniform(seed, what, n):
    return _rng(seed, what).uniform(-1.0, 1.0, n)


def _spai_params(seed):
    """Initial weights in the model's layout: W1[24][64] b1 W2[64][64] b2
    W3[64][9] b3, the output layer small."""
    rng = _rng(seed, 3)
    parts = [rng.uniform(-0.5, 0.5, 24 * 64), np.zeros(64),
             rng.uniform(-0.3, 0.3, 64 * 64), np.zeros(64),
             rng.uniform(-0.02, 0.02, 64 * 9), np.zeros(9)]
    return np.concatenate(parts).astype(np.float32)


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind in ("multiply", "spmv"):
        dt = np.float64 if c["dtype"] == "f64" else np.float32
        s["A"] = _matrix(c, seed)
        s["x"] = spk.DeviceVector.from_numpy(_uniform(seed, 4, _rows(c)), dt)
        if kind == "spmv":
            s["y"] = spk.DeviceVector.zeros(_rows(c), dt)
            s["out"] = _tensor(s["y"])
        # an FP32 product keeps an FP32 copy of the values, made once
        s["A"].spmv(s["x"], spk.DeviceVector.zeros(_rows(c), dt))
    elif kind == "cg":
        s["A"] = _matrix(c, seed)
        s["M"] = spk.jacobi(s["A"])
        s["b"] = spk.DeviceVector.from_numpy(_uniform(seed, 4, _rows(c)))
        s["cfg"] = spk.CGConfig(c["tol"], 20000, 20000)
    elif kind == "ir_cg":
        rp, ci, v = _diffusion(c["ny"], c["nx"], _rng(seed, 1), True)
        s["A"] = spk.CsrMatrix.from_host(_rows(c), _rows(c), rp, ci, v)
        s["M"] = spk.jacobi(s["A"])
        s["b"] = spk.DeviceVector.from_numpy(
            _csr_apply(rp, ci, v, _uniform(seed, 4, _rows(c))))
        s["cfg"] = spk.IrConfig(tolerance=c["tol"], max_outer=200,
                                inner_tolerance=1e-1, restart=0,
                                max_inner=100000,
                                inner_method=spk.IR_CG_RELIABLE)
    elif kind in ("gmres", "fgmres", "bicgstab"):
        s["A"] = spk.convdiff_3d(c["nx"], c["ny"], c["nz"], 1.0, *_velocity(c))
        s["M"] = (spk.ilu0 if c["precond"] == "ilu0" else spk.jacobi)(s["A"])
        s["b"] = spk.DeviceVector.from_numpy(
            _convdiff_apply(c, _uniform(seed, 4, _rows(c))))
        if kind == "bicgstab":
            s["cfg"] = spk.BicgstabConfig(c["tol"], 5000)
        else:
            s["cfg"] = spk.GmresConfig(c["tol"], c["restart"], 5000)
    elif kind == "ilu0_setup":
        s["A"] = spk.convdiff_3d(c["nx"], c["ny"], c["nz"], 1.0, *_velocity(c))
        s["r"] = spk.DeviceVector.from_numpy(_uniform(seed, 4, _rows(c)))
    elif kind == "batched":
        rp, ci, v, off = _batch(c, seed)
        n = int(off[-1])
        A = spk.CsrMatrix.from_host(n, n, rp, ci, v)
        s["B"] = spk.BatchedSystems.from_blocks(A, off)
        s["b"] = spk.DeviceVector.from_numpy(
            _csr_apply(rp, ci, v, _uniform(seed, 4, n)))
        s["cfg"] = spk.BatchConfig(tolerance=c["tol"], inner_tolerance=1e-2)
    elif kind == "spai":
        n = c["side"] ** 2
        s["mats"] = []
        for k in range(c["count"]):
            rp, ci, v = _diffusion(c["side"], c["side"], _rng(seed, 10 + k), True)
            s["mats"].append(spk.CsrMatrix.from_host(n, n, rp, ci, v))
        s["params"] = _spai_params(seed)
        s["r"] = spk.DeviceVector.from_numpy(_uniform(seed, 4, n))
    return s


# ------------------------------------------------------------------ run

def run(state):
    s = state
    c, kind = s["case"], s["case"]["kind"]
    if kind == "multiply":
        return _tensor(spk.multiply(s["A"], s["x"]))
    if kind == "spmv":
        s["A"].spmv(s["x"], s["y"])
        return s["out"]
    if kind == "ilu0_setup":
        F = spk.ilu0(s["A"])
        z = spk.DeviceVector(F.n)
        spk.ilu_apply(F, s["r"], z)
        return _tensor(z)
    if kind == "spai":
        model = spk.SpaiModel(0)
        model.params = s["params"]
        hist = model.train(s["mats"], epochs=c["epochs"], learning_rate=2e-3,
                           batch_matrices=c["batch"], shuffle_seed=7)
        M = model.preconditioner(s["mats"][0])
        z = spk.DeviceVector(s["r"].n)
        M.apply(s["r"], z)
        return {"loss": hist, "params": model.params, "z": _tensor(z)}
    x = spk.DeviceVector.zeros(s["b"].n)
    if kind == "cg":
        spk.conjugate_gradient(s["b"], x, s["cfg"], s["A"], s["M"])
    elif kind == "ir_cg":
        spk.ir_solve(s["b"], x, s["cfg"], s["A"], s["M"])
    elif kind == "gmres":
        spk.gmres(s["b"], x, s["cfg"], s["A"], spk.identity, s["M"])
    elif kind == "fgmres":
        spk.fgmres(s["b"], x, s["cfg"], s["A"], s["M"])
    elif kind == "bicgstab":
        spk.bicgstab(s["b"], x, s["cfg"], s["A"], s["M"])
    elif kind == "batched":
        s["B"].solve(s["cfg"], s["b"], x)
    return _tensor(x)


# ------------------------------------------------------------------ work

def _nnz(c):
    if c.get("matrix") == "powerlaw":
        # the truncated law's mean length, and the diagonal
        top = min(4096, c["n"] // 2)
        return int(c["n"] * (1 + 9 * 4 ** 0.9 * (top ** 0.1 - 4 ** 0.1)
                             + top * (4 / top) ** 0.9))
    if "nz" in c:
        a, b, d = c["nx"], c["ny"], c["nz"]
        return 7 * a * b * d - 2 * (a * b + b * d + a * d)
    if c.get("matrix") == "poisson2d":
        return 5 * c["nx"] * c["ny"] - 2 * (c["nx"] + c["ny"])
    return 9 * c["nx"] * c["ny"]


def work(case):
    """Bytes and operations of one pass.  A solver's iterations cannot be
    known beforehand: their number is estimated from the size (about what
    the method takes), and one iteration reads the matrix once and each of
    its vectors once."""
    c, kind = case, case["kind"]
    if kind in ("multiply", "spmv"):
        w = 8 if c["dtype"] == "f64" else 4
        n, nnz = _rows(c), _nnz(c)
        return {"bytes": nnz * (w + 4) + 4 * n + 2 * w * n, "flops": 2 * nnz}
    if kind == "batched":
        mean = (c["side_min"] + c["side_max"]) / 2
        n, it = c["count"] * mean ** 2, 5.0 * mean
        return {"bytes": it * n * (5 * 8 + 44), "flops": it * n * 22}
    if kind == "spai":
        n = c["side"] ** 2
        rows = n * c["count"] * c["epochs"]
        return {"bytes": rows * 9 * 12 + n * 9 * 28,
                "flops": rows * 3 * 12416 + n * 12416}
    n, nnz = _rows(c), _nnz(c)
    spmv = nnz * 12 + 4 * n + 16 * n
    if kind == "ilu0_setup":
        # the matrix read, the factors written and read once by the apply
        return {"bytes": 3 * (nnz * 12 + 4 * n) + 3 * 8 * n, "flops": 8 * nnz}
    if kind == "cg":
        if c["matrix"] == "poisson2d":
            it = 24.0 / math.sqrt(c["shift"])
        else:
            it = 3.4 * (c["nx"] * c["ny"] * c["nz"]) ** (1 / 3)
        return {"bytes": it * (spmv + 88 * n), "flops": it * (2 * nnz + 10 * n)}
    if kind == "ir_cg":
        it = 6.0 * max(c["nx"], c["ny"])
        return {"bytes": it * (nnz * 8 + 4 * n + 52 * n), "flops": it * (2 * nnz + 10 * n)}
    mean = n ** (1 / 3)
    if kind == "bicgstab":
        it = 1.2 * mean
        return {"bytes": it * (2 * spmv + 120 * n), "flops": it * (4 * nnz + 20 * n)}
    it = (0.8 if c["precond"] == "ilu0" else 6.0) * mean
    basis = min(it, c["restart"]) / 2  # vectors a step reads on average
    per = spmv + (nnz * 12 + 24 * n if c["precond"] == "ilu0" else 24 * n)
    return {"bytes": it * (per + 8 * n * basis),
            "flops": it * (4 * nnz + 4 * n * basis)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("multiply", "spmv"):
        # sums of up to 4096 products in another order
        return {"rel": 1e-15} if case["dtype"] == "f64" else {"rel": 8e-7}
    if kind == "ilu0_setup":
        return {"rel": 1e-14}
    if kind == "spai":
        return {"rel": 1e-2, "max": 0.5}
    # a solver's answer depends on where its residual test ends it: two runs
    # with sums in another order stop at residuals of the same size
    return {"rel": 1e-6, "max": 2e-5}


# ------------------------------------------------------------------ exact

def _path_basis(n, dirichlet):
    """Orthonormal eigenvectors (columns) and eigenvalues of the 1D path:
    2 on the diagonal (Dirichlet) or the degree (free ends)."""
    j = torch.arange(n, dtype=torch.float64)
    if dirichlet:
        k = j + 1
        v = torch.sin(math.pi * (j[:, None] + 1) * k[None, :] / (n + 1))
        v = v * math.sqrt(2.0 / (n + 1))
        return v, 2.0 - 2.0 * torch.cos(math.pi * k / (n + 1))
    v = torch.cos(math.pi * (j[:, None] + 0.5) * j[None, :] / n)
    return v / v.norm(dim=0), 2.0 - 2.0 * torch.cos(math.pi * j / n)


def _poisson_solve(c, b):
    """The Poisson system solved by its eigenvectors, axis by axis."""
    dims = [c[k] for k in ("nz", "ny", "nx") if k in c]
    u = torch.from_numpy(b).reshape(dims)
    basis = [_path_basis(n, "nz" in c) for n in dims]
    for inverse in (True, False):
        for axis, (v, _) in enumerate(basis):
            u = torch.movedim(torch.movedim(u, axis, -1) @ (v if inverse else v.T),
                              -1, axis)
        if inverse:
            lam = torch.zeros(dims, dtype=torch.float64) + c.get("shift", 0.0)
            for axis, (_, e) in enumerate(basis):
                lam = lam + e.reshape([-1 if a == axis else 1 for a in range(len(dims))])
            u = u / lam
    return u.reshape(-1)


def _ilu0_apply(c, r):
    """z = U^-1 L^-1 r for ILU(0) of the upwind operator: a 7-point pattern
    has no fill between its neighbours, so only the pivots change.  Cells of
    one plane i + j + k = const are independent."""
    vel = _velocity(c)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    plane = (i + j + k).reshape(-1)
    order = np.argsort(plane, kind="stable")
    cuts = np.searchsorted(plane[order], np.arange(nx + ny + nz - 1))
    planes = np.split(order, cuts[1:])
    # one layer of padding on every side: neighbours outside are dropped by
    # a zero weight
    n, step = nx * ny * nz, (1, nx, nx * ny)
    inside = [(q.reshape(-1) > 0, q.reshape(-1) < m - 1)
              for q, m in ((i, nx), (j, ny), (k, nz))]
    d, y, z = np.zeros(n), np.zeros(n), np.zeros(n)
    for p in planes:
        piv, s = np.full(len(p), 6.0 + sum(vel)), r[p].copy()
        for a, st, (low, _) in zip(vel, step, inside):
            at = p[low[p]]
            lik = -(1.0 + a) / d[at - st]
            piv[low[p]] -= lik * -1.0
            s[low[p]] -= lik * y[at - st]
        d[p], y[p] = piv, s
    for p in reversed(planes):
        s = y[p].copy()
        for st, (_, high) in zip(step, inside):
            at = p[high[p]]
            s[high[p]] -= -1.0 * z[at + st]
        z[p] = s / d[p]
    return z


class _Spai:
    """The learned inverse's forward pass and loss in 64 bits."""

    def __init__(self, rp, ci, v):
        rp, ci, v = (torch.from_numpy(a).to(_device()) for a in (rp, ci, v))
        n, ln = len(rp) - 1, rp.diff()
        self.n, self.v, self.col = n, v, ci
        self.row = torch.repeat_interleave(torch.arange(n, device=v.device), ln)
        dpos = torch.nonzero(ci == self.row).reshape(-1)
        # the entry's place from the diagonal (slot 4) on
        self.slot = torch.arange(len(ci), device=v.device) - dpos[self.row] + 4
        self.diag = v[dpos]
        rsum = self._rows(v)
        x = torch.zeros(3, n, 9, dtype=torch.float64, device=v.device)
        di, dj = self.diag[self.row], self.diag[ci]
        x[0, self.row, self.slot] = v / di
        x[1, self.row, self.slot] = (dj - di) / (dj + di)
        x[2, self.row, self.slot] = rsum[ci] / dj
        keep = [0, 1, 2, 3, 5, 6, 7, 8]
        self.x = torch.cat([x[f][:, keep] for f in range(3)], 1)
        # (M A) on its own pattern: entry k of M times the entries of row ci[k]
        cnt = ln[ci]
        self.outer = torch.repeat_interleave(torch.arange(len(ci), device=v.device), cnt)
        first = rp[ci] - (torch.cumsum(cnt, 0) - cnt)
        self.inner = first[self.outer] + torch.arange(len(self.outer), device=v.device)
        key, self.where = torch.unique(self.row[self.outer] * n + ci[self.inner],
                                       return_inverse=True)
        self.unit = (key // n == key % n).double()

    def _rows(self, e):
        return torch.zeros(self.n, dtype=torch.float64, device=e.device).index_add(
            0, self.row, e)

    def inverse(self, p):
        w1, b1, w2, b2, w3, b3 = p
        h = torch.relu(torch.relu(self.x @ w1 + b1) @ w2 + b2)
        y = (h @ w3 + b3)[self.row, self.slot] + (self.slot == 4)
        return y / self.diag[self.row]

    def loss_sum(self, p):
        m = self.inverse(p)
        ma = torch.zeros_like(self.unit).index_add(
            0, self.where, m[self.outer] * self.v[self.inner])
        return ((self.unit - ma) ** 2).sum()

    def apply(self, p, r):
        return self._rows(self.inverse(p) * r[self.col])


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _mix(seed, k):
    mask = (1 << 64) - 1
    z = (seed + (k + 1) * 0x9E3779B97F4A7C15) & mask
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
    return z ^ (z >> 31)


def _spai_exact(c, seed):
    """Adam on the mean row loss over batches of matrices, shuffled each
    epoch (Fisher-Yates on splitmix64 draws), then z = M r."""
    sp = [_Spai(*_diffusion(c["side"], c["side"], _rng(seed, 10 + k), True))
          for k in range(c["count"])]
    flat = torch.from_numpy(_spai_params(seed).astype(np.float64)).to(_device())
    sizes = [24 * 64, 64, 64 * 64, 64, 64 * 9, 9]
    shapes = [(24, 64), (64,), (64, 64), (64,), (64, 9), (9,)]

    def split(f):
        return [q.reshape(s) for q, s in zip(torch.split(f, sizes), shapes)]

    m1, m2 = torch.zeros_like(flat), torch.zeros_like(flat)
    hist, step = [], 0
    for e in range(c["epochs"]):
        order = list(range(c["count"]))
        for k in range(c["count"] - 1, 0, -1):
            q = _mix(7, e * c["count"] + k) % (k + 1)
            order[k], order[q] = order[q], order[k]
        for b in range(0, c["count"], c["batch"]):
            part = [sp[k] for k in order[b:b + c["batch"]]]
            f = flat.clone().requires_grad_(True)
            loss = sum(a.loss_sum(split(f)) for a in part) / sum(a.n for a in part)
            (g,) = torch.autograd.grad(loss, f)
            hist.append(loss.item())
            step += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            flat = flat - 2e-3 * (m1 / (1 - 0.9 ** step)) / (
                torch.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)
    z = sp[0].apply(split(flat),
                    torch.from_numpy(_uniform(seed, 4, sp[0].n)).to(_device()))
    return {"loss": np.array(hist), "params": flat.cpu(), "z": z}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("multiply", "spmv"):
        x = torch.from_numpy(_uniform(seed, 4, _rows(c)))
        if c["dtype"] == "f32":  # the product's inputs are rounded to FP32
            x = x.float().double()
        m = c["matrix"]
        if m == "powerlaw":
            rows, cols, vals = (t.cpu() for t in _powerlaw(c["n"], seed))
            if c["dtype"] == "f32":
                vals = vals.float().double()
            return torch.zeros(c["n"], dtype=torch.float64).index_add(
                0, rows, vals * x[cols])
        if m == "diffusion":
            rp, ci, v = _diffusion(c["ny"], c["nx"], _rng(seed, 1), True)
            if c["dtype"] == "f32":
                v = v.astype(np.float32).astype(np.float64)
            return _csr_apply(rp, ci, v, x.numpy())
        dims = [c[k] for k in ("nz", "ny", "nx") if k in c]
        u = x.reshape(dims)
        y = (6.0 if m == "poisson3d" else c.get("shift", 0.0)) * u
        for axis, size in enumerate(dims):
            lo, hi = u.narrow(axis, 0, size - 1), u.narrow(axis, 1, size - 1)
            if m == "poisson2d":  # the diagonal is the number of neighbours
                y.narrow(axis, 1, size - 1).add_(hi)
                y.narrow(axis, 0, size - 1).add_(lo)
            y.narrow(axis, 1, size - 1).sub_(lo)
            y.narrow(axis, 0, size - 1).sub_(hi)
        return y.reshape(-1)
    if kind == "cg":
        return _poisson_solve(c, _uniform(seed, 4, _rows(c)))
    if kind == "ilu0_setup":
        return _ilu0_apply(c, _uniform(seed, 4, _rows(c)))
    if kind == "batched":
        return _uniform(seed, 4, int(_batch(c, seed)[3][-1]))
    if kind == "spai":
        return _spai_exact(c, seed)
    return _uniform(seed, 4, _rows(c))
