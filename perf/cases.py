"""The calls that programs make of this library, as measured cases.

Every case is one public call (or the few calls of a user's own loop body) on
a system that the program keeps resident: sparse products, vector BLAS, the
Krylov solvers with their preconditioners, the batched solver and the assembly
of a matrix from triplets.  Matrices are the grids and random patterns of the
repository's own benchmark; vectors are drawn from the seed.  ``exact`` states
the same results in 64-bit torch / numpy without the library.

A case is a dict: ``kind`` names the call, ``matrix`` the pattern, ``nx`` /
``ny`` / ``nz`` or ``rows`` / ``cols`` / ``mean`` its size, ``dtype`` the value
type, ``tuned`` whether the program ran the SpMV autotuner once after upload
(the C++ headers never do), ``tol`` the relative residual a solver stops at.
"""
import math

import numpy as np
import torch

import monolish_amd as m

_CTX = None
_DEV = "cuda"


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = m.Context(0)
    return _CTX


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # a small system inside a user's own loop: one SpMV, one dot, one
        # axpyz and one norm; launches and the two host scalars count
        {"name": "loop_poisson2d_64", "kind": "loop", "matrix": "poisson2d", "nx": 64, "ny": 64,
         "dtype": "f64"},
        # the headline product: a 3D 7-point operator, autotuned once
        {"name": "matvec_stencil7_192", "kind": "matvec", "matrix": "stencil7", "nx": 192,
         "ny": 192, "nz": 192, "dtype": "f64", "tuned": True},
        # an FP32 27-point operator on a ragged grid as the C++ headers run
        # it: the plan made at upload
        {"name": "matvec_stencil27_f32", "kind": "matvec", "matrix": "stencil27", "nx": 101,
         "ny": 97, "nz": 89, "dtype": "f32", "tuned": False},
        # irregular rows, scattered columns (graph and contact problems)
        {"name": "matvec_lognormal_1m", "kind": "matvec", "matrix": "lognormal", "rows": 1000000,
         "cols": 1000000, "mean": 32, "dtype": "f64", "tuned": True},
        # the transposed product of a rectangular matrix (least squares)
        {"name": "matvec_t_rect_f32", "kind": "matvec_t", "matrix": "lognormal", "rows": 400000,
         "cols": 250000, "mean": 20, "dtype": "f32", "tuned": False},
        # assembly: shuffled triplets with duplicates to a device CRS, and
        # the CRS back on the host
        {"name": "assemble_stencil7", "kind": "assemble", "matrix": "stencil7", "nx": 112,
         "ny": 104, "nz": 96, "dtype": "f64"},
        # the small Krylov solve: Jacobi-PCG, latency of an iteration
        {"name": "cg_poisson2d_256", "kind": "cg", "matrix": "poisson2d", "nx": 256, "ny": 256,
         "dtype": "f64", "tol": 1e-10},
        # the large Krylov solve: mixed precision on a 27-point operator
        {"name": "mixed_cg_stencil27_128", "kind": "mixed_cg", "matrix": "stencil27", "nx": 128,
         "ny": 128, "nz": 128, "dtype": "f64", "tol": 1e-10},
        # a nonsymmetric system
        {"name": "bicgstab_convdiff_500", "kind": "bicgstab", "matrix": "convdiff", "nx": 500,
         "ny": 500, "peclet": 20.0, "dtype": "f64", "tol": 1e-10},
        # many uneven small systems in one call
        {"name": "batch_cg_512", "kind": "batch", "matrix": "mmatrix", "systems": 512,
         "nmin": 500, "nmax": 20000, "dtype": "f64", "tol": 1e-10},
        # triangular preconditioners: narrow levels (2D) and wide ones (3D)
        {"name": "sor_cg_poisson2d_256", "kind": "sor_cg", "matrix": "poisson2d", "nx": 256,
         "ny": 256, "dtype": "f64", "tol": 1e-8},
        {"name": "ic_cg_stencil27_96", "kind": "ic_cg", "matrix": "stencil27", "nx": 96, "ny": 96,
         "nz": 96, "dtype": "f64", "tol": 1e-8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    dtype = rng.choice(["f64", "f64", "f32"])
    tuned = rng.random() < 0.5
    kind = rng.choice(["loop", "matvec", "matvec", "matvec_t", "assemble", "cg", "cg", "mixed_cg",
                       "bicgstab", "batch", "sor_cg", "ic_cg", "ilu_cg"])
    if kind == "loop":
        return {"kind": kind, "matrix": "poisson2d", "nx": _log(rng, 8, 700),
                "ny": _log(rng, 8, 700), "dtype": dtype}
    if kind == "matvec":
        what = rng.choice(["poisson2d", "stencil7", "stencil27", "lognormal"])
        c = {"kind": kind, "matrix": what, "dtype": dtype, "tuned": tuned}
        if what == "poisson2d":
            return dict(c, nx=_log(rng, 20, 2500), ny=_log(rng, 20, 2500))
        if what == "lognormal":
            rows = _log(rng, 2000, 1000000)
            return dict(c, rows=rows, cols=_log(rng, max(2000, rows // 4), min(1000000, rows * 4)),
                        mean=rng.randint(4, 32))
        hi = 190 if what == "stencil7" else 125
        return dict(c, nx=_log(rng, 10, hi), ny=_log(rng, 10, hi), nz=_log(rng, 10, hi))
    if kind == "matvec_t":
        rows = _log(rng, 2000, 500000)
        return {"kind": kind, "matrix": "lognormal", "rows": rows,
                "cols": _log(rng, max(2000, rows // 4), min(500000, rows * 4)),
                "mean": rng.randint(4, 24), "dtype": dtype, "tuned": False}
    if kind == "assemble":
        return {"kind": kind, "matrix": "stencil7", "nx": _log(rng, 16, 110),
                "ny": _log(rng, 16, 110), "nz": _log(rng, 16, 100), "dtype": dtype}
    if kind == "cg":
        if rng.random() < 0.5:
            return {"kind": kind, "matrix": "poisson2d", "nx": _log(rng, 20, 500),
                    "ny": _log(rng, 20, 500), "dtype": "f64", "tol": 1e-10}
        return {"kind": kind, "matrix": "stencil7", "nx": _log(rng, 12, 120),
                "ny": _log(rng, 12, 120), "nz": _log(rng, 12, 120), "dtype": "f64", "tol": 1e-10}
    if kind == "mixed_cg":
        return {"kind": kind, "matrix": "stencil27", "nx": _log(rng, 24, 125),
                "ny": _log(rng, 24, 125), "nz": _log(rng, 24, 125), "dtype": "f64", "tol": 1e-10}
    if kind == "bicgstab":
        return {"kind": kind, "matrix": "convdiff", "nx": _log(rng, 30, 490),
                "ny": _log(rng, 30, 490), "peclet": round(rng.uniform(1, 50), 1), "dtype": "f64",
                "tol": 1e-10}
    if kind == "batch":
        return {"kind": kind, "matrix": "mmatrix", "systems": _log(rng, 16, 500), "nmin": 500,
                "nmax": _log(rng, 2000, 20000), "dtype": "f64", "tol": 1e-10}
    if kind == "sor_cg":
        return {"kind": kind, "matrix": "poisson2d", "nx": _log(rng, 24, 250),
                "ny": _log(rng, 24, 250), "dtype": "f64", "tol": 1e-8}
    if rng.random() < 0.5:
        return {"kind": kind, "matrix": "poisson2d", "nx": _log(rng, 24, 250),
                "ny": _log(rng, 24, 250), "dtype": "f64", "tol": 1e-8}
    return {"kind": kind, "matrix": "stencil27", "nx": _log(rng, 16, 95), "ny": _log(rng, 16, 95),
            "nz": _log(rng, 16, 95), "dtype": "f64", "tol": 1e-8}


# ---------------------------------------------------------------- matrices --
def _np_dtype(case):
    return np.float64 if case["dtype"] == "f64" else np.float32


def _t_dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(1000003 * int(seed) + 17)


def _uniform(n, g):
    return torch.rand(n, generator=g, device=_DEV, dtype=torch.float64) * 2 - 1


def _grid(dims, stencil):
    """CRS (row_ptr, col, val) of a constant-coefficient stencil on a grid,
    dims slowest first, stencil = [(offset tuple, value)] in column order."""
    n = math.prod(dims)
    i = torch.arange(n, device=_DEV)
    coord, rest = [], i
    for d in reversed(dims):
        coord.insert(0, rest % d)
        rest = rest // d
    keep = torch.empty((n, len(stencil)), dtype=torch.bool, device=_DEV)
    shift = []
    for k, (off, _) in enumerate(stencil):
        ok = torch.ones(n, dtype=torch.bool, device=_DEV)
        s = 0
        for c, o, d in zip(coord, off, dims):
            ok &= (c + o >= 0) & (c + o < d)
            s = s * d + o
        keep[:, k] = ok
        shift.append(s)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=_DEV)
    rp[1:] = keep.sum(1).cumsum(0)
    col = (i[:, None] + torch.tensor(shift, device=_DEV)[None, :])[keep].to(torch.int32)
    val = torch.tensor([v for _, v in stencil], dtype=torch.float64, device=_DEV)
    val = val[None, :].expand(n, -1)[keep]
    return rp, col, val


def _matrix(case, g):
    """(rows, cols, row_ptr int64, col int32, val float64) on the device."""
    what = case["matrix"]
    if what == "lognormal":
        rows, cols, mean = case["rows"], case["cols"], case["mean"]
        length = torch.empty(rows, device=_DEV, dtype=torch.float64)
        length.log_normal_(math.log(mean) - 0.5, 1.0, generator=g)
        length = length.round().clamp(1, min(2048, cols)).to(torch.int64)
        row = torch.repeat_interleave(torch.arange(rows, device=_DEV), length)
        col = torch.randint(cols, (row.numel(),), generator=g, device=_DEV)
        key = torch.unique(row * cols + col)  # ascending columns, none twice
        row, col = key // cols, key % cols
        rp = torch.zeros(rows + 1, dtype=torch.int64, device=_DEV)
        rp[1:] = torch.bincount(row, minlength=rows).cumsum(0)
        return rows, cols, rp, col.to(torch.int32), _uniform(key.numel(), g)
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    if what == "poisson2d":
        dims = (ny, nx)
        st = [((-1, 0), -1.0), ((0, -1), -1.0), ((0, 0), 4.0), ((0, 1), -1.0), ((1, 0), -1.0)]
    elif what == "convdiff":
        c = case["peclet"] / (max(nx, ny) + 1)
        dims = (ny, nx)
        st = [((-1, 0), -1.0), ((0, -1), -1.0 - c), ((0, 0), 4.0 + c), ((0, 1), -1.0),
              ((1, 0), -1.0)]
    else:
        dims = (nz, ny, nx)
        st = []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    o = (dz, dy, dx)
                    if what == "stencil27" or abs(dz) + abs(dy) + abs(dx) <= 1:
                        centre = 26.01 if what == "stencil27" else 6.0
                        st.append((o, centre if o == (0, 0, 0) else -1.0))
    rp, col, val = _grid(dims, st)
    n = math.prod(dims)
    return n, n, rp, col, val


def _sizes(case):
    r = np.random.default_rng(9000 + case["systems"])
    return np.floor(np.exp(r.uniform(math.log(case["nmin"]), math.log(case["nmax"]),
                                     case["systems"]))).astype(np.int64)


def _batch(case, g):
    """Independent SPD M-matrices as one block-diagonal CRS: 5-15 random
    off-diagonals a row U[-1,0), symmetrised, diagonal = their sum + 0.5."""
    sizes = torch.from_numpy(_sizes(case)).to(_DEV)
    n = int(sizes.sum())
    first = sizes.cumsum(0) - sizes
    size_of = torch.repeat_interleave(sizes, sizes)
    base = torch.repeat_interleave(first, sizes)
    k = torch.randint(5, 16, (n,), generator=g, device=_DEV)
    row = torch.repeat_interleave(torch.arange(n, device=_DEV), k)
    u = torch.rand(row.numel(), generator=g, device=_DEV, dtype=torch.float64)
    col = base[row] + (u * size_of[row]).to(torch.int64)
    off = row != col
    row, col = row[off], col[off]
    key = torch.unique(torch.minimum(row, col) * n + torch.maximum(row, col))
    # multiples of 2^-21: the diagonal's sums are exact in any order
    v = torch.randint(1, 1 << 20, (key.numel(),), generator=g, device=_DEV).double() * -2.0 ** -21
    lo, hi = key // n, key % n
    diag = torch.zeros(n, dtype=torch.float64, device=_DEV).index_add_(0, lo, -v)
    diag = diag.index_add_(0, hi, -v) + 0.5
    here = torch.arange(n, device=_DEV)
    row, col = torch.cat([lo, hi, here]), torch.cat([hi, lo, here])
    order = torch.argsort(row * n + col)
    val = torch.cat([v, v, diag])[order]
    row, col = row[order], col[order]
    rp = torch.zeros(n + 1, dtype=torch.int64, device=_DEV)
    rp[1:] = torch.bincount(row, minlength=n).cumsum(0)
    return sizes.cpu().numpy(), first.cpu().numpy(), rp, col, val


def _triplets(case, seed):
    """Shuffled host triplets of the matrix with 5 % of them given twice
    (another value; the later one holds)."""
    g = _gen(seed)
    rows, cols, rp, col, _ = _matrix(case, g)
    row = torch.repeat_interleave(torch.arange(rows, device=_DEV), rp[1:] - rp[:-1])
    twice = torch.randint(col.numel(), (col.numel() // 20,), generator=g, device=_DEV)
    pick = torch.cat([torch.arange(col.numel(), device=_DEV), twice])
    pick = pick[torch.randperm(pick.numel(), generator=g, device=_DEV)]
    val = _uniform(pick.numel(), g).to(_t_dtype(case))
    return (rows, cols, row[pick].to(torch.int32).cpu().numpy(), col[pick].cpu().numpy(),
            val.cpu().numpy())


# ----------------------------------------------------------------- prepare --
class _Buffer:
    def __init__(self, v):
        self.vector = v
        self.__cuda_array_interface__ = {"shape": (v.size,), "typestr": v.dtype.str,
                                         "data": (v.device_ptr, False), "version": 2}


def _tensor(v):
    """The vector's device memory as a torch tensor."""
    return torch.as_tensor(_Buffer(v), device=_DEV)


def _crs(case, rows, cols, rp, col, val):
    return m.CRS(_ctx(), rows, cols, rp.to(torch.int32).cpu().numpy(), col.cpu().numpy(),
                 val.to(_t_dtype(case)).cpu().numpy())


def _vec(t, dt):
    return m.Vector(_ctx(), t.cpu().numpy(), dtype=dt)


def prepare(case, seed):
    kind, dt = case["kind"], _np_dtype(case)
    if kind == "assemble":
        return {"case": case, "triplets": _triplets(case, seed)}
    g = _gen(seed)
    s = {"case": case}
    if kind == "batch":
        sizes, first, rp, col, val = _batch(case, g)
        n = int(sizes.sum())
        b = _uniform(n, g)
        rp, col, val = rp.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy()
        s["b"], s["x"] = _vec(b, dt), m.Vector(_ctx(), n=n, dtype=dt)
        s["A"], s["bs"], s["xs"] = [], [], []
        for r0, k in zip(first.tolist(), sizes.tolist()):
            e0, e1 = rp[r0], rp[r0 + k]
            s["A"].append(m.CRS(_ctx(), k, k, rp[r0:r0 + k + 1] - e0, col[e0:e1] - r0, val[e0:e1]))
            s["bs"].append(s["b"].view(r0, k))
            s["xs"].append(s["x"].view(r0, k))
        s["out"] = _tensor(s["x"])
        return s
    rows, cols, rp, col, val = _matrix(case, g)
    s["A"] = A = _crs(case, rows, cols, rp, col, val)
    if case.get("tuned"):
        A.autotune(reps=20)
    nin, nout = (rows, cols) if kind == "matvec_t" else (cols, rows)
    s["b"] = _vec(_uniform(nin, g), dt)
    s["x"] = m.Vector(_ctx(), n=nout, dtype=dt)
    s["out"] = _tensor(s["x"])
    if kind == "loop":
        s["z"] = m.Vector(_ctx(), n=rows, dtype=dt)
        s["out2"] = _tensor(s["z"])
    elif kind not in ("matvec", "matvec_t"):
        # the C++ headers take an absolute tolerance, as the program states it
        s["tol"] = case["tol"] * m.nrm2(s["b"])
    return s


# --------------------------------------------------------------------- run --
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "assemble":
        rows, cols, r, c, v = s["triplets"]
        A = m.CRS.from_coo(_ctx(), rows, cols, r, c, v, sort=2)
        out = A.download()
        A.free()
        return out
    A, b, x = s["A"], s["b"], s["x"]
    if kind == "matvec":
        m.matvec(A, b, x)
        return s["out"]
    if kind == "matvec_t":
        m.matvec_t(A, b, x)
        return s["out"]
    if kind == "loop":
        m.matvec(A, b, x)
        d = m.dot(b, x)
        m.axpyz(-0.125, x, b, s["z"])
        return s["out"], s["out2"], d, m.nrm2(s["z"])
    x.fill(0.0)
    if kind == "batch":
        m.batch_solve(_ctx(), m.METHOD_CG, A, s["xs"], s["bs"], tol=case["tol"],
                      tol_is_relative=True, precond=m.PRECOND_JACOBI)
    elif kind == "mixed_cg":
        m.mixed_cg(A, x, b, tol=case["tol"], tol_is_relative=True, delta=1e-3)
    elif kind == "bicgstab":
        m.bicgstab(A, x, b, tol=s["tol"], precond=m.PRECOND_JACOBI, mode=m.MODE_FUSED)
    else:
        pre = {"cg": m.PRECOND_JACOBI, "sor_cg": m.PRECOND_SOR, "ic_cg": m.PRECOND_IC,
               "ilu_cg": m.PRECOND_ILU}[kind]
        m.cg(A, x, b, tol=s["tol"], precond=pre)
    return s["out"]


# -------------------------------------------------------------------- work --
def _entries(case):
    """(rows, cols, entries), closely."""
    what = case["matrix"]
    if what == "lognormal":
        return case["rows"], case["cols"], case["rows"] * case["mean"]
    if what == "mmatrix":
        lo, hi = case["nmin"], case["nmax"]
        n = case["systems"] * (hi - lo) / math.log(hi / lo)
        return n, n, 21 * n
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    n = nx * ny * nz
    if what in ("poisson2d", "convdiff"):
        return n, n, 5 * n - 2 * nx - 2 * ny
    if what == "stencil7":
        return n, n, 7 * n - 2 * (nx * ny + ny * nz + nx * nz)
    return n, n, (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)


def _iterations(case):
    """About how many iterations the solver needs for this tolerance."""
    kind, what = case["kind"], case["matrix"]
    if what == "mmatrix":
        return 26
    side = max(case["nx"], case["ny"], case.get("nz", 1))
    digits = -math.log10(case["tol"]) / 10
    jacobi = {"poisson2d": 3.4, "convdiff": 2.0, "stencil7": 3.0, "stencil27": 2.2}[what] * side
    return max(1, round(digits * jacobi * {"sor_cg": 0.6, "ic_cg": 0.35, "ilu_cg": 0.35}.get(kind, 1)))


def work(case):
    """One pass.  A solver reads the system once and writes x once as long as
    its matrix and vectors fit the chip's 256 MB last-level cache; beyond that
    every iteration has to stream them (at FP32 sizes in mixed precision)."""
    kind = case["kind"]
    sv = 8 if case["dtype"] == "f64" else 4
    rows, cols, nnz = _entries(case)
    if kind == "assemble":
        # triplets read once; row_ptr, columns and values written once
        return {"bytes": 1.05 * nnz * (8 + sv) + nnz * (4 + sv) + 4 * (rows + 1), "flops": 0}
    matrix = nnz * (4 + sv) + 4 * (rows + 1)
    once = matrix + sv * (rows + cols)
    if kind in ("matvec", "matvec_t"):
        return {"bytes": once, "flops": 2 * nnz}
    if kind == "loop":
        return {"bytes": once + sv * rows, "flops": 2 * nnz + 6 * rows}
    it = _iterations(case)
    per = 2 * nnz + 10 * rows
    if kind == "bicgstab":
        per = 4 * nnz + 20 * rows
    elif kind in ("sor_cg", "ic_cg", "ilu_cg"):
        per += 2 * nnz
    wide = 4 if kind == "mixed_cg" else sv
    stream = nnz * (4 + wide) + 4 * (rows + 1) + 7 * wide * rows  # x, r, p, q, z and the scale
    if stream <= 256 << 20:
        return {"bytes": once, "flops": it * per}
    return {"bytes": once + it * stream, "flops": it * per}


# --------------------------------------------------------------- tolerance --
def tolerance(case):
    """Products and sums: rounding of sums in another order.  Solutions: two
    correct solves stop at the same residual and differ by up to the
    condition number times it."""
    if case["kind"] == "assemble":
        return "exact"
    if case["kind"] in ("loop", "matvec", "matvec_t"):
        return {"rel": 2e-15 if case["dtype"] == "f64" else 1e-6}
    return {"rel": 6e-8 if case["tol"] < 1e-9 else 2e-6}


# ------------------------------------------------------------------- exact --
def _apply(rp, col, val, rows):
    A = torch.sparse_csr_tensor(rp, col.to(torch.int64), val, size=(rows, rows))
    return lambda x: torch.mv(A, x)


def _cg(mul, d, b):
    """Jacobi-PCG in 64 bits to the rounding level."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / d
    p, zr, stop = z.clone(), torch.dot(z, r), 1e-14 * float(b.norm())
    for k in range(20000):
        q = mul(p)
        a = zr / torch.dot(p, q)
        x += a * p
        r -= a * q
        if k % 16 == 15 and float(r.norm()) < stop:
            break
        z = r / d
        zr, old = torch.dot(z, r), zr
        p = z + (zr / old) * p
    return x


def _bicgstab(mul, d, b):
    """BiCGSTAB with Jacobi, restarted on its true residual, to the rounding
    level."""
    x = torch.zeros_like(b)
    for _ in range(4):
        r = b - mul(x)
        r0, rho, stop = r.clone(), torch.dot(r, r), 1e-6 * float(r.norm())
        p = r.clone()
        for k in range(5000):
            ph = p / d
            v = mul(ph)
            a = rho / torch.dot(r0, v)
            s = r - a * v
            sh = s / d
            t = mul(sh)
            w = torch.dot(t, s) / torch.dot(t, t)
            x += a * ph + w * sh
            r = s - w * t
            if k % 16 == 15 and float(r.norm()) < stop:
                break
            rho, old = torch.dot(r0, r), rho
            p = r + (rho / old) * (a / w) * (p - w * v)
        if float((b - mul(x)).norm()) < 1e-13 * float(b.norm()):
            break
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "assemble":
        rows, cols, r, c, v = _triplets(case, seed)
        key = r.astype(np.int64) * cols + c
        order = np.argsort(key, kind="stable")
        key = key[order]
        last = np.append(key[1:] != key[:-1], True)  # of equal ones the last given holds
        key, v = key[last], v[order][last]
        rp = np.zeros(rows + 1, np.int32)
        rp[1:] = np.cumsum(np.bincount(key // cols, minlength=rows))
        return rp, (key % cols).astype(np.int32), v
    g = _gen(seed)
    if kind == "batch":
        sizes, _, rp, col, val = _batch(case, g)
        n = int(sizes.sum())
        b = _uniform(n, g)
        row = torch.repeat_interleave(torch.arange(n, device=_DEV), rp[1:] - rp[:-1])
        d = val[row == col]
        return _cg(_apply(rp, col, val, n), d, b)
    rows, cols, rp, col, val = _matrix(case, g)
    val = val.to(_t_dtype(case)).double()
    row = torch.repeat_interleave(torch.arange(rows, device=_DEV), rp[1:] - rp[:-1])
    nin, nout = (rows, cols) if kind == "matvec_t" else (cols, rows)
    b = _uniform(nin, g).to(_t_dtype(case)).double()
    if kind in ("matvec", "matvec_t", "loop"):
        src, dst = (row, col.long()) if kind == "matvec_t" else (col.long(), row)
        y = torch.zeros(nout, dtype=torch.float64, device=_DEV).index_add_(0, dst, val * b[src])
        if kind != "loop":
            return y
        z = b - 0.125 * y
        return y, z, float(torch.dot(b, y)), float(z.norm())
    d = val[row == col]
    solve = _bicgstab if kind == "bicgstab" else _cg
    return solve(_apply(rp, col, val, rows), d, b)
