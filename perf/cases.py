"""The calls that programs make through ``bml_amd.hip``, as measurable cases.

A case is one step of a client program: a thresholded product, a purification
step written with the separate calls, whole density-matrix solves, the set-up
of a solve, block products.  ``prepare`` builds what the program holds before
the step (seeded matrices resident on the GPU), ``run`` makes the calls, and
``exact`` forms the same products with torch in 64 bits.

Matrices leave ``run`` as views of their device arrays.  Slots past a row's
count are not part of a matrix; where a call may leave old entries there, the
result is copied into a matrix of another width first (a copy moves live
entries only), as programs that keep a result beside a work matrix do.
"""
import math

import numpy as np
import torch

from bml_amd import generators as G
from bml_amd import hip
from bml_amd.ell import Blk

THR = 1e-5
TYPESTR = {np.dtype(np.float32): "<f4", np.dtype(np.float64): "<f8",
           np.dtype(np.complex64): "<c8", np.dtype(np.complex128): "<c16"}


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # a molecule-sized sparse product on the default (bit-exact) engine:
        # latency and launches
        {"name": "x2_small", "op": "x2", "N": 500, "draws": 8, "band": 64, "dtype": "float64"},
        # the random banded product, N = 4096 and ~32 entries a row
        {"name": "x2_banded", "op": "x2", "N": 4096, "draws": 16, "band": 256,
         "dtype": "float64"},
        # C <- alpha A B + beta C with two different matrices, single
        # precision, an odd dimension and width
        {"name": "multiply_f32", "op": "multiply", "N": 10007, "draws": 11, "band": 200,
         "dtype": "float32", "alpha": -2.0, "beta": 1.0},
        # what every solve starts with: drop small entries, spectral bounds,
        # map the spectrum to [0, 1], trace
        {"name": "setup_lattice", "op": "setup", "L": 32, "Lz": 32, "dtype": "float64"},
        # one purification step as a client writes it (bml_multiply_x2 then
        # bml_add_norm), 32^3 lattice iterate
        {"name": "step_lattice32", "op": "step", "L": 32, "Lz": 32, "iters": 8,
         "dtype": "float64"},
        # the complex Hermitian product (Peierls phases), ~280 entries a row
        {"name": "x2_peierls", "op": "x2_peierls", "L": 24, "dtype": "complex128"},
        # a whole density matrix of a small system (molecular dynamics calls
        # this once per time step)
        {"name": "sp2_small", "op": "sp2", "L": 8, "Lz": 9, "M": 256, "maxit": 40,
         "dtype": "float64"},
        # solves of many independent systems of ragged sizes in one call
        {"name": "sp2_batch", "op": "batch", "systems": 16, "lo": 256, "hi": 8192, "maxit": 30,
         "dtype": "float64"},
        # two iterations of a solve whose density matrix is wide (thousands
        # of entries a row), on the unordered setting, single precision, the
        # result handed on as full rows
        {"name": "sp2_wide_f32", "op": "wide", "L": 24, "iters": 2, "dtype": "float32"},
        # the block product on 32 x 32 blocks (matrix cores), double
        {"name": "eb_x2_f64", "op": "eb_x2", "L": 16, "Lz": 8, "b": 32, "dtype": "float64"},
        # a whole block density matrix
        {"name": "eb_sp2_f64", "op": "eb_sp2", "L": 8, "Lz": 6, "b": 32, "maxit": 30,
         "dtype": "float64"},
        # block product with alpha and beta on ragged small blocks
        {"name": "eb_multiply_f32", "op": "eb_multiply", "NB": 3001, "bmin": 2, "bmax": 7,
         "fill": 9, "dtype": "float32", "alpha": 1.0, "beta": -0.5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["x2", "x2", "multiply", "setup", "step", "step", "x2_peierls", "sp2",
                     "batch", "wide", "eb_x2", "eb_sp2", "eb_multiply"])
    real = rng.choice(["float32", "float64"])
    if op in ("x2", "multiply"):
        c = {"op": op, "N": _log(rng, 200, 20000), "draws": rng.randint(3, 24),
             "band": rng.randint(48, 400), "dtype": real}
        if op == "multiply":
            c["alpha"] = rng.choice([1.0, -2.0, 0.75])
            c["beta"] = rng.choice([0.0, 1.0, -0.5])
        return c
    if op == "setup":
        return {"op": op, "L": rng.randint(6, 36), "Lz": rng.randint(5, 36), "dtype": real}
    if op == "step":
        return {"op": op, "L": rng.randint(9, 30), "Lz": rng.randint(9, 30),
                "iters": rng.randint(3, 9), "dtype": real}
    if op == "x2_peierls":
        return {"op": op, "L": rng.randint(8, 24), "dtype": rng.choice(["complex64", "complex128"])}
    if op == "sp2":
        return {"op": op, "L": rng.randint(6, 14), "Lz": rng.randint(5, 15), "M": 256,
                "maxit": 40, "dtype": real}
    if op == "batch":
        lo = _log(rng, 200, 600)
        return {"op": op, "systems": rng.randint(5, 16), "lo": lo, "hi": _log(rng, 1000, 8000),
                "maxit": rng.randint(12, 30), "dtype": real}
    if op == "wide":
        return {"op": op, "L": rng.randint(17, 24), "iters": rng.randint(1, 2), "dtype": real}
    if op in ("eb_x2", "eb_sp2"):
        c = {"op": op, "L": rng.randint(5, 12), "Lz": rng.randint(4, 8),
             "b": rng.choice([20, 27, 32, 32, 32]), "dtype": real if op == "eb_x2" else "float64"}
        if op == "eb_sp2":
            c["L"], c["Lz"] = min(c["L"], 8), min(c["Lz"], 6)
            c["maxit"] = 30
        return c
    return {"op": op, "NB": _log(rng, 60, 4000), "bmin": rng.randint(1, 4),
            "bmax": rng.randint(5, 16), "fill": rng.randint(3, 12),
            "dtype": rng.choice(["float32", "float64", "complex128"]),
            "alpha": rng.choice([1.0, 2.0]), "beta": rng.choice([0.0, -0.5])}


# ---- views of device arrays ----------------------------------------------------

class _Device:
    """A device array for torch; holds the matrix it belongs to."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2}


def _ell(A):
    """(value, index, nnz) of an ellpack_hip matrix, as the device holds them."""
    s = A._s
    return {"value": torch.as_tensor(_Device(A, s.value, (s.N, s.M), TYPESTR[A.dtype]),
                                     device="cuda"),
            "index": torch.as_tensor(_Device(A, s.index, (s.N, s.M), "<i4"), device="cuda"),
            "nnz": torch.as_tensor(_Device(A, s.nnz, (s.N,), "<i4"), device="cuda")}


def _blk(A):
    s = A._s
    return {"value": torch.as_tensor(_Device(A, s.value, (s.NB, s.MB, s.bt, s.bt),
                                             TYPESTR[A.dtype]), device="cuda"),
            "indexb": torch.as_tensor(_Device(A, s.indexb, (s.NB, s.MB), "<i4"), device="cuda"),
            "nnzb": torch.as_tensor(_Device(A, s.nnzb, (s.NB,), "<i4"), device="cuda")}


# ---- inputs ---------------------------------------------------------------------

def _banded(c, seed):
    f = 2 * c["draws"] + 1
    return G.random_banded(N=c["N"], M=4 * f + 8, draws=c["draws"],
                           band=min(c["band"], c["N"] - 1), seed=seed,
                           dtype=np.dtype(c["dtype"]))


def _product_width(c):
    """Holds every distinct column of a product of two banded matrices."""
    return min(c["N"], 4 * min(c["band"], c["N"] - 1) + 1)


def _lattice(c, seed, hopping=-0.1, disorder=0.01):
    return G.lattice_hamiltonian(c["L"], c["L"], c.get("Lz", c["L"]), M=16, hopping=hopping,
                                 disorder=disorder, seed=seed, dtype=np.dtype(c["dtype"]))


def _iterate(H, M, iters, thr):
    """The iterate of a solve after `iters` steps, alone in a matrix."""
    X = hip.zero_matrix(H.precision, H.N, M)
    dH = hip.from_ell(H)
    hip.sp2(dH, X, float(H.N // 2), threshold=thr, tol=0.0, maxit=iters)
    Y = hip.zero_matrix(H.precision, H.N, M + 8)
    hip.copy(X, Y)
    X.free()
    dH.free()
    return Y


def _block_lattice(c, seed, MB=8):
    return G.block_lattice_hamiltonian(c["L"], c["L"], c["Lz"], b=c["b"], MB=MB, onsite_shift=6.0,
                                       coupling=0.02, seed=seed, dtype=np.dtype(c["dtype"]))


def _ragged_blocks(c, seed, which):
    """A random block matrix: diagonal block plus `fill` block columns near
    the diagonal in every block row, sizes between bmin and bmax."""
    bs = np.random.default_rng(seed).integers(c["bmin"], c["bmax"] + 1, c["NB"]).astype(np.int32)
    bs[0] = c["bmax"]
    rng = np.random.default_rng([seed, which])
    NB, f, bmax = c["NB"], min(c["fill"], c["NB"] - 1), c["bmax"]
    reach = max(3 * f, 1)
    off = np.argsort(rng.random((NB, 2 * reach)), axis=1)[:, :f] - reach
    off = np.where(off >= 0, off + 1, off)
    cols = np.concatenate([np.arange(NB)[:, None], (np.arange(NB)[:, None] + off) % NB], axis=1)
    # columns that meet after the wrap (few block rows): the first one stays
    dt = np.dtype(c["dtype"])
    out = Blk.zeros(bs, f + 1, dt, bmax)
    vals = rng.uniform(-1.0, 1.0, size=(NB, f + 1, bmax, bmax))
    if dt.kind == "c":
        vals = vals + 1j * rng.uniform(-1.0, 1.0, size=vals.shape)
    r = np.arange(bmax)
    vals *= (r[None, None, :, None] < bs[:, None, None, None])
    for ib in range(NB):
        _, first = np.unique(cols[ib], return_index=True)
        keep = np.sort(first)
        n = len(keep)
        out.indexb[ib, :n] = cols[ib][keep]
        out.nnzb[ib] = n
        out.value[ib, :n] = vals[ib, :n] * (r[None, None, :] < bs[out.indexb[ib, :n]][:, None, None])
    return out


# ---- prepare / run ---------------------------------------------------------------

def prepare(case, seed):
    c, op = case, case["op"]
    # the default engine everywhere but for wide density matrices
    hip.set_row_engine(hip.ROW_ENGINE_UNORDERED if op == "wide" else hip.ROW_ENGINE_EXACT)
    dt = np.dtype(c["dtype"])
    prec = hip.precision_of(dt)
    s = {"case": c}
    if op == "x2":
        s["X"] = hip.from_ell(_banded(c, seed))
        s["X2"] = hip.zero_matrix(prec, c["N"], _product_width(c))
        s["out"] = _ell(s["X2"])
    elif op == "multiply":
        s["A"] = hip.from_ell(_banded(c, 2 * seed))
        s["B"] = hip.from_ell(_banded(c, 2 * seed + 1))
        s["C0"] = hip.from_ell(_banded(c, 2 * seed + 2), _product_width(c))
        s["C"] = hip.copy_new(s["C0"])
        s["out"] = _ell(s["C"])
    elif op == "setup":
        H = _lattice(c, seed, hopping=-0.1, disorder=0.1)
        s["H"] = hip.from_ell(H)
        s["A"] = hip.copy_new(s["H"])
        s["out"] = _ell(s["A"])
    elif op == "step":
        s["X"] = _iterate(_lattice(c, seed), 256, c["iters"], THR)
        N = s["X"].N
        s["X2"] = hip.zero_matrix(prec, N, 512)
        s["Y"] = hip.zero_matrix(prec, N, s["X"].M)
        s["out"] = {"x2": _ell(s["X2"]), "next": _ell(s["Y"])}
    elif op == "x2_peierls":
        H = G.peierls_hamiltonian(c["L"], M=16, seed=seed, dtype=dt)
        s["X"] = _iterate(H, 512, 3, 1e-6)
        s["X2"] = hip.zero_matrix(prec, H.N, min(H.N, 640))
        s["out"] = _ell(s["X2"])
    elif op == "sp2":
        H = _lattice(c, seed)
        s["H"] = hip.from_ell(H)
        s["X"] = hip.zero_matrix(prec, H.N, c["M"])
        s["Y"] = hip.zero_matrix(prec, H.N, c["M"] + 8)
        s["out"] = _ell(s["Y"])
    elif op == "batch":
        # sizes spread evenly over the range (of their logarithm), so the work
        # does not depend on the seed
        sizes = np.exp(np.linspace(math.log(c["lo"]), math.log(c["hi"]), c["systems"]))
        s["H"], s["X"], s["Y"] = [], [], []
        for k, n in enumerate(sizes):
            Lx, Ly, Lz = G.near_cubic(int(n))
            H = G.lattice_hamiltonian(Lx, Ly, Lz, M=16, hopping=-0.1, disorder=0.01,
                                      seed=seed + 1000 * k, dtype=dt)
            s["H"].append(hip.from_ell(H))
            s["X"].append(hip.zero_matrix(prec, H.N, 256))
            s["Y"].append(hip.zero_matrix(prec, H.N, 264))
        s["nocc"] = [float(h.N // 2) for h in s["H"]]
        s["out"] = [_ell(y) for y in s["Y"]]
    elif op == "wide":
        H = _lattice(c, seed, hopping=-0.5, disorder=0.05)
        M = min(H.N, 3072)
        s["H"] = hip.from_ell(H)
        s["X"] = hip.zero_matrix(prec, H.N, M)
        # the window engine's sums do not depend on the order of the adds, so
        # the iterate is the same whenever it is made
        hip.set_row_engine(hip.ROW_ENGINE_WINDOW)
        hip.sp2(s["H"], s["X"], H.N / 2, threshold=THR, tol=1e-8, maxit=16)
        hip.set_row_engine(hip.ROW_ENGINE_UNORDERED)
        s["X0"] = hip.copy_new(s["X"])
        s["out"] = _ell(s["X"])
        s["slot"] = torch.arange(M, device="cuda", dtype=torch.int32)[None, :]
        s["D"] = torch.zeros((H.N, H.N + 1), dtype=getattr(torch, c["dtype"]), device="cuda")
    elif op == "eb_x2":
        H = _block_lattice(c, seed)
        dH = hip.from_blk(H)
        X = hip.block_matrix(H.precision, H.bsize, min(H.NB, 160))
        hip.eb_sp2(dH, X, H.N / 2, threshold=THR, tol=0.0, maxit=10)
        s["X"] = hip.block_matrix(H.precision, H.bsize, min(H.NB, 64))
        hip.eb_copy(X, s["X"])
        X.free()
        dH.free()
        s["X2"] = hip.block_matrix(H.precision, H.bsize, min(H.NB, 160))
        s["Y"] = hip.block_matrix(H.precision, H.bsize, min(H.NB, 64) + 1)
        s["out"] = _blk(s["Y"])
    elif op == "eb_sp2":
        H = _block_lattice(c, seed)
        s["H"] = hip.from_blk(H)
        s["X"] = hip.block_matrix(H.precision, H.bsize, min(H.NB, 160))
        s["Y"] = hip.block_matrix(H.precision, H.bsize, min(H.NB, 64) + 1)
        s["nocc"] = H.N / 2
        s["out"] = _blk(s["Y"])
    elif op == "eb_multiply":
        A, B, C0 = (_ragged_blocks(c, seed, k) for k in range(3))
        MC = min(c["NB"], (c["fill"] + 1) ** 2)
        s["A"], s["B"] = hip.from_blk(A), hip.from_blk(B)
        s["C0"] = hip.from_blk(C0, MC)
        s["C"] = hip.eb_copy_new(s["C0"])
        s["Y"] = hip.block_matrix(prec, A.bsize, MC + 1)
        s["out"] = _blk(s["Y"])
    else:
        raise ValueError(op)
    hip.synchronize()
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "x2":
        tr = hip.multiply_x2(s["X"], s["X2"], THR)
        return {"X2": s["out"], "traces": list(tr)}
    if op == "multiply":
        if c["beta"] != 0.0:
            hip.copy(s["C0"], s["C"])
        hip.multiply(s["A"], s["B"], s["C"], c["alpha"], c["beta"], THR)
        return s["out"]
    if op == "setup":
        hip.copy(s["H"], s["A"])
        hip.threshold(s["A"], 0.02)
        lo, hi = hip.gershgorin(s["A"])
        hip.normalize(s["A"], lo, hi)
        return {"A": s["out"], "bounds": [lo, hi], "trace": hip.trace(s["A"])}
    if op == "step":
        tr = hip.multiply_x2(s["X"], s["X2"], THR)
        hip.copy(s["X"], s["Y"])
        norm = hip.add_norm(s["Y"], s["X2"], 2.0, -1.0, THR)
        return {**s["out"], "traces": list(tr), "norm": norm}
    if op == "x2_peierls":
        tr = hip.multiply_x2(s["X"], s["X2"], 1e-6)
        return {"X2": s["out"], "traces": list(tr)}
    if op == "sp2":
        r, hist = hip.sp2(s["H"], s["X"], float(s["H"].N // 2), threshold=THR, tol=1e-3,
                          maxit=c["maxit"])
        hip.copy(s["X"], s["Y"])
        return {"X": s["out"], "iterations": r.iterations, "trace": r.trace_x}
    if op == "batch":
        res = hip.sp2_batch(s["H"], s["X"], s["nocc"], threshold=THR, tol=1e-3,
                            maxit=c["maxit"])
        for x, y in zip(s["X"], s["Y"]):
            hip.copy(x, y)
        return {"X": s["out"], "iterations": np.array([r.iterations for r in res])}
    if op == "wide":
        hip.copy(s["X0"], s["X"])
        r, hist = hip.sp2(s["H"], s["X"], s["X"].N / 2, threshold=THR, tol=1e-8,
                          maxit=c["iters"], resume=True)
        # the consumer takes full rows (a row's entries come in no fixed
        # order); the last column collects the dead slots
        x, D = s["out"], s["D"]
        at = torch.where(s["slot"] < x["nnz"][:, None], x["index"], s["X"].N).long()
        D.zero_().scatter_(1, at, x["value"])
        return {"X": D[:, :-1], "trace": r.trace_x, "trace2": r.trace_x2}
    if op == "eb_x2":
        tr = hip.eb_multiply_x2(s["X"], s["X2"], THR)
        hip.eb_copy(s["X2"], s["Y"])
        return {"X2": s["out"], "traces": list(tr)}
    if op == "eb_sp2":
        r, hist = hip.eb_sp2(s["H"], s["X"], s["nocc"], threshold=THR, tol=1e-8,
                             maxit=c["maxit"])
        hip.eb_copy(s["X"], s["Y"])
        return {"X": s["out"], "iterations": r.iterations, "trace": r.trace_x}
    hip.eb_copy(s["C0"], s["C"])
    hip.eb_multiply(s["A"], s["B"], s["C"], c["alpha"], c["beta"], THR)
    hip.eb_copy(s["C"], s["Y"])
    return s["out"]


# ---- what a pass cannot do without ---------------------------------------------

def _distinct(products, span):
    """Expected distinct columns of `products` draws over `span` columns."""
    return span * (1.0 - math.exp(-products / span))


def work(case):
    """Every input entry read once, every output entry written once (value and
    column), two flops per partial product (eight for complex).  The fills of
    the lattice iterates (entries a row) are rounded measured figures."""
    c, op = case, case["op"]
    dt = np.dtype(c["dtype"])
    e = dt.itemsize + 4
    f2 = 8 if dt.kind == "c" else 2
    if op in ("x2", "multiply"):
        N, f = c["N"], 2 * c["draws"] + 1
        out = _distinct(f * f, min(N, 2.5 * c["band"]))
        ins = f * (1 if op == "x2" else 3)
        return {"bytes": N * (e * (ins + out) + 12), "flops": f2 * N * f * f}
    if op == "setup":
        N = c["L"] ** 2 * c["Lz"]
        return {"bytes": 2 * 7 * N * e, "flops": 40 * N}
    if op == "step":
        N = c["L"] ** 2 * c["Lz"]
        f = min(N, 177.0)
        return {"bytes": N * e * 3 * f, "flops": f2 * N * f * f}
    if op == "x2_peierls":
        N = c["L"] ** 3
        f = min(N, 279.0)
        return {"bytes": N * e * (f + min(N, 434)), "flops": f2 * N * f * f}
    if op in ("sp2", "batch"):
        sizes = [c["L"] ** 2 * c["Lz"]] if op == "sp2" else np.exp(
            np.linspace(math.log(c["lo"]), math.log(c["hi"]), c["systems"]))
        n, it = float(np.sum(sizes)), 10
        return {"bytes": n * e * (7 + 170), "flops": it * f2 * n * 150 * 150}
    if op == "wide":
        N = c["L"] ** 3
        f = min(0.5 * N, 2510.0)
        # X is symmetric: the upper triangle of its square is enough
        return {"bytes": N * e * f + dt.itemsize * float(N) * N, "flops": c["iters"] * N * f * f}
    if op in ("eb_x2", "eb_sp2"):
        NB, t = c["L"] ** 2 * c["Lz"], c["b"] ** 2
        if op == "eb_x2":
            return {"bytes": NB * t * dt.itemsize * (25 + 25), "flops": 2.0 * NB * 25 * 25 * t * c["b"]}
        return {"bytes": NB * t * dt.itemsize * (7 + 25),
                "flops": 20 * 2.0 * NB * 20 * 20 * t * c["b"]}
    NB, b, f = c["NB"], 0.5 * (c["bmin"] + c["bmax"]), c["fill"] + 1
    out = _distinct(f * f, 9 * f)
    return {"bytes": NB * b * b * dt.itemsize * (3 * f + out), "flops": f2 * NB * f * f * b ** 3}


# ---- 64-bit results ---------------------------------------------------------------

def _pairs(ia, na, ib, nb, r0, r1, N):
    """Partial products of rows r0..r1 of A*B in (jp, kp) order: positions in
    A's and B's entry arrays, the group (distinct column of its row) each one
    adds into, and of every group its row, column and rank in the order in
    which the row first meets its columns."""
    dev = ia.device
    MA, MB = ia.shape[1], ib.shape[1]
    rows = torch.arange(r0, r1, device=dev)
    live = torch.arange(MA, device=dev)[None, :] < na[r0:r1, None]
    pa = (rows[:, None] * MA + torch.arange(MA, device=dev))[live]
    row = rows[:, None].expand(-1, MA)[live]
    j = ia[r0:r1][live].long()
    cnt = nb[j].long()
    start = torch.cumsum(cnt, 0) - cnt
    total = int(cnt.sum())
    which = torch.repeat_interleave(torch.arange(len(j), device=dev), cnt)
    kp = torch.arange(total, device=dev) - start[which]
    pb = j[which] * MB + kp
    key = row[which] * N + ib.reshape(-1)[pb].long()
    skey, order = torch.sort(key, stable=True)
    new = torch.ones(total, dtype=torch.bool, device=dev)
    new[1:] = skey[1:] != skey[:-1]
    gid = torch.cumsum(new, 0) - 1
    group = torch.empty_like(gid)
    group[order] = gid
    first = order[new]
    gkey = skey[new]
    by = torch.argsort(first)
    rank = torch.empty_like(by)
    rank[by] = torch.arange(len(by), device=dev)
    return pa[which], pb, group, gkey // N, gkey % N, rank


def _place(row, rank, keep, r0, r1):
    """Slots of the kept groups in their rows (first-met order)."""
    row, rank = row[keep] - r0, rank[keep]
    by = torch.argsort(rank)
    r = row[by]
    o = torch.argsort(r, stable=True)
    rs = r[o]
    n = torch.bincount(rs, minlength=r1 - r0)
    slot = torch.empty_like(rs)
    slot[o] = torch.arange(len(rs), device=rs.device) - (torch.cumsum(n, 0) - n)[rs]
    out = torch.empty_like(slot)
    out[by] = slot
    return row, out


def _wide(v):
    return v.to(torch.complex128 if v.is_complex() else torch.float64)


def _x2_exact(A, MC, thr):
    """X^2 above thr (and the diagonal) in the layout of the exact engine.
    In single precision only the traces: what rounding leaves on the other
    side of thr would shift the rest of its row."""
    N = A["value"].shape[0]
    ia, na = A["index"], A["nnz"]
    v = _wide(A["value"]).reshape(-1)
    out = torch.zeros((N, MC), dtype=v.dtype, device=v.device)
    f = max(1, int(na.max()))
    chunk = max(1, 30_000_000 // (f * f))
    live = torch.arange(ia.shape[1], device=ia.device)[None, :] < na[:, None]
    diag = live & (ia == torch.arange(N, device=ia.device)[:, None])
    tr = [float(_wide(A["value"])[diag].real.sum()), 0.0]
    for r0 in range(0, N, chunk):
        r1 = min(N, r0 + chunk)
        pa, pb, g, row, col, rank = _pairs(ia, na, ia, na, r0, r1, N)
        acc = torch.zeros(len(row), dtype=v.dtype, device=v.device)
        p = v[pa] * v[pb]
        if acc.is_complex():
            torch.view_as_real(acc).index_add_(0, g, torch.view_as_real(p))
        else:
            acc.index_add_(0, g, p)
        keep = (acc.abs() > thr) | (row == col)
        tr[1] += float(acc[row == col].real.sum())
        r, slot = _place(row, rank, keep, r0, r1)
        out[r + r0, slot] = acc[keep]
    single = A["value"].dtype in (torch.float32, torch.complex64)
    return (None if single else out), tr


def exact(case, seed):
    c, op = case, case["op"]
    if op in ("x2", "x2_peierls"):
        s = prepare(case, seed)
        out, tr = _x2_exact(_ell(s["X"]), s["X2"].M, THR if op == "x2" else 1e-6)
        return {"X2": {"value": out, "index": None, "nnz": None}, "traces": tr}
    if op == "step":
        s = prepare(case, seed)
        out, tr = _x2_exact(_ell(s["X"]), s["X2"].M, THR)
        return {"x2": {"value": out, "index": None, "nnz": None}, "next": None, "traces": tr,
                "norm": None}
    if op == "setup":
        H = _lattice(c, seed, hopping=-0.1, disorder=0.1).astype(np.float64)
        H.value[np.abs(H.value) <= np.dtype(c["dtype"]).type(0.02)] = 0.0
        n = (H.value != 0).sum(1)
        by = np.argsort(H.value == 0, axis=1, kind="stable")
        v, ix = np.take_along_axis(H.value, by, 1), np.take_along_axis(H.index, by, 1)
        at = (np.arange(H.M)[None, :] < n[:, None]) & (ix == np.arange(H.N)[:, None])
        d = v[at]
        rad = np.abs(v).sum(1) - np.abs(d)
        lo, hi = float((d - rad).min()), float((d + rad).max())
        out = np.where(at, (hi - v) / (hi - lo), -v / (hi - lo))
        tr = float(out[at].sum())
        return {"A": None, "bounds": [lo, hi], "trace": tr}
    if op == "wide":
        if c["iters"] != 1 or c["dtype"] != "float64" or c["L"] > 20:
            return None
        s = prepare(case, seed)
        N = s["X"].N
        x = _ell(s["X0"])
        at = torch.arange(s["X0"].M, device="cuda")[None, :] < x["nnz"][:, None]
        D = torch.zeros((N, N), dtype=torch.float64, device="cuda")
        D[torch.arange(N, device="cuda")[:, None].expand_as(at)[at], x["index"][at].long()] = \
            x["value"][at]
        t = float(D.diagonal().sum())
        Y = D @ D
        t2 = float((D * D).sum())
        eye = torch.eye(N, dtype=torch.bool, device=D.device)
        Y = torch.where((Y.abs() > THR) | eye, Y, torch.zeros_like(Y))
        nocc = N / 2
        Z = Y if abs(t2 - nocc) < abs(2 * t - t2 - nocc) else 2 * D - Y
        return {"X": torch.where(Z.abs() > THR, Z, torch.zeros_like(Z)), "trace": t, "trace2": t2}
    if op == "eb_x2":
        s = prepare(case, seed)
        A = _blk(s["X"])
        NB, MB, b = A["indexb"].shape[0], A["indexb"].shape[1], s["X"].bt
        v = _wide(A["value"]).reshape(NB * MB, b, b)
        Y = torch.zeros((NB, s["Y"].MB, b, b), dtype=v.dtype, device=v.device)
        tr = [0.0, 0.0]
        at = (torch.arange(MB, device=v.device)[None, :] < A["nnzb"][:, None]) & (
            A["indexb"] == torch.arange(NB, device=v.device)[:, None])
        tr[0] = float(v.reshape(NB, MB, b, b)[at].diagonal(dim1=1, dim2=2).sum())
        for r0 in range(0, NB, 64):
            r1 = min(NB, r0 + 64)
            pa, pb, g, row, col, rank = _pairs(A["indexb"], A["nnzb"], A["indexb"], A["nnzb"],
                                               r0, r1, NB)
            acc = torch.zeros((len(row), b, b), dtype=v.dtype, device=v.device)
            for k in range(0, len(pa), 20000):
                acc.index_add_(0, g[k:k + 20000], torch.bmm(v[pa[k:k + 20000]].contiguous(),
                                                            v[pb[k:k + 20000]].contiguous()))
            keep = (acc.abs().amax(dim=(1, 2)) > THR) | (row == col)
            tr[1] += float(acc[row == col].diagonal(dim1=1, dim2=2).sum())
            r, slot = _place(row, rank, keep, r0, r1)
            Y[r + r0, slot] = acc[keep]
        return {"X2": {"value": Y, "indexb": None, "nnzb": None}, "traces": tr}
    return None
