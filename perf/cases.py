"""The work that a user of this library has it do, as cases that can be timed
and compared: H*X with a compressed inverse, H*H products, inversions, and a
batch of independent operators, from the smallest calls to the largest.

Operators are -div(a grad u) + u on a grid, log a a Gaussian random field
(sigma 1, correlation length 0.1); the compressed operands are their inverses
(Green's operators), computed once by DirectInvert as a program does before it
applies or multiplies them. One case is too large for that here and takes
random factors at full rank instead.
"""
import math

import numpy as np
import torch

import dmhm_amd
from dmhm_amd import workloads as W

OVERSAMPLE = 4


def _case(name, op, sizes, levels, rank, precision, **more):
    c = {"name": name, "op": op, "nx": sizes[0], "ny": sizes[1], "nz": sizes[2] if len(sizes) == 3 else 0,
         "levels": levels, "rank": rank, "precision": precision}
    c.update(more)
    return c


def listed():
    return [
        # One application of a small inverse inside an iterative solver: all latency.
        _case("apply_64_f64", "apply", (64, 64), 4, 8, "f64", k=1, transposed=False, operand="inverse"),
        # A single-precision preconditioner applied once per Krylov step.
        _case("apply_256_f32", "apply", (256, 256), 6, 16, "f32", k=1, transposed=False, operand="inverse"),
        # The adjoint application of two-sided methods (BiCG, LSQR, adjoint solves).
        _case("apply_256_f64_trans", "apply", (256, 256), 6, 16, "f64", k=1, transposed=True, operand="inverse"),
        # Many right-hand sides at once: block solvers, sampling a Gaussian field.
        _case("apply_256_f64_k64", "apply", (256, 256), 6, 16, "f64", k=64, transposed=False, operand="inverse"),
        # The largest matrix a user applies to one vector (7 GB of factors).
        _case("apply_512_f32", "apply", (512, 512), 7, 32, "f32", k=1, transposed=False, operand="random"),
        # A 3D inverse on a ragged grid applied to a few vectors.
        _case("apply_3d_f32_k6", "apply", (27, 33, 30), 3, 16, "f32", k=6, transposed=False, operand="inverse"),
        # A small product at a relative tolerance, on a ragged grid.
        _case("product_97x83_f64_tol", "product", (97, 83), 4, 12, "f64", tol=1e-10, update=False),
        # The product of two full inverses: the step that every Schulz iteration is made of.
        _case("product_256_f64", "product", (256, 256), 6, 16, "f64", tol=0.0, update=False),
        # The update form C := alpha A B + beta C in 3D, single precision.
        _case("product_3d_f32_update", "product", (20, 22, 24), 3, 16, "f32", tol=0.0, update=True),
        # A small operator inverted and used to solve for a few right-hand sides.
        _case("invert_64_f64", "invert", (64, 64), 4, 8, "f64", method="direct", k=4),
        # The inversion of the 256^2 operator to 1e-8: direct start, Schulz refinement.
        _case("invert_256_f64", "invert", (256, 256), 6, 16, "f64", method="schulz", k=4),
        # Products of a set of independent small operators (parameter studies).
        _case("batch_24_f32", "batch", (48, 64), 4, 8, "f32", count=24),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["apply", "apply", "apply", "product", "product", "invert", "batch"])
    precision = rng.choice(["f64", "f32"])
    if op == "batch":
        lo, hi = sorted(_log_uniform(rng, 24, 64) for _ in range(2))
        c = _case("", op, (lo, hi), 4, rng.randint(4, 8), precision, count=_log_uniform(rng, 2, 24))
    else:
        if rng.random() < 0.3:
            top = 30 if op == "apply" else 22
            sizes, levels = tuple(rng.randint(12, top) for _ in range(3)), 3
            rank = rng.randint(6, 16)
        else:
            side = _log_uniform(rng, 32, {"apply": 250, "product": 220, "invert": 160}[op])
            sizes = (side, max(24, int(side * rng.uniform(0.75, 1.0))))
            # Leaves of 8 to 16 points a side.
            levels = 1 + max(2, int(math.floor(math.log2(side / 8.0))))
            rank = rng.randint(4, 16)
        if op == "apply":
            c = _case("", op, sizes, levels, rank, precision, k=_log_uniform(rng, 1, 64),
                      transposed=rng.random() < 0.3, operand="inverse")
        elif op == "product":
            c = _case("", op, sizes, levels, rank, precision, tol=1e-10 if precision == "f64" and rng.random() < 0.4 else 0.0,
                      update=rng.random() < 0.3)
        else:
            c = _case("", op, sizes, levels, rank, "f64", method=rng.choice(["direct", "schulz"]),
                      k=_log_uniform(rng, 1, 16))
    del c["name"]
    return c


def _sizes(case):
    return [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] else [])


def _operator(sizes, levels, seed):
    """CSR of the operator in hierarchical ordering, and the natural -> hierarchical map."""
    a = W.coefficient_lognormal(tuple(s + 2 for s in sizes), 1.0, 0.1, seed, features=256)
    rowptr, colind, vals, sz, hmap = W.flux_operator(a, levels)
    return {"rowptr": rowptr, "colind": colind, "vals": vals, "sizes": sz, "map": hmap}


def _matrix(op, levels, rank):
    cls = dmhm_amd.HMat2d if len(op["sizes"]) == 2 else dmhm_amd.HMat3d
    return cls.from_csr(op["sizes"], levels, rank, True, op["rowptr"], op["colind"], op["vals"])


def _inverse(op, levels, rank, precision):
    X = _matrix(op, levels, rank)
    X.DirectInvert()
    return X if precision == "f64" else X.Convert(dmhm_amd.DMHM_F32)


def _columns(n, k, precision, seed, to="cuda"):
    """n x k right-hand sides, column-major."""
    g = torch.Generator().manual_seed(seed)
    b = torch.randn((k, n), generator=g, dtype=torch.float64)
    if precision == "f32":
        b = b.float()
    return b.to(to).t()


def _batch_sides(case):
    return [case["nx"] if i % 2 == 0 else case["ny"] for i in range(case["count"])]


def prepare(case, seed):
    dmhm_amd.init(0)
    s = {"case": case}
    levels, rank, prec = case["levels"], case["rank"], case["precision"]
    if case["op"] == "batch":
        sides = _batch_sides(case)
        ops = [_operator([m, m], levels, 1000 * seed + i) for i, m in enumerate(sides)]
        s["B"] = dmhm_amd.HBatch.create([_inverse(o, levels, rank, prec) for o in ops])
        s["w"] = [_columns(m * m, 4, prec, 1000 * seed + i) for i, m in enumerate(sides)]
        return s
    sizes = _sizes(case)
    n = int(np.prod(sizes))
    if case["op"] == "apply" and case["operand"] == "random":
        H = dmhm_amd.HMat2d.zeros(sizes, levels, rank, True, dmhm_amd.DMHM_F32 if prec == "f32" else dmhm_amd.DMHM_F64)
        H.SetToRandom(seed + 1)
        s["H"], s["x"] = H, _columns(n, case["k"], prec, seed)
        return s
    op = _operator(sizes, levels, seed)
    if case["op"] == "apply":
        s["H"], s["x"] = _inverse(op, levels, rank, prec), _columns(n, case["k"], prec, seed)
    elif case["op"] == "product":
        s["H"], s["x"] = _inverse(op, levels, rank, prec), _columns(n, 8, prec, seed)
    else:
        s["H"], s["x"] = _matrix(op, levels, rank), _columns(n, case["k"], prec, seed)
    return s


def run(s):
    case = s["case"]
    if case["op"] == "apply":
        H = s["H"]
        return H.TransposeMultiply(1.0, s["x"]) if case["transposed"] else H.Multiply(1.0, s["x"])
    if case["op"] == "product":
        H = s["H"]
        opts = {"tol_mode": 1, "rel_tol": case["tol"]} if case["tol"] > 0 else {}
        if case["update"]:
            C = H.Copy()
            H.Multiply(0.5, H, 1.0, C, **opts)
        else:
            C = H.Multiply(1.0, H, **opts)
        return C.Multiply(1.0, s["x"])
    if case["op"] == "invert":
        X = s["H"].Copy()
        if case["method"] == "direct":
            X.DirectInvert()
        else:
            X.SchulzInvert(start="direct", stopTol=1e-8, maxIterations=80, stall_stop=True)
        return X.Multiply(1.0, s["x"])
    C = s["B"].Multiply(1.0, s["B"])
    return [C.member(i).Multiply(1.0, w) for i, w in enumerate(s["w"])]


def _entries(sizes, levels, rank):
    """Stored entries of the dense leaves and of the rank-`rank` factors, and the mean leaf's size."""
    lv = dmhm_amd.geometry_leaves(sizes, levels, True).astype(np.int64)
    rows, cols = lv[:, 3], lv[:, 5]
    dense = lv[:, 0] == 1
    r = np.minimum(rank, np.minimum(rows, cols))
    return (int((rows * cols)[dense].sum()), int(((rows + cols) * r)[~dense].sum()),
            float(rows[dense].mean()) if dense.any() else 0.0)


def _product_flops(sizes, levels, rank):
    """The dense leaf products, and A and B each applied to rank + oversample
    columns from both sides (the sketch and its projection)."""
    dense, low, leaf = _entries(sizes, levels, rank)
    t = dmhm_amd.hmat.geometry_product_terms(sizes, levels, True)
    return 2.0 * leaf ** 3 * t["dd_to_dense"] + 8.0 * (rank + OVERSAMPLE) * (dense + low)


def work(case):
    e = 8 if case["precision"] == "f64" else 4
    levels, rank = case["levels"], case["rank"]
    if case["op"] == "batch":
        b = f = 0.0
        for m in _batch_sides(case):
            dense, low, _ = _entries([m, m], levels, rank)
            b += e * (3.0 * (dense + low) + 8.0 * m * m)
            f += _product_flops([m, m], levels, rank) + 8.0 * (dense + low)
        return {"bytes": b, "flops": f}
    sizes = _sizes(case)
    n = int(np.prod(sizes))
    dense, low, _ = _entries(sizes, levels, rank)
    stored = dense + low
    if case["op"] == "apply":
        return {"bytes": e * (stored + 2.0 * n * case["k"]), "flops": 2.0 * case["k"] * stored}
    flops = _product_flops(sizes, levels, rank)
    if case["op"] == "product":
        # Read A (= B) once, write C, read C again for its application.
        return {"bytes": e * (3.0 * stored + 16.0 * n), "flops": flops + 16.0 * stored}
    # Elimination costs about what one product does; the refinement is two
    # products more. The operator's leaves are read, the inverse is written
    # and read again for the solves.
    return {"bytes": e * (dense + 2.0 * stored + 2.0 * n * case["k"]),
            "flops": flops * (1.0 if case["method"] == "direct" else 3.0) + 2.0 * case["k"] * stored}


def _solver(op):
    """x -> A^-1 x in 64 bits, rows in hierarchical ordering: block elimination over the last axis of the grid."""
    sizes, hmap = op["sizes"], op["map"].astype(np.int64)
    n, m = int(np.prod(sizes)), int(sizes[-1])
    p = n // m
    nat = np.empty(n, dtype=np.int64)
    nat[hmap] = np.arange(n)
    rows = nat[np.repeat(np.arange(n), np.diff(op["rowptr"]))]
    cols, vals = nat[op["colind"]], op["vals"]
    D = np.zeros((m, p, p))
    E = np.zeros((m, p))                      # E[j]: coupling of slab j to slab j - 1 (diagonal)
    same = rows // p == cols // p
    np.add.at(D, (rows[same] // p, rows[same] % p, cols[same] % p), vals[same])
    low = rows // p == cols // p + 1
    E[rows[low] // p, rows[low] % p] = vals[low]
    inv = np.empty_like(D)                    # inverses of the Schur complements
    for j in range(m):
        S = D[j] if j == 0 else D[j] - E[j][:, None] * inv[j - 1] * E[j][None, :]
        inv[j] = np.linalg.inv(S)

    def solve(b):
        y = b[hmap].reshape(m, p, -1).copy()
        for j in range(1, m):
            y[j] -= E[j][:, None] * (inv[j - 1] @ y[j - 1])
        for j in range(m - 1, -1, -1):
            r = y[j] if j == m - 1 else y[j] - E[j + 1][:, None] * y[j + 1]
            y[j] = inv[j] @ r
        return y.reshape(n, -1)[nat]

    return solve


def exact(case, seed):
    levels = case["levels"]
    if case["op"] == "batch":
        out = []
        for i, m in enumerate(_batch_sides(case)):
            solve = _solver(_operator([m, m], levels, 1000 * seed + i))
            w = _columns(m * m, 4, case["precision"], 1000 * seed + i, to="cpu").double().numpy()
            out.append(torch.from_numpy(solve(solve(w))))
        return out
    if case["op"] == "apply" and case["operand"] == "random":
        return None                           # factors drawn by the library's own generator
    sizes = _sizes(case)
    n = int(np.prod(sizes))
    solve = _solver(_operator(sizes, levels, seed))
    k = 8 if case["op"] == "product" else case["k"]
    x = _columns(n, k, case["precision"], seed, to="cpu").double().numpy()
    y = solve(x)                              # the operator is symmetric: its transposed inverse is its inverse
    if case["op"] == "product":
        y = 0.5 * solve(y) + y if case["update"] else solve(y)
    return torch.from_numpy(y)
