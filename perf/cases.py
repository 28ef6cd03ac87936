"""The work that a user has this engine do, as cases that can be timed and compared.

Points lie on a cylinder of radius 1 with 12,500 points per unit of height (the
benchmark's density) unless the case says otherwise, the covariance is
exp(-r / 0.5) + 1e-2 I, compression ACA+ at eps 1e-4: the workloads of the
benchmark, the GP likelihood and the tests.  Vectors of the device entry points
are in the cluster tree's numbering, as those entry points take them, and
their calls are queued on a stream of the caller; host entry points take user
numbering.

Kinds of a case:
  gemv       y = A x on device vectors, the assembled matrix in hand
  gemv_host  hmat_interface_t.gemv on host vectors, user numbering
  assemble   a new matrix over a tree in hand, assembled, applied to a block
             of vectors (what the GP gradient does with dK/dl)
  factor     a new matrix over a tree in hand: assembly, factorisation, solve
             (one evaluation of a likelihood, one system of a batch)
  solve      the factor in hand, one block of right-hand sides
  gp         negative log-likelihood of a Gaussian process and its gradient
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hmat-oss_amd"))

import hmat_amd  # noqa: E402
from hmat_amd.gp import gp_nll  # noqa: E402

LENGTH, NUGGET, EPS, ETA, SHIFT = 0.5, 1e-2, 1e-4, 2.0, 0.05
KINDS = {"exponential": hmat_amd.KERNEL_EXPONENTIAL, "gaussian": hmat_amd.KERNEL_GAUSSIAN,
         "dlength": hmat_amd.KERNEL_EXPONENTIAL_DLENGTH,
         "shifted": hmat_amd.KERNEL_SHIFTED_EXPONENTIAL, "helmholtz": hmat_amd.KERNEL_HELMHOLTZ}
# mean rank of the admissible blocks (by their rows + columns), measured on these point sets
MEAN_RANK = {"exponential": 6, "gaussian": 6, "dlength": 6, "shifted": 6, "helmholtz": 23}
GP_PROBES = 64


def _case(name, kind, n, **kw):
    c = {"name": name, "kind": kind, "n": n, "height": n / 12500.0, "leaf": 128, "nrhs": 1,
         "kernel": "exponential", "type": "f64", "symmetric": True, "algo": "none"}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest product: launches and latency (an inner loop on a small system)
        _case("gemv_2k", "gemv", 2000),
        # the C API's own product on host vectors, as a program written for the
        # reference calls it
        _case("gemv_host_10k", "gemv_host", 10007),
        # the headline product: one right-hand side, HBM traffic
        _case("gemv_200k", "gemv", 200000),
        # the residual of a block of right-hand sides (refinement, block Krylov)
        _case("gemv_8rhs_50k", "gemv", 50021, nrhs=8),
        # single precision, non-symmetric storage (the matrices that H-LU takes)
        _case("gemv_f32_nonsym_30k", "gemv", 30011, nrhs=4, leaf=100, kernel="shifted", type="f32",
              symmetric=False),
        # complex product of the Helmholtz workload
        _case("gemv_helmholtz_20k", "gemv", 20000, kernel="helmholtz", type="c128", symmetric=False),
        # assembly of the covariance's derivative and its product with the probes
        _case("assemble_50k", "assemble", 50000, nrhs=8, kernel="dlength"),
        # a small system from points to solution in double precision
        _case("llt_f64_4k", "factor", 4000, type="f64", algo="llt"),
        # the precision workload: single-precision factor, refinement to 1e-10
        _case("llt_mixed_40k", "factor", 40009, type="mixed", algo="llt", nrhs=8),
        # a non-symmetric system by H-LU
        _case("lu_f64_6k", "factor", 6007, type="f64", algo="lu", kernel="shifted",
              symmetric=False, leaf=100, nrhs=2),
        # repeated solves with one factor
        _case("solve_f64_20k", "solve", 20011, type="f64", algo="llt", nrhs=8),
        # one step of a hyperparameter fit: likelihood and gradient, forward and backward
        _case("gp_8k", "gp", 8000, height=4.0, type="mixed", algo="llt"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "gemv_host", "assemble", "factor", "factor", "solve", "gp"])
    leaf = rng.choice([48, 64, 100, 128, 200, 256])
    if kind in ("gemv", "gemv_host"):
        n = _log_uniform(rng, 1000, 150000 if kind == "gemv" else 40000)
        type_ = rng.choice(["f64", "f64", "f32", "c128"]) if kind == "gemv" else "f64"
        if type_ == "c128":
            n = min(n, _log_uniform(rng, 1000, 20000))
            return _case("", kind, n, leaf=rng.choice([64, 100, 128]), nrhs=rng.choice([1, 1, 3, 16]),
                         kernel="helmholtz", type=type_, symmetric=False)
        sym = rng.random() < 0.7
        return _case("", kind, n, leaf=leaf, nrhs=rng.choice([1, 1, 1, 2, 5, 8, 16, 65]),
                     kernel=rng.choice(["exponential", "gaussian"]) if sym else "shifted", type=type_,
                     symmetric=sym)
    if kind == "assemble":
        return _case("", kind, _log_uniform(rng, 1000, 80000), leaf=leaf, nrhs=rng.choice([1, 8, 65]),
                     kernel=rng.choice(["exponential", "gaussian", "dlength"]))
    if kind == "gp":
        n = _log_uniform(rng, 1000, 9000)
        return _case("", kind, n, height=n / rng.choice([2000.0, 4000.0]), leaf=rng.choice([64, 100, 128]),
                     type="mixed", algo="llt")
    if kind == "factor" and rng.random() < 0.3:
        return _case("", kind, _log_uniform(rng, 1000, 6000), leaf=rng.choice([64, 100, 128]),
                     kernel="shifted", symmetric=False, algo="lu", nrhs=rng.choice([1, 2, 7]))
    return _case("", kind, _log_uniform(rng, 1000, 24000), leaf=rng.choice([64, 100, 128]),
                 type=rng.choice(["f64", "mixed"]) if kind == "factor" else "f64", algo="llt",
                 nrhs=rng.choice([1, 3, 8, 16]))


# ---- inputs --------------------------------------------------------------------
def _points(case, seed):
    """Uniform points on the cylinder, and the Helmholtz kernel's regularisation
    (the mean spacing of the points) and wave number (ten points per wavelength)."""
    u = np.random.default_rng(seed).random((case["n"], 2))
    th = 2.0 * math.pi * u[:, 0]
    p = np.empty((case["n"], 3))
    p[:, 0], p[:, 1], p[:, 2] = np.cos(th), np.sin(th), case["height"] * u[:, 1]
    reg = 0.5 * math.sqrt(2.0 * math.pi * case["height"] / case["n"])
    return p, reg, 2.0 * math.pi / (10.0 * reg)


def _dtype(case):
    return {"f32": torch.float32, "c128": torch.complex128}.get(case["type"], torch.float64)


def _vectors(case, seed):
    """nrhs standard normal vectors, one per row, on the device."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7 + 1)
    return torch.randn(case["nrhs"], case["n"], dtype=_dtype(case), device="cuda", generator=g)


def _new_matrix(case, tree):
    vt = {"f32": hmat_amd.HMAT_SIMPLE_PRECISION, "c128": hmat_amd.HMAT_DOUBLE_COMPLEX}
    return hmat_amd.HMatrix(tree, eta=ETA, lower_symmetric=case["symmetric"], lowrank_eps=EPS,
                            value_type=vt.get(case["type"], hmat_amd.HMAT_DOUBLE_PRECISION))


def _assemble(case, h, reg, wavenumber):
    if case["kernel"] == "helmholtz":
        h.assemble(kind=KINDS["helmholtz"], wavenumber=wavenumber, reg=reg, nugget=1.0, eps=EPS,
                   method="aca_partial")
    else:
        h.assemble(kind=KINDS[case["kernel"]], length=LENGTH, eps=EPS, shift=SHIFT,
                   nugget=0.0 if case["kernel"] == "dlength" else _nugget(case))


def _nugget(case):
    # the non-symmetric kernel's diagonal is not its largest entry: regularised
    # more, as the H-LU tests do
    return 0.2 if case["kernel"] == "shifted" else NUGGET


_ALGO = {"llt": hmat_amd.FACT_LLT, "lu": hmat_amd.FACT_LU}


def prepare(case, seed):
    pts, reg, wk = _points(case, seed)
    s = {"case": case, "tree": hmat_amd.ClusterTree(pts, case["leaf"]), "reg": reg, "wk": wk}
    kind = case["kind"]
    s["stream"] = torch.cuda.Stream()
    if kind == "gp":
        g = np.random.default_rng(seed + 1)
        # observations with unit variance along the cylinder plus noise
        y = np.sin(3.0 * pts[:, 0]) + np.cos(2.0 * pts[:, 2]) + 0.1 * g.standard_normal(case["n"])
        s["y"] = torch.tensor(y, device="cuda")
        s["seed"] = int(seed)
    else:
        s["x"] = _vectors(case, seed)
        s["out"] = torch.zeros_like(s["x"])
    if kind in ("gemv", "gemv_host", "solve"):
        h = _new_matrix(case, s["tree"])
        _assemble(case, h, reg, wk)
        if kind == "solve":
            h.factorize(_ALGO[case["algo"]])
        s["h"] = h
        if kind == "gemv_host":
            s["xh"] = np.asfortranarray(s["x"].cpu().numpy().T)
        else:
            h.set_stream(s["stream"].cuda_stream)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind, nrhs = case["kind"], case["nrhs"]
    precision = 1 if case["type"] == "f32" else 0
    if kind == "gemv":
        s["h"].gemv_device(s["x"].data_ptr(), s["out"].data_ptr(), nrhs, precision=precision)
        return s["out"]
    if kind == "gemv_host":
        return s["h"].gemv(s["xh"])
    if kind == "solve":
        with torch.cuda.stream(s["stream"]):
            s["out"].copy_(s["x"])
        s["h"].solve_device(s["out"].data_ptr(), nrhs)
        return s["out"]
    if kind == "gp":
        length = torch.tensor(LENGTH, dtype=torch.float64, requires_grad=True)
        nugget = torch.tensor(NUGGET, dtype=torch.float64, requires_grad=True)
        y = s["y"].detach().requires_grad_(True)
        nll = gp_nll(length, nugget, y, s["tree"], eps=EPS, probes=GP_PROBES, seed=s["seed"])
        nll.backward()
        return {"nll": nll.detach(), "dlength": length.grad, "dnugget": nugget.grad, "dy": y.grad}
    h = _new_matrix(case, s["tree"])
    h.set_stream(s["stream"].cuda_stream)
    _assemble(case, h, s["reg"], s["wk"])
    if kind == "assemble":
        h.gemv_device(s["x"].data_ptr(), s["out"].data_ptr(), nrhs, precision=precision)
        s["stream"].synchronize()
        h.close()
        return s["out"]
    mixed = case["type"] == "mixed"
    h.factorize(_ALGO[case["algo"]], mixed=mixed)
    with torch.cuda.stream(s["stream"]):
        s["out"].copy_(s["x"])
    if mixed:
        h.solve_refined_device(s["out"].data_ptr(), nrhs, tol=1e-10, max_iter=60)
    else:
        h.solve_device(s["out"].data_ptr(), nrhs)
    out = {"x": s["out"]}
    if case["algo"] == "llt" and not mixed:
        out["logdet"] = 2.0 * h.logdet()
    s["stream"].synchronize()
    h.close()
    return out


# ---- what a pass cannot do without ------------------------------------------------
def _entries(case):
    """Stored entries of the compressed matrix: full leaves, and admissible
    blocks at the kernel's mean rank; and sum over leaves of n + 2 m."""
    pts, _, _ = _points(case, 0)
    h = _new_matrix(case, hmat_amd.ClusterTree(pts, case["leaf"]))
    p = h.partition().astype(np.int64)
    h.close()
    full = (p[p[:, 4] == 0][:, 1] * p[p[:, 4] == 0][:, 3]).sum()
    rk = p[p[:, 4] == 1]
    return int(full), int((rk[:, 1] + rk[:, 3]).sum() * MEAN_RANK[case["kernel"]])


def work(case):
    n, nrhs, kind = case["n"], case["nrhs"], case["kind"]
    full, rk = _entries(case)
    size = {"f32": 4, "c128": 16}.get(case["type"], 8)
    flop = 8 if case["type"] == "c128" else 2
    both = 2 if case["symmetric"] else 1
    vectors = 2 * n * nrhs * size
    product = flop * both * (full + rk) * nrhs
    if kind in ("gemv", "gemv_host"):
        return {"bytes": (full + rk) * size + vectors, "flops": product}
    if kind == "assemble":
        # entries written once and read once by the product; about 30 operations
        # per evaluated entry (distance, square root, exponential)
        return {"bytes": 2 * (full + rk) * size + vectors, "flops": 30 * (full + rk) + product}
    if kind == "solve":
        return {"bytes": (full + rk) * size + vectors, "flops": 2 * product}
    # the matrix written by the assembly, read by the factorisation, the factor
    # written and read by one solve; operations of an H-factorisation
    # n (k log2(n / leaf))^2, twice for LU
    levels = max(1.0, math.log2(n / case["leaf"]))
    ops = 4.0 * n * (MEAN_RANK[case["kernel"]] * levels) ** 2 * (1 if case["symmetric"] else 2)
    ops += n * case["leaf"] ** 2
    if kind == "gp":
        nrhs = GP_PROBES + 1
    factor = 4 if case["type"] == "mixed" else 8
    return {"bytes": (full + rk) * (16 + 2 * factor) + 2 * n * nrhs * 8,
            "flops": int(ops + 2 * flop * both * (full + rk) * nrhs)}


def tolerance(case):
    kind, type_ = case["kind"], case["type"]
    if kind in ("gemv", "gemv_host"):
        # 64-bit sums of the same stored matrix; in 32 bits the stored entries
        # and the result are rounded (6e-8 each)
        return {"rel": 1e-6 if type_ == "f32" else 1e-11}
    if kind == "assemble":
        # four times the distance of the compressed product to the exact one (1e-4)
        return {"rel": 4e-4}
    if kind == "gp":
        # the log-determinant of a factor compressed at eps and rounded to 32
        # bits: 2e-6 to 3e-5 off the exact one
        return {"rel": 1e-4}
    if type_ == "mixed":
        # refined to a residual of 1e-10: four times that
        return {"rel": 4e-10}
    # a factor compressed at eps applied once: its solutions are 1e-3 (N = 4,000)
    # to 4e-3 (N = 20,000) off both the exact one and the assembled matrix's own
    return {"rel": 2e-3 + 6e-7 * case["n"]}


# ---- the same in plain torch, 64 bits ----------------------------------------------
def _tree_order(pts, leaf):
    """User index of every position of the cluster tree's numbering: median
    bisection along the longest side of the bounding box, the last axis
    avoided unless it is 1.2 times longer than the next."""
    idx = np.arange(len(pts))

    def divide(o, size, axis):
        if size <= leaf:
            return
        q = pts[idx[o:o + size]]
        ext = q.max(axis=0) - q.min(axis=0)
        by = np.argsort(ext, kind="stable")
        d = int(by[-1])
        if axis >= 0 and d == axis and ext[by[-1]] <= 1.2 * ext[by[-2]]:
            d = int(by[-2])
        idx[o:o + size] = idx[o:o + size][np.argsort(q[:, d], kind="stable")]
        divide(o, size // 2, d)
        divide(o + size // 2, size - size // 2, d)
    divide(0, len(pts), -1)
    return idx


def _rows(case, P, r, reg, wk, kernel=None, nugget=None):
    """Rows r of the exact matrix over the points P (device, n x 3)."""
    kernel = kernel or case["kernel"]
    d2 = torch.zeros(len(r), len(P), dtype=torch.float64, device=P.device)
    for a in range(3):
        t = P[r, a][:, None] - P[None, :, a]
        if kernel == "shifted" and a == 2:
            t -= SHIFT
        d2 += t * t
    at = (torch.arange(len(r), device=P.device), r)
    if kernel == "helmholtz":
        d = torch.sqrt(d2 + reg * reg)
        k = torch.exp(1j * wk * d) / (4.0 * math.pi * d)
        k[at] = 1.0 / (4.0 * math.pi * reg) + 1.0
        return k
    if kernel == "gaussian":
        k = torch.exp(-d2 / LENGTH ** 2)
    elif kernel == "dlength":
        d = torch.sqrt(d2)
        return d / LENGTH ** 2 * torch.exp(-d / LENGTH)
    else:
        k = torch.exp(-torch.sqrt(d2) / LENGTH)
    k[at] += _nugget(case) if nugget is None else nugget
    return k


def _product(case, P, X, reg, wk, **kw):
    """K X for X (n x c), rows of K formed a slab at a time."""
    n = len(P)
    slab = max(1, min(n, (1 << 28) // n))
    return torch.cat([_rows(case, P, torch.arange(i, min(n, i + slab), device=P.device), reg, wk, **kw) @ X
                      for i in range(0, n, slab)])


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind in ("factor", "solve", "gp") and n > 22000:
        return None
    pts, reg, wk = _points(case, seed)
    if kind not in ("gemv_host", "gp"):
        pts = pts[_tree_order(pts, case["leaf"])]
    P = torch.tensor(pts, device="cuda")
    if kind == "gp":
        s = prepare(case, seed)
        y = s["y"]
        rng = np.random.default_rng(int(seed))
        Z = torch.tensor(np.where(rng.integers(0, 2, size=(n, GP_PROBES)) == 0, -1.0, 1.0), device="cuda")
        L = torch.linalg.cholesky(_rows(case, P, torch.arange(n, device="cuda"), reg, wk))
        S = torch.cholesky_solve(torch.cat([y[:, None], Z], dim=1), L)
        a, S = S[:, 0], S[:, 1:]
        D = _product(case, P, torch.cat([a[:, None], Z], dim=1), reg, wk, kernel="dlength")
        nll = 0.5 * (y @ a) + torch.log(torch.diagonal(L)).sum() + 0.5 * n * math.log(2.0 * math.pi)
        return {"nll": nll, "dlength": 0.5 * ((S * D[:, 1:]).sum() / GP_PROBES - a @ D[:, 0]).cpu(),
                "dnugget": 0.5 * ((Z * S).sum() / GP_PROBES - a @ a).cpu(), "dy": a}
    X = _vectors(case, seed).T
    if case["type"] == "f32":
        X = X.double()
    if kind in ("gemv", "gemv_host", "assemble"):
        y = _product(case, P, X, reg, wk)
        return y.cpu().numpy() if kind == "gemv_host" else y.T.contiguous()
    K = _rows(case, P, torch.arange(n, device="cuda"), reg, wk)
    if case["algo"] == "lu":
        return {"x": torch.linalg.solve(K, X).T.contiguous()}
    L = torch.linalg.cholesky(K)
    x = torch.cholesky_solve(X, L).T.contiguous()
    if kind == "solve":
        return x
    if case["type"] == "mixed":
        return {"x": x}
    return {"x": x, "logdet": 2.0 * torch.log(torch.diagonal(L)).sum().item()}
