"""The work that programs built on this library have it do, as timed cases.

Each case is one call, or the short sequence of calls that always go together,
through the Python binding (``darray_optimizer_amd.Handle``), on inputs that
are resident on the GPU, as the C ABI takes them.  The path is the kernel-SVM
pipeline: RBF range finder (one problem or a batch), its error, the Nystrom
factor, the SVM solver on that factor, and the regularised core solve.

* ``listed()``        the cases, by name
* ``draw(rng)``       one more case of the same ranges
* ``prepare(c, s)``   what the program holds before the call, made from seed s
* ``run(state)``      one pass; returns everything the calls compute
* ``work(c)``         bytes and flops that no implementation can do without
* ``exact(c, s)``     the same outputs in 64 bits by plain torch, where defined
"""
from __future__ import annotations

import math
import random

import torch

import darray_optimizer_amd as dh

F64 = torch.float64
PREC = {"f64": dh.DH_PREC_F64, "bf16": dh.DH_PREC_BF16, "f16": dh.DH_PREC_F16,
        "fp8": dh.DH_PREC_FP8}


def listed():
    return [
        # The headline solve of bench.py: 65536 points, rank 256 + 16, two
        # power iterations, FP16 passes (the mixed mode at FP64's error).
        {"name": "lra_f16_65536", "kind": "lra", "prec": "f16", "n": 65536, "d": 128, "l": 272,
         "q": 2, "labels": False},
        # The same solve in double precision, the reference of every error ratio.
        {"name": "lra_f64_65536", "kind": "lra", "prec": "f64", "n": 65536, "d": 128, "l": 272,
         "q": 2, "labels": False},
        # The single-machine workload of the CPU baseline (n = 8192, l = 138).
        {"name": "lra_f64_8192", "kind": "lra", "prec": "f64", "n": 8192, "d": 64, "l": 138,
         "q": 1, "labels": False},
        # The smallest problem of the batched workload run alone, with labels
        # and an odd size: launches and latency count.
        {"name": "lra_bf16_2051", "kind": "lra", "prec": "bf16", "n": 2051, "d": 16, "l": 42,
         "q": 1, "labels": True},
        # More than 256 features: K is formed in row blocks (double precision).
        {"name": "lra_f64_wide", "kind": "lra", "prec": "f64", "n": 9000, "d": 600, "l": 74,
         "q": 1, "labels": True},
        # One-vs-rest / per-gamma problems of mixed sizes in one call, planned
        # once: n ~ U{2048..32768}, d in {16, 64, 256}, k in {32, 64, 128, 256}.
        {"name": "lra_batched_f16_24", "kind": "batched", "prec": "f16", "count": 24,
         "n_min": 2048, "n_max": 32768, "q": 1},
        # The largest problems: FP8 distances, rank 512 + 32, 256 features.
        {"name": "lra_fp8_131072", "kind": "lra", "prec": "fp8", "n": 131072, "d": 256, "l": 544,
         "q": 1, "labels": False},
        # Error of a finished solve, ||K - Q W^T|| and ||K|| (Knorm).
        {"name": "knorm_65536", "kind": "knorm", "n": 65536, "d": 128, "l": 272, "labels": False},
        # Nystrom factor of a finished solve at the headline size.
        {"name": "nystrom_65536", "kind": "nystrom", "n": 65536, "d": 128, "l": 272, "k": 256},
        # Barrier SVM training on a Nystrom factor, whole call.
        {"name": "svm_barrier_20000", "kind": "svm", "n": 20000, "d": 64, "k": 200, "C": 1.0},
        # Regularised core solve: kernel tile, Cholesky and two triangular
        # solves with 64 right-hand sides, double precision.
        {"name": "core_posv_f64_16384", "kind": "posv", "n": 16384, "d": 128, "nrhs": 64,
         "lam": 0.1},
        # The same core in single precision, the reference's type, at an odd
        # size: kernel tile and Cholesky factor.
        {"name": "core_potrf_f32_6001", "kind": "potrf32", "n": 6001, "d": 64, "lam": 1.0},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["lra", "lra", "lra", "lra_wide", "batched", "knorm", "nystrom", "svm",
                       "posv", "potrf32"])
    if kind == "lra":
        prec = rng.choice(["f64", "bf16", "f16", "fp8"])
        d = _log_int(rng, 16, 256)
        l = _log_int(rng, 16, min(272, 8 * d))
        n = _log_int(rng, max(1500, 4 * l), 65536)
        return {"kind": "lra", "prec": prec, "n": n, "d": d, "l": l, "q": rng.randint(0, 2),
                "labels": rng.random() < 0.5}
    if kind == "lra_wide":
        l = _log_int(rng, 16, 160)
        return {"kind": "lra", "prec": "f64", "n": _log_int(rng, 1500, 16384),
                "d": rng.randint(257, 700), "l": l, "q": rng.randint(0, 1),
                "labels": rng.random() < 0.5}
    if kind == "batched":
        return {"kind": "batched", "prec": rng.choice(["bf16", "f16"]), "count": rng.randint(6, 28),
                "n_min": 2048, "n_max": rng.choice([8192, 16384, 32768]), "q": rng.randint(0, 2)}
    if kind == "knorm":
        d = _log_int(rng, 16, 300)
        return {"kind": "knorm", "n": _log_int(rng, 2000, 65536), "d": d,
                "l": _log_int(rng, 16, min(272, 8 * d)), "labels": rng.random() < 0.5}
    if kind == "nystrom":
        l = _log_int(rng, 24, 272)
        return {"kind": "nystrom", "n": _log_int(rng, 3000, 65536), "d": _log_int(rng, 64, 256),
                "l": l, "k": rng.randint(max(1, l // 2), l)}
    if kind == "svm":
        return {"kind": "svm", "n": _log_int(rng, 2000, 40000), "d": _log_int(rng, 32, 128),
                "k": _log_int(rng, 24, 256), "C": rng.choice([0.5, 1.0, 2.0])}
    if kind == "posv":
        return {"kind": "posv", "n": _log_int(rng, 600, 16384), "d": _log_int(rng, 16, 256),
                "nrhs": _log_int(rng, 1, 128), "lam": rng.choice([0.1, 0.3, 1.0])}
    return {"kind": "potrf32", "n": _log_int(rng, 600, 16384), "d": _log_int(rng, 16, 256),
            "lam": rng.choice([1.0, 3.0])}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _mixture(g, n, d, centres, sigma, labels):
    """Gaussian mixture with centres in [-1, 1]^d, point per row (FP64), and
    +-1 labels by the parity of the point's centre."""
    ctr = 2.0 * torch.rand((centres, d), dtype=F64, device="cuda", generator=g) - 1.0
    which = torch.randint(0, centres, (n,), device="cuda", generator=g)
    X = ctr[which] + sigma * torch.randn((n, d), dtype=F64, device="cuda", generator=g)
    return X, ((1 - 2 * (which % 2)).to(F64) if labels else None)


def _lra_inputs(case, g):
    X, y = _mixture(g, case["n"], case["d"], 16, 0.25, case["labels"])
    Om = torch.randn((case["l"], case["n"]), dtype=F64, device="cuda", generator=g)
    return X, y, Om, 0.5 / case["d"]


def _batch_inputs(case, seed):
    g = _gen(seed)
    out = []
    # The sizes are the case's own (the same for every seed); the seed makes the values.
    sizes = random.Random(case["count"] * 7919 + case["n_max"] + case["q"])
    for _ in range(case["count"]):
        n = sizes.randint(case["n_min"], case["n_max"])
        d = sizes.choice([16, 64, 256])
        l = sizes.choice([32, 64, 128, 256]) + 10
        X, y = _mixture(g, n, d, 4, 0.3, True)
        Om = torch.randn((l, n), dtype=F64, device="cuda", generator=g)
        out.append((X, y, Om, 1.0 / d))
    return out


def _rows(X, j0, j1, gamma, y=None, XB=None, yB=None):
    """Rows j0..j1 of K(X, XB) in FP64 by plain torch."""
    XB = X if XB is None else XB
    A = X[j0:j1]
    D = torch.mm(A, XB.t())
    D.mul_(-2.0).add_((A * A).sum(1)[:, None]).add_((XB * XB).sum(1)[None, :])
    D.clamp_(min=0.0).mul_(-gamma).exp_()
    if y is not None:
        D.mul_(y[j0:j1, None]).mul_((y if yB is None else yB)[None, :])
    return D


def _kernel_times(X, gamma, P, y=None):
    """K P for the (l, n) tensor P (n x l column-major), as an (l, n) tensor."""
    n = X.shape[0]
    out = torch.empty_like(P)
    Pt = P.t().contiguous()
    step = max(256, min(n, (1 << 28) // n))
    for j0 in range(0, n, step):
        j1 = min(n, j0 + step)
        out[:, j0:j1] = torch.mm(_rows(X, j0, j1, gamma, y), Pt).t()
    return out


def _upper_inverse(R):
    return torch.linalg.solve_triangular(R, torch.eye(R.shape[0], dtype=F64, device="cuda"),
                                         upper=True)


def _orth(Y):
    """Q of the QR factorisation with positive diagonal, (l, n) tensors."""
    Yt = Y.t().contiguous()
    for _ in range(3):
        R = torch.linalg.cholesky(torch.mm(Yt.t(), Yt), upper=True)
        Yt = torch.mm(Yt, _upper_inverse(R))
    return Yt.t().contiguous()


def _basis(g, n, d, l, labels):
    """Points, labels, an orthonormal basis Q from l landmark columns of K, and W = K Q."""
    X, y = _mixture(g, n, d, 16, 0.25, labels)
    gamma = 0.5 / d
    marks = torch.randperm(n, device="cuda", generator=g)[:l]
    Y = _rows(X, 0, n, gamma, y, X[marks], None if y is None else y[marks]).t().contiguous()
    Q = _orth(Y)
    return X, y, gamma, Q, _kernel_times(X, gamma, Q, y)


def prepare(case, seed):
    kind, g, h = case["kind"], _gen(seed), dh.Handle(0)
    if kind == "lra":
        X, y, Om, gamma = _lra_inputs(case, g)
        return {"kind": kind, "h": h, "X": X, "y": y, "Om": Om, "gamma": gamma, "q": case["q"],
                "prec": PREC[case["prec"]], "Q": torch.empty_like(Om), "W": torch.empty_like(Om)}
    if kind == "batched":
        probs = [{"X": X, "y": y, "Omega": Om, "gamma": gamma, "q": case["q"],
                  "Q": torch.empty_like(Om), "W": torch.empty_like(Om)}
                 for X, y, Om, gamma in _batch_inputs(case, seed)]
        return {"kind": kind, "h": h, "probs": probs, "prec": PREC[case["prec"]]}
    n, d = case["n"], case["d"]
    if kind == "knorm":
        X, y, gamma, Q, W = _basis(g, n, d, case["l"], case["labels"])
        return {"kind": kind, "h": h, "X": X, "y": y, "gamma": gamma, "Q": Q, "W": W}
    if kind == "nystrom":
        _, _, _, Q, W = _basis(g, n, d, case["l"], True)
        k = case["k"]
        return {"kind": kind, "h": h, "Q": Q, "W": W, "k": k,
                "Z": torch.empty((k, n), dtype=F64, device="cuda"),
                "lam": torch.empty(k, dtype=F64, device="cuda")}
    if kind == "svm":
        X, y = _mixture(g, n, d, 16, 0.25, True)
        gamma = 0.5 / d
        marks = torch.randperm(n, device="cuda", generator=g)[:case["k"]]
        Kl = _rows(X, 0, n, gamma, y, X[marks], y[marks])
        R = torch.linalg.cholesky(Kl[marks] + 1e-6 * torch.eye(case["k"], dtype=F64, device="cuda"),
                                  upper=True)
        Z = torch.mm(Kl, _upper_inverse(R)).t().contiguous()
        return {"kind": kind, "h": h, "Z": Z, "y": y, "C": case["C"],
                "a": torch.empty(n, dtype=F64, device="cuda")}
    X, _ = _mixture(g, n, d, 16, 0.25, False)
    if kind == "posv":
        B = torch.randn((case["nrhs"], n), dtype=F64, device="cuda", generator=g)
        return {"kind": kind, "h": h, "X": X, "gamma": 0.5 / d, "lam": case["lam"], "B": B,
                "S": torch.empty_like(B), "K": torch.empty((n, n), dtype=F64, device="cuda")}
    return {"kind": kind, "h": h, "X": X.float(), "gamma": 0.5 / d, "lam": case["lam"],
            "K": torch.empty((n, n), dtype=torch.float32, device="cuda")}


def run(s):
    kind, h = s["kind"], s["h"]
    if kind == "lra":
        info = h.lra(s["X"], s["Om"], s["gamma"], s["q"], s["Q"], s["W"], y=s["y"], prec=s["prec"])
        return {"Q": s["Q"], "W": s["W"], "info": info}
    if kind == "batched":
        info, each = h.lra_batched(s["probs"], prec=s["prec"])
        return {"info": info, "each": torch.tensor(each),
                "Q": [p["Q"] for p in s["probs"]], "W": [p["W"] for p in s["probs"]]}
    if kind == "knorm":
        e2, k2 = h.lra_error(s["X"], s["gamma"], s["Q"], s["W"], y=s["y"])
        return {"err2": e2, "norm2": k2}
    if kind == "nystrom":
        info = h.nystrom(s["Q"], s["W"], s["k"], s["Z"], s["lam"])
        return {"Z": s["Z"], "lam": s["lam"], "info": info}
    if kind == "svm":
        stats, f = h.svm_barrier(s["Z"], s["y"], s["C"], s["a"])
        return {"a": s["a"], "f": f, "stats": torch.tensor(stats)}
    K = s["K"]
    h.rbf_tile(s["X"], s["X"], s["gamma"], K)
    K.diagonal().add_(s["lam"])
    if kind == "posv":
        s["S"].copy_(s["B"])
        info = h.posv(K, s["S"])
        return {"U": K, "X": s["S"], "info": info}
    return {"U": K, "info": h.potrf(K)}


# ------------------------------------------------------------------- work

def _lra_work(n, d, l, q):
    # q + 2 passes of n^2 distances and n^2 x l products, q + 1 orthonormal bases.
    flops = (q + 2) * 2.0 * n * n * (d + l) + (q + 1) * 4.0 * n * l * l
    return flops, 8.0 * (n * d + 3.0 * n * l)


def work(case):
    kind = case["kind"]
    if kind == "lra":
        f, b = _lra_work(case["n"], case["d"], case["l"], case["q"])
        return {"bytes": b, "flops": f}
    if kind == "batched":
        sizes = random.Random(case["count"] * 7919 + case["n_max"] + case["q"])
        f = b = 0.0
        for _ in range(case["count"]):
            n = sizes.randint(case["n_min"], case["n_max"])
            d = sizes.choice([16, 64, 256])
            l = sizes.choice([32, 64, 128, 256]) + 10
            df, db = _lra_work(n, d, l, case["q"])
            f, b = f + df, b + db
        return {"bytes": b, "flops": f}
    n = case["n"]
    if kind == "knorm":
        d, l = case["d"], case["l"]
        # The distances are symmetric; the products Q W^T are not.
        return {"bytes": 8.0 * n * (d + 2 * l), "flops": 1.0 * n * n * d + 2.0 * n * n * l}
    if kind == "nystrom":
        l, k = case["l"], case["k"]
        return {"bytes": 8.0 * n * (2 * l + k), "flops": 2.0 * n * l * l + 2.0 * n * l * k + 9.0 * l**3}
    if kind == "svm":
        # Some hundred Newton systems, each at least one product with Z and Z^T.
        return {"bytes": 100.0 * 8.0 * n * case["k"], "flops": 100.0 * 4.0 * n * case["k"]}
    d = case["d"]
    if kind == "posv":
        return {"bytes": 8.0 * n * n + 8.0 * n * (d + 2 * case["nrhs"]),
                "flops": 1.0 * n * n * d + n**3 / 3.0 + 2.0 * n * n * case["nrhs"]}
    return {"bytes": 4.0 * n * n + 4.0 * n * d, "flops": 1.0 * n * n * d + n**3 / 3.0}


# ------------------------------------------------------------------ exact

def _lra_exact(X, y, Om, gamma, q):
    Y = _kernel_times(X, gamma, Om, y)
    for _ in range(q):
        Y = _kernel_times(X, gamma, _orth(Y), y)
    Q = _orth(Y)
    return Q, _kernel_times(X, gamma, Q, y)


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "lra":
        if case["n"] > 65536:
            return None
        X, y, Om, gamma = _lra_inputs(case, g)
        Q, W = _lra_exact(X, y, Om, gamma, case["q"])
        # Single columns of a 16-bit or FP8 basis are not those of the exact
        # one (the small singular directions are rounding), so only W is held to it.
        return {"Q": Q if case["prec"] == "f64" else None,
                "W": W if case["prec"] != "fp8" else None, "info": None}
    if kind == "batched":
        got = [_lra_exact(X, y, Om, gamma, case["q"])
               for X, y, Om, gamma in _batch_inputs(case, seed)]
        return {"info": None, "each": None, "Q": [None for _ in got], "W": [W for _, W in got]}
    n, d = case["n"], case["d"]
    if kind == "knorm":
        X, y, gamma, Q, W = _basis(g, n, d, case["l"], case["labels"])
        e2 = k2 = 0.0
        Wc = W.contiguous()
        step = max(256, min(n, (1 << 28) // n))
        for j0 in range(0, n, step):
            j1 = min(n, j0 + step)
            Kb = _rows(X, j0, j1, gamma, y)
            k2 += float((Kb * Kb).sum())
            Kb.sub_(torch.mm(Q[:, j0:j1].t().contiguous(), Wc))
            e2 += float((Kb * Kb).sum())
        return {"err2": e2, "norm2": k2}
    if kind == "nystrom":
        _, _, _, Q, W = _basis(g, n, d, case["l"], True)
        M = torch.mm(Q, W.t().contiguous())
        lam = torch.linalg.eigvalsh(0.5 * (M + M.t())).flip(0)[:case["k"]]
        return {"Z": None, "lam": lam, "info": None}  # Z's columns have no set sign
    if kind == "svm":
        return None  # the iterates' end point, not the optimum, is what the solver returns
    X, _ = _mixture(g, n, d, 16, 0.25, False)
    if kind == "posv":
        B = torch.randn((case["nrhs"], n), dtype=F64, device="cuda", generator=g)
        K = _rows(X, 0, n, 0.5 / d)
        low = torch.tril(K, -1)
        K.diagonal().add_(case["lam"])
        U = torch.linalg.cholesky(K, upper=True)
        S = torch.linalg.solve_triangular(U.t().contiguous(), B.t().contiguous(), upper=False)
        S = torch.linalg.solve_triangular(U, S, upper=True)
        # Column-major storage: row j of the tensor is column j of the matrix.
        return {"U": torch.triu(U).t() + low.t(), "X": S.t().contiguous(), "info": None}
    X = X.float().double()
    K = _rows(X, 0, n, 0.5 / d)
    low = torch.tril(K, -1)
    K.diagonal().add_(case["lam"])
    U = torch.linalg.cholesky(K, upper=True)
    return {"U": torch.triu(U).t() + low.t(), "info": None}
