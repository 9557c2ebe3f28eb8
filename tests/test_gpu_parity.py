"""HIP path vs the FP64 oracle and the golden vectors, through the C ABI.

Tolerances are relative Frobenius errors written per test: FP64 paths must
agree with the oracle to <= 1e-10 (the path's stated bar; most are far
tighter), FP32 paths to FP32 rounding."""
from pathlib import Path

import numpy as np
import pytest

import darray_optimizer_amd as dh
import oracle as orc

pytestmark = pytest.mark.gpu
G = np.load(Path(__file__).resolve().parent / "golden" / "golden.npz")


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(b), 1e-300))


def dev_pts(X, dtype=None):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(X))
    return (t.to(dtype) if dtype else t).cuda()


def dev_vec(v, dtype=None):
    import torch
    if v is None:
        return None
    t = torch.from_numpy(np.ascontiguousarray(v))
    return (t.to(dtype) if dtype else t).cuda()


def dev_mat(A, dtype=None):
    return dh.to_dev(np.asarray(A, dtype=np.float64), dtype)


def empty_mat(m, n, dtype):
    import torch
    return torch.zeros((n, m), dtype=dtype, device="cuda")


# ---------------------------------------------------------------- RBF tile

@pytest.mark.parametrize("m,n,d,labels", [(1, 1, 1, False), (64, 64, 16, True),
                                          (100, 77, 13, True), (130, 257, 130, False)])
def test_rbf_tile_f64(dev, m, n, d, labels):
    import torch
    rng = np.random.default_rng(m * 1000 + n)
    Xi, Xj = rng.uniform(0, 1, (m, d)), rng.uniform(0, 1, (n, d))
    yi = rng.choice([-1.0, 1.0], m) if labels else None
    yj = rng.choice([-1.0, 1.0], n) if labels else None
    K = empty_mat(m, n, torch.float64)
    dev.rbf_tile(dev_pts(Xi), dev_pts(Xj), 1.0 / d, K, dev_vec(yi), dev_vec(yj))
    ref = orc.rbf_tile(Xi, Xj, 1.0 / d, yi, yj, clamp=True)
    assert rel(dh.from_dev(K), ref) < 1e-13


def test_rbf_tile_f32(dev):
    import torch
    rng = np.random.default_rng(5)
    Xi, Xj = rng.uniform(0, 1, (300, 64)), rng.uniform(0, 1, (200, 64))
    K = empty_mat(300, 200, torch.float32)
    dev.rbf_tile(dev_pts(Xi, torch.float32), dev_pts(Xj, torch.float32), 1 / 64.0, K)
    ref = orc.rbf_tile(Xi.astype(np.float32), Xj.astype(np.float32), 1 / 64.0, clamp=True)
    assert rel(dh.from_dev(K), ref) < 2e-6


def test_rbf_tile_golden(dev):
    import torch
    m, n = G["tile_Xi"].shape[0], G["tile_Xj"].shape[0]
    K = empty_mat(m, n, torch.float64)
    dev.rbf_tile(dev_pts(G["tile_Xi"]), dev_pts(G["tile_Xj"]), float(G["tile_gamma"]), K,
                 dev_vec(G["tile_yi"]), dev_vec(G["tile_yj"]))
    assert rel(dh.from_dev(K), G["tile_K"]) < 1e-14


# --------------------------------------------------------- fused projection

PROJ_SHAPES = [(1, 1, 1, 1), (64, 64, 64, 16), (100, 77, 13, 9), (129, 65, 33, 40),
               (300, 257, 130, 138), (200, 190, 200, 300), (96, 500, 128, 272),
               (150, 300, 257, 40), (70, 130, 600, 17)]  # d > 256: materialised K blocks


@pytest.mark.parametrize("m,n,d,l", PROJ_SHAPES)
def test_rbf_project_f64(dev, m, n, d, l):
    import torch
    rng = np.random.default_rng(m + 7 * n + 13 * d + l)
    Xi, Xj = rng.uniform(0, 1, (m, d)), rng.uniform(0, 1, (n, d))
    yi, yj = rng.choice([-1.0, 1.0], m), rng.choice([-1.0, 1.0], n)
    O = rng.standard_normal((n, l))
    Y0 = rng.standard_normal((m, l))
    Y = dev_mat(Y0)
    dev.rbf_project_f64(dev_pts(Xi), dev_pts(Xj), dev_mat(O), 1.0 / d, Y, dev_vec(yi),
                        dev_vec(yj), beta=0.5)
    ref = orc.rbf_project(Xi, Xj, O, 1.0 / d, yi, yj, beta=0.5, Y=Y0)
    assert rel(dh.from_dev(Y), ref) < 1e-12


def test_rbf_project_golden(dev):
    X = dev_pts(G["proj_X"])
    Y = dev_mat(G["proj_Y0"])
    dev.rbf_project_f64(X, X, dev_mat(G["proj_O"]), float(G["proj_gamma"]), Y,
                        beta=float(G["proj_beta"]))
    assert rel(dh.from_dev(Y), G["proj_Y"]) < 1e-14


# -------------------------------------------------------------------- GEMM

GEMM_SHAPES = [(1, 1, 1), (40, 40, 3000), (257, 129, 65), (2100, 2050, 40), (17, 300, 0)]


@pytest.mark.parametrize("ta", ["N", "T"])
@pytest.mark.parametrize("tb", ["N", "T"])
@pytest.mark.parametrize("m,n,k", GEMM_SHAPES)
def test_gemm_f64(dev, ta, tb, m, n, k):
    import torch
    rng = np.random.default_rng(m + n + k)
    A = rng.standard_normal((k, m) if ta == "T" else (m, k))
    B = rng.standard_normal((n, k) if tb == "T" else (k, n))
    C0 = rng.standard_normal((m, n))
    Cd = dev_mat(C0)
    dev.gemm(ta, tb, dev_mat(A), dev_mat(B), Cd, alpha=-1.5, beta=0.25)
    opA = A.T if ta == "T" else A
    opB = B.T if tb == "T" else B
    assert rel(dh.from_dev(Cd), -1.5 * opA @ opB + 0.25 * C0) < 1e-13


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T")])
def test_gemm_f32(dev, ta, tb):
    import torch
    rng = np.random.default_rng(11)
    m, n, k = 300, 200, 1500
    A = rng.standard_normal((k, m) if ta == "T" else (m, k)).astype(np.float32)
    B = rng.standard_normal((n, k) if tb == "T" else (k, n)).astype(np.float32)
    Cd = empty_mat(m, n, torch.float32)
    dev.gemm(ta, tb, dh.to_dev(A), dh.to_dev(B), Cd)
    opA = (A.T if ta == "T" else A).astype(np.float64)
    opB = (B.T if tb == "T" else B).astype(np.float64)
    assert rel(dh.from_dev(Cd), opA @ opB) < 1e-5


def test_syrk_upper_only(dev):
    rng = np.random.default_rng(12)
    A = rng.standard_normal((300, 150))
    C0 = rng.standard_normal((150, 150))
    Cd = dev_mat(C0)
    dev.syrk_ut(dev_mat(A), Cd, alpha=-1.0, beta=1.0)
    out = dh.from_dev(Cd)
    iu, il = np.triu_indices(150), np.tril_indices(150, -1)
    assert rel(out[iu], (C0 - A.T @ A)[iu]) < 1e-13
    np.testing.assert_array_equal(out[il], C0[il])


# -------------------------------------------------------------------- TRSM

@pytest.mark.parametrize("m", [45, 130, 300])
@pytest.mark.parametrize("side,trans", [("L", "T"), ("L", "N"), ("R", "N")])
def test_trsm_f64(dev, m, side, trans):
    rng = np.random.default_rng(m)
    U = np.triu(rng.standard_normal((m, m))) + 8 * np.eye(m)
    U_full = U + np.tril(rng.standard_normal((m, m)), -1)  # lower garbage must be ignored
    B = rng.standard_normal((m, 37)) if side == "L" else rng.standard_normal((53, m))
    Bd = dev_mat(B)
    dev.trsm(side, trans, "N", dev_mat(U_full), Bd, alpha=-0.5)
    ref = orc.trsm(side, trans, U, B, alpha=-0.5)
    assert rel(dh.from_dev(Bd), ref) < 1e-12


@pytest.mark.parametrize("side,trans,m,nrhs", [("L", "T", 700, 64), ("L", "N", 700, 64),
                                                ("L", "T", 300, 600), ("L", "N", 130, 513)])
def test_trsm_f64_block_sweep_and_recursion(dev, side, trans, m, nrhs):
    """Side-L solves with up to 512 right-hand sides run as a sweep over 64-row
    blocks; wider ones take the recursive halving.  Both against the oracle."""
    rng = np.random.default_rng(m + nrhs)
    U = np.triu(rng.standard_normal((m, m))) + 8 * np.eye(m)
    B = rng.standard_normal((m, nrhs))
    Bd = dev_mat(B)
    dev.trsm(side, trans, "N", dev_mat(U), Bd)
    assert rel(dh.from_dev(Bd), orc.trsm(side, trans, U, B)) < 1e-12


def test_trsm_golden(dev):
    U = G["trsm_U"]
    for side, trans, Bk, ref in (("L", "T", "trsm_B", "trsm_LUT"), ("L", "N", "trsm_B", "trsm_LUN"),
                                 ("R", "N", "trsm_Br", "trsm_RUN")):
        Bd = dev_mat(G[Bk])
        dev.trsm(side, trans, "N", dev_mat(U), Bd)
        assert rel(dh.from_dev(Bd), G[ref]) < 1e-13


def test_trsm_f32(dev):
    import torch
    rng = np.random.default_rng(13)
    U = (np.triu(rng.standard_normal((200, 200))) + 8 * np.eye(200)).astype(np.float32)
    B = rng.standard_normal((200, 64)).astype(np.float32)
    Bd = dh.to_dev(B)
    dev.trsm("L", "T", "N", dh.to_dev(U), Bd)
    ref = orc.trsm("L", "T", U.astype(np.float64), B.astype(np.float64))
    assert rel(dh.from_dev(Bd), ref) < 1e-5


# ---------------------------------------------------------------- Cholesky

@pytest.mark.parametrize("n,bs", [(1000, 256), (300, 64), (257, 256)])
def test_potrf_f64_min_ij_known_answer(dev, n, bs):
    # perftest_cholesky.cpp:46-53,76-84: U must be all ones; probe A(n-1,n-1) = 1.
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    A = np.minimum(i + 1, j + 1).astype(np.float64)
    Ad = dev_mat(A)
    assert dev.potrf(Ad, bs) == 0
    U = dh.from_dev(Ad)
    assert abs(U[n - 1, n - 1] - 1) <= 1e-5
    np.testing.assert_allclose(np.triu(U), np.triu(np.ones((n, n))), rtol=0, atol=1e-9)
    np.testing.assert_array_equal(np.tril(U, -1), np.tril(A, -1))


def test_potrf_f32_min_ij_probe(dev):
    import torch
    n = 512
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    A = np.minimum(i + 1, j + 1).astype(np.float32)
    Ad = dh.to_dev(A)
    assert dev.potrf(Ad, 256) == 0
    U = dh.from_dev(Ad)
    assert abs(U[n - 1, n - 1] - 1) <= 1e-5  # the reference's FP32 probe tolerance


def test_potrf_f64_vs_oracle_and_golden(dev):
    Ad = dev_mat(G["chol_A"])
    assert dev.potrf(Ad, 32) == 0
    assert rel(np.triu(dh.from_dev(Ad)), G["chol_U"]) < 1e-13
    rng = np.random.default_rng(14)
    M = rng.standard_normal((700, 700))
    A = M.T @ M / 700 + np.eye(700)
    Ad = dev_mat(A)
    assert dev.potrf(Ad, 256) == 0
    Uo, info = orc.potrf_upper(A, 256)
    assert info == 0
    assert rel(np.triu(dh.from_dev(Ad)), np.triu(Uo)) < 1e-12


def test_potrf_test3_known_answer(dev):
    n = 10
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    m = np.where(i >= j, 1.0 + i + j, 0.0)
    Ad = dev_mat(m @ m.T)
    assert dev.potrf(Ad, 4) == 0
    np.testing.assert_allclose(np.triu(dh.from_dev(Ad)), m.T, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("bs", [64, 256])
@pytest.mark.parametrize("bad", [0, 23, 200, 299])
def test_potrf_reports_first_bad_minor(dev, bad, bs):
    # bs = 256: the FP64 diagonal block of order 256 is the register
    # factorisation; the last 44 columns and every bs = 64 block are not.
    rng = np.random.default_rng(15)
    M = rng.standard_normal((300, 300))
    A = M.T @ M + 300 * np.eye(300)
    A[bad, bad] = -1.0
    Ad = dev_mat(A)
    assert dev.potrf(Ad, bs) == bad + 1


def test_potrf_lookahead_orders_with_the_handle_stream(dev):
    """The look-ahead runs part of each trailing update on a second stream:
    it must start after work queued before the call on the handle's stream
    (here the copy that fills A) and finish before the call returns."""
    import torch
    rng = np.random.default_rng(16)
    n = 1500
    M = rng.standard_normal((n, n))
    A = M.T @ M / n + np.eye(n)
    src = dev_mat(A)
    side = torch.cuda.Stream()
    h = dh.Handle(0, stream=side)
    try:
        with torch.cuda.stream(side):
            Ad = torch.full_like(src, float("nan"))
            torch.cuda._sleep(2_000_000)  # keep the copy below queued behind other work
            Ad.copy_(src)
        assert h.potrf(Ad, 256) == 0
        side.synchronize()
        Uo, info = orc.potrf_upper(A, 256)
        assert info == 0
        assert rel(np.triu(dh.from_dev(Ad)), np.triu(Uo)) < 1e-12
    finally:
        h.close()


# ------------------------------------------------------------- CholeskyQR2

def test_cholqr2_golden(dev):
    Yd = dev_mat(G["qr_Y"])
    R = empty_mat(12, 12, __import__("torch").float64)
    assert dev.cholqr2(Yd, R) == 0
    assert rel(dh.from_dev(Yd), G["qr_Q"]) < 1e-12
    assert rel(dh.from_dev(R), G["qr_R"]) < 1e-12


@pytest.mark.parametrize("m,n", [(20000, 138), (3000, 1), (3000, 257), (5000, 272), (6000, 544),
                                 (5000, 300), (2503, 417), (4000, 600), (131, 130), (4099, 200),
                                 (70001, 129)])
def test_cholqr2_tall(dev, m, n):
    # n <= 272: register-resident Cholesky (257: one real column in the last
    # 16-block); n <= 544: one-workgroup Cholesky and the row solve as two
    # register solves around a GEMM (300, 417: ragged second block); n = 600:
    # blocked fallback.
    # 128 < n <= 272 also takes the register-blocked Gram: (131, 130) one slab
    # per 16 rows with a ragged last chunk, (70001, 129) ragged row slabs.
    import torch
    rng = np.random.default_rng(16)
    Y = rng.standard_normal((m, n)) @ np.diag(np.logspace(0, -4, n))
    Yd = dev_mat(Y)
    R = empty_mat(n, n, torch.float64)
    assert dev.cholqr2(Yd, R) == 0
    Q, Rh = dh.from_dev(Yd), dh.from_dev(R)
    assert np.linalg.norm(Q.T @ Q - np.eye(n)) < 1e-13
    assert rel(Q @ Rh, Y) < 1e-13
    np.testing.assert_array_equal(np.tril(Rh, -1), 0)
    _, Ro, info = orc.cholqr2(Y)
    assert info == 0 and rel(Rh, Ro) < 1e-10


@pytest.mark.parametrize("n", [10, 250, 400, 600])
def test_cholqr2_breakdown(dev, n):
    # Exactly dependent columns: every CholeskyQR variant must report breakdown
    # (for n = 250 and 400 in a late panel).
    rng = np.random.default_rng(17)
    Y = rng.standard_normal((2000, n))
    Y[:, (3 * n) // 4] = Y[:, 2]
    assert dev.cholqr2(dev_mat(Y)) > 0


@pytest.mark.parametrize("n", [30, 400])
def test_cholqr_shifted_fallback_ill_conditioned(dev, n):
    # kappa(Y) = 1e11 is beyond CholeskyQR2 (~u^{-1/2}); the shifted
    # CholeskyQR3 fallback must still return an orthonormal Q with QR = Y
    # (n = 400: the shifted Cholesky as two order-272 register blocks).
    import torch
    rng = np.random.default_rng(18)
    U, _ = np.linalg.qr(rng.standard_normal((4000, n)))
    V, _ = np.linalg.qr(rng.standard_normal((n, n)))
    Y = U @ np.diag(np.logspace(0, -11, n)) @ V.T
    Yd = dev_mat(Y)
    R = empty_mat(n, n, torch.float64)
    assert dev.cholqr2(Yd, R) == 0
    Q, Rh = dh.from_dev(Yd), dh.from_dev(R)
    assert np.linalg.norm(Q.T @ Q - np.eye(n)) < 1e-12
    assert rel(Q @ Rh, Y) < 1e-13


# ------------------------------------------------------------------ LRA

@pytest.mark.parametrize("q", [0, 1, 2])
@pytest.mark.parametrize("labels", [False, True])
def test_lra_f64_vs_oracle(dev, labels, q):
    # q = 2: the power iterations alternate the basis between Q and W and end in Q.
    import torch
    n, d, l = 1536, 64, 40
    X = dh.fill_uniform(0, d, n).T.copy()  # DArray set_uniform layout, points as rows
    Om = dh.fill_normal(1, n, l)
    y = np.where(np.arange(n) % 3 == 0, -1.0, 1.0) if labels else None
    Q = empty_mat(n, l, torch.float64)
    W = empty_mat(n, l, torch.float64)
    assert dev.lra(dev_pts(X), dev_mat(Om), 1.0 / d, q, Q, W, dev_vec(y)) == 0
    Qo, Wo, info = orc.lra(X, Om, 1.0 / d, q, y, orth="householder")
    assert info == 0
    Qg, Wg = dh.from_dev(Q), dh.from_dev(W)
    assert rel(Qg @ Wg.T, Qo @ Wo.T) < 1e-10  # QB with B = W^T, sign invariant
    assert rel(Qg @ Qg.T, Qo @ Qo.T) < 1e-10
    e2, k2 = dev.lra_error(dev_pts(X), 1.0 / d, Q, W, dev_vec(y))
    eo, ko = orc.lra_error(X, 1.0 / d, Qo, Wo, y)
    assert abs(k2 - ko) / ko < 1e-12
    assert abs(np.sqrt(e2 / k2) - np.sqrt(eo / ko)) <= 1e-10 + 1e-6 * np.sqrt(eo / ko)


def test_lra_above_256_features(dev):
    """Above 256 features the passes materialise K in row blocks (FP64); every
    precision runs them, so the low-precision requests return the FP64 result
    bit for bit."""
    import torch
    n, d, l = 700, 300, 24
    X = dh.fill_uniform(3, d, n).T.copy()
    Om = dh.fill_normal(4, n, l)
    y = np.where(np.arange(n) % 4 == 0, -1.0, 1.0)
    out = {}
    for prec in (dh.DH_PREC_F64, dh.DH_PREC_BF16, dh.DH_PREC_F16, dh.DH_PREC_FP8):
        Q = empty_mat(n, l, torch.float64)
        W = empty_mat(n, l, torch.float64)
        assert dev.lra(dev_pts(X), dev_mat(Om), 1.0 / d, 1, Q, W, dev_vec(y), prec=prec) == 0
        out[prec] = (dh.from_dev(Q), dh.from_dev(W))
    Qo, Wo, info = orc.lra(X, Om, 1.0 / d, 1, y, orth="householder")
    assert info == 0
    Qg, Wg = out[dh.DH_PREC_F64]
    assert rel(Qg @ Wg.T, Qo @ Wo.T) < 1e-10
    for prec in (dh.DH_PREC_BF16, dh.DH_PREC_F16, dh.DH_PREC_FP8):
        assert np.array_equal(out[prec][0], Qg) and np.array_equal(out[prec][1], Wg)


def test_lra_golden(dev):
    import torch
    X = G["lra_X"]
    n, l = X.shape[0], G["lra_Omega"].shape[1]
    Q = empty_mat(n, l, torch.float64)
    W = empty_mat(n, l, torch.float64)
    assert dev.lra(dev_pts(X), dev_mat(G["lra_Omega"]), float(G["lra_gamma"]), 1, Q, W) == 0
    Qg, Wg = dh.from_dev(Q), dh.from_dev(W)
    assert rel(Qg @ Wg.T, G["lra_QWt"]) < 1e-10


def test_lra_error_golden(dev):
    import torch
    X = G["lra_X"]
    Qo, Wo, _ = orc.lra(X, G["lra_Omega"], float(G["lra_gamma"]), 1)
    e2, k2 = dev.lra_error(dev_pts(X), float(G["lra_gamma"]), dev_mat(Qo), dev_mat(Wo))
    np.testing.assert_allclose([e2, k2], G["lra_err2"], rtol=1e-8, atol=1e-22)


def test_lra_f64_full_size_properties(dev):
    """n = 65536, d = 128, l = 272, q = 2 (the FP64 GPU configuration): the oracle
    cannot run here, so check size-independent properties."""
    import torch
    n, d, k, p, q = 65536, 128, 256, 16, 2
    l = k + p
    X = dh.fill_mixture(0, d, n, 16, 0.25)
    Om = dh.fill_normal(1, n, l)
    Xd = dev_pts(X)
    Q = empty_mat(n, l, torch.float64)
    W = empty_mat(n, l, torch.float64)
    assert dev.lra(Xd, dev_mat(Om), 0.5 / d, q, Q, W) == 0
    QtQ = (Q @ Q.T).cpu().numpy()
    assert np.linalg.norm(QtQ - np.eye(l)) < 1e-12
    e2, k2 = dev.lra_error(Xd, 0.5 / d, Q, W)
    w2 = float((W * W).sum())
    # Q orthonormal: ||K - QQ^T K||^2 = ||K||^2 - ||Q^T K||^2
    assert abs(e2 - (k2 - w2)) <= 1e-9 * k2
    assert 0 <= np.sqrt(e2 / k2) < 0.5


# ------------------------------------------------------------- core solve

def _rbf_core(n, d, seed=21, shift=1e-3):
    X = dh.fill_mixture(seed, d, n, 16, 0.25)
    return orc.rbf_tile(X, X, 0.5 / d) + shift * np.eye(n)


@pytest.mark.parametrize("n,nrhs,bs", [(700, 13, 256), (1000, 64, 128)])
def test_posv_f64_vs_oracle(dev, n, nrhs, bs):
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n))
    A = M.T @ M / n + np.eye(n)
    B = rng.standard_normal((n, nrhs))
    Ad, Bd = dev_mat(A), dev_mat(B)
    assert dev.posv(Ad, Bd, bs) == 0
    U, info = orc.potrf_upper(A, bs)
    Xo = orc.trsm("L", "N", np.triu(U), orc.trsm("L", "T", np.triu(U), B))
    assert info == 0 and rel(dh.from_dev(Bd), Xo) < 1e-10
    assert rel(np.triu(dh.from_dev(Ad)), np.triu(U)) < 1e-12


def test_posv_f64_reports_failure(dev):
    A = np.eye(50)
    A[30, 30] = -1.0
    assert dev.posv(dev_mat(A), dev_mat(np.ones((50, 2))), 16) == 31


def test_posv_mixed_rbf_core(dev):
    """FP32 Cholesky + FP64 refinement on an RBF core + 1e-3 I (kappa ~ 1e6)."""
    import torch
    n, nrhs = 2048, 16
    A = _rbf_core(n, 32)
    rng = np.random.default_rng(22)
    B = rng.standard_normal((n, nrhs))
    X = torch.zeros((nrhs, n), dtype=torch.float64, device="cuda")
    info, iters, berr = dev.posv_mixed(dev_mat(np.triu(A)), dev_mat(B), X, 256, 1e-10, 100)
    assert info == 0 and berr <= 1e-10, (iters, berr)
    Xh = dh.from_dev(X)
    R = B - A @ Xh
    anorm = np.linalg.norm(A)
    be = max(np.linalg.norm(R[:, j]) / (anorm * np.linalg.norm(Xh[:, j]) + np.linalg.norm(B[:, j]))
             for j in range(nrhs))
    assert be <= 1e-10
    Xref = np.linalg.solve(A, B)
    assert rel(Xh, Xref) <= 1e-10 * np.linalg.cond(A)


def test_posv_mixed_falls_back_to_fp64(dev):
    # Eigenvalues down to 1e-10 relative: FP32 Cholesky breaks down, FP64 does not.
    import torch
    rng = np.random.default_rng(23)
    n = 300
    Qm, _ = np.linalg.qr(rng.standard_normal((n, n)))
    A = (Qm * np.logspace(0, -10, n)) @ Qm.T
    A = (A + A.T) / 2
    B = rng.standard_normal((n, 3))
    X = torch.zeros((3, n), dtype=torch.float64, device="cuda")
    info, iters, berr = dev.posv_mixed(dev_mat(A), dev_mat(B), X, 64, 1e-10, 30)
    assert info == 0 and iters == -1
    assert rel(A @ dh.from_dev(X), B) < 1e-5


@pytest.mark.parametrize("fn", ["potrf", "posv"])
def test_lookahead_cholesky_with_split_k_updates(dev, fn):
    """bs = 1024 at n = 4096: the trailing updates have k = 1024 and few output
    tiles, so they split k on both the handle's stream and the look-ahead
    stream, which run concurrently with separate partials buffers."""
    import os
    n, bs = 4096, 1024
    rng = np.random.default_rng(31)
    M = rng.standard_normal((n, n))
    A = M.T @ M / n + np.eye(n)
    orc.set_threads(min(16, os.cpu_count() or 1))
    try:
        U, info = orc.potrf_upper(A, bs)
    finally:
        orc.set_threads(1)
    assert info == 0
    Ad = dev_mat(A)
    if fn == "potrf":
        assert dev.potrf(Ad, bs) == 0
    else:
        B = rng.standard_normal((n, 8))
        Bd = dev_mat(B)
        assert dev.posv(Ad, Bd, bs) == 0
        assert rel(A @ dh.from_dev(Bd), B) < 1e-10
    e = rel(np.triu(dh.from_dev(Ad)), np.triu(U))
    print(f"{fn} n={n} bs={bs}: factor vs oracle {e:.2e}", flush=True)
    assert e < 1e-12


def test_posv_mixed_max_iter_reached_falls_back(dev):
    """A tolerance the FP32 refinement cannot reach within one correction: the
    solve is redone in FP64 (iters = -1) and the returned X is the FP64 one."""
    import torch
    n = 400
    A = _rbf_core(n, 16)
    B = np.random.default_rng(24).standard_normal((n, 4))
    X = torch.zeros((4, n), dtype=torch.float64, device="cuda")
    info, iters, berr = dev.posv_mixed(dev_mat(np.triu(A)), dev_mat(B), X, 64, 1e-15, 1)
    assert info == 0 and iters == -1
    assert berr <= 1e3 * n * 2.0**-53
    assert rel(dh.from_dev(X), np.linalg.solve(A, B)) < 1e-6


def test_posv_mixed_diverging_refinement_falls_back(dev):
    """kappa = 1e9: u32 * kappa > 1, so FP32 refinement cannot converge (or the
    FP32 factorisation breaks down); either way the FP64 path answers."""
    import torch
    rng = np.random.default_rng(25)
    n = 300
    Qm, _ = np.linalg.qr(rng.standard_normal((n, n)))
    A = (Qm * np.logspace(0, -9, n)) @ Qm.T
    A = (A + A.T) / 2
    B = rng.standard_normal((n, 2))
    X = torch.zeros((2, n), dtype=torch.float64, device="cuda")
    info, iters, berr = dev.posv_mixed(dev_mat(A), dev_mat(B), X, 64, 1e-10, 30)
    print(f"kappa 1e9: info {info} iters {iters} berr {berr:.2e}", flush=True)
    assert info == 0 and iters == -1 and berr <= 1e-10


def test_posv_mixed_nan_rhs_is_reported(dev):
    """A NaN in B gives a non-finite backward error: never reported as converged."""
    import torch
    n = 128
    A = _rbf_core(n, 8)
    B = np.ones((n, 2))
    B[5, 1] = np.nan
    X = torch.zeros((2, n), dtype=torch.float64, device="cuda")
    with pytest.raises(dh.DHError) as ei:
        dev.posv_mixed(dev_mat(np.triu(A)), dev_mat(B), X, 64, 1e-10, 10)
    assert ei.value.status == -1003


@pytest.mark.parametrize("n", [2, 15, 16, 17, 31, 33, 96, 97, 112, 113, 209, 271])
def test_cholqr2_block_edges(dev, n):
    """The register Cholesky at the edges of its 16-column panels and of the
    deal of its blocks to the waves: Q^T Q = I, Q R = Y, R upper with a
    positive diagonal and equal to numpy's up to signs."""
    import torch
    rng = np.random.default_rng(n)
    Y = rng.standard_normal((1500, n)) * np.logspace(0, -3, n)
    Yd = dev_mat(Y)
    Rd = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    assert dev.cholqr2(Yd, Rd) == 0
    Q, R = dh.from_dev(Yd), dh.from_dev(Rd)
    assert np.linalg.norm(Q.T @ Q - np.eye(n)) < 1e-12
    assert rel(Q @ R, Y) < 1e-13
    assert np.all(np.diag(R) > 0) and np.all(np.tril(R, -1) == 0)
    assert rel(R, np.abs(np.diag(np.sign(np.diag(np.linalg.qr(Y)[1])))) @
               (np.sign(np.diag(np.linalg.qr(Y)[1]))[:, None] * np.linalg.qr(Y)[1])) < 1e-11


@pytest.mark.parametrize("bad", [1, 4, 5, 16, 17, 30, 47])
def test_cholqr2_reports_the_failing_pivot(dev, bad):
    """A zero column is the first failing pivot of its sweep, wherever it lies in
    the four-row steps and the panels; the shifted sweep then fails at the same
    place in its second pass or returns a completed basis status."""
    rng = np.random.default_rng(bad)
    Y = rng.standard_normal((400, 48))
    Y[:, bad - 1] = 0.0
    st = dev.cholqr2(dev_mat(Y))
    assert st > 0 and st % 1000000 == bad


@pytest.mark.parametrize("n,d,l,labels", [(17, 3, 5, True), (64, 16, 16, False),
                                          (65, 33, 1, False), (1000, 40, 96, True),
                                          (2051, 130, 200, True), (900, 70, 280, False),
                                          (300, 257, 20, True), (11700, 257, 3, False)])
def test_lra_passes_on_kept_kernel_values(dev, n, d, l, labels):
    """The FP64 range finder forms K once, from one triangle, and all its passes
    read it back: W must be K Q for the returned Q, as the one-launch pass forms
    it.  Both sum n products K_ij Q_jc, in different orders, so element
    (i, c) may differ by 2 n u (K |Q|)_ic; K is in (0, 1]."""
    import torch
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)) * 0.3
    y = dev_vec(rng.choice([-1.0, 1.0], n)) if labels else None
    Xd = dev_pts(X)
    Om = dev_mat(rng.standard_normal((n, l)))
    Q, W, P = (empty_mat(n, l, torch.float64) for _ in range(3))
    assert dev.lra(Xd, Om, 1.0 / d, 2, Q, W, y=y) == 0
    dev.rbf_project_f64(Xd, Xd, Q, 1.0 / d, P, yi=y, yj=y)
    A = empty_mat(n, l, torch.float64)
    dev.rbf_project_f64(Xd, Xd, Q.abs(), 1.0 / d, A)
    assert bool(((W - P).abs() <= 2 * n * 2.0**-53 * A).all())


def test_lra_in_two_threads_gives_the_same_bits():
    """Two handles at once: one holds the device's scratch buffer, the other
    forms K in every pass, and both return the bits of a call on its own."""
    import threading

    import torch
    rng = np.random.default_rng(5)
    X = dev_pts(rng.standard_normal((3000, 20)) * 0.3)
    Om = dev_mat(rng.standard_normal((3000, 40)))
    hs = [dh.Handle(0) for _ in range(2)]
    out = [[empty_mat(3000, 40, torch.float64) for _ in range(2)] for _ in range(3)]
    hs[0].lra(X, Om, 0.05, 1, *out[2])
    torch.cuda.synchronize()

    def work(i):
        for _ in range(20):
            hs[i].lra(X, Om, 0.05, 1, *out[i])

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for o in out[:2]:
        assert torch.equal(o[0], out[2][0]) and torch.equal(o[1], out[2][1])
    for h in hs:
        h.close()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,ld,bs,bad", [(1, 1, 256, 0), (63, 63, 256, 40), (65, 66, 256, 65),
                                         (130, 131, 100, 0), (257, 257, 256, 257),
                                         (700, 704, 160, 401), (2304, 2304, 256, 0),
                                         (2307, 2309, 256, 2200), (2501, 2504, 128, 0)])
def test_potrf_block_edges(dev, n, ld, bs, bad, f32):
    """The blocked Cholesky at the edges of its 64-row steps, panels and
    128 x 128 update tiles, with aligned and odd leading dimensions.  Backward
    error: |A - U^T U| <= (n + 1) u |U^T| |U| elementwise, whose Frobenius norm
    is at most (n + 1) u trace(A).  The strict lower part is not touched, and a
    pivot made negative is reported as the failing minor."""
    import torch
    dt, u = (torch.float32, 2.0**-24) if f32 else (torch.float64, 2.0**-53)
    g = torch.Generator(device="cuda").manual_seed(n)
    M = torch.randn((n, n + 8), dtype=torch.float64, device="cuda", generator=g)
    A = (M @ M.t() / n + torch.eye(n, dtype=torch.float64, device="cuda")).to(dt)
    K = torch.full((n, ld), 7.0, dtype=dt, device="cuda")[:, :n]
    K.copy_(torch.tril(A) + torch.triu(torch.full_like(A, -3.0), 1))  # row j = column j
    if bad:
        K[bad - 1, bad - 1] = -1.0
        assert dev.potrf(K, bs) == bad
        return
    assert dev.potrf(K, bs) == 0
    U = torch.tril(K).double()  # U^T as rows
    err = (U @ U.t() - A.double()).norm()
    assert float(err) <= (n + 1) * u * float(torch.trace(A.double()))
    assert bool((torch.triu(K, 1) == torch.triu(torch.full_like(A, -3.0), 1)).all())


@pytest.mark.parametrize("n,d,l,labels", [(6401, 1, 1, False), (6528, 16, 16, True),
                                          (6500, 130, 17, True), (7001, 33, 40, False),
                                          (6690, 300, 5, True)])
def test_lra_error_on_symmetric_tiles(dev, n, d, l, labels):
    """||K - Q W^T||^2 and ||K||^2 from 128 x 128 tiles of one triangle against
    plain FP64 on the whole matrix.  With e = K - Q W^T off by D, the first sum is
    off by at most 2 |e| |D|; |D| is bounded elementwise by (l + 2) u |Q||W|^T for
    the product and by the exponent's error for K <= 1, on either side."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + d)
    X = torch.randn((n, d), dtype=torch.float64, device="cuda", generator=g) / d**0.5
    y = (1.0 - 2.0 * (torch.arange(n, device="cuda") % 2)).double() if labels else None
    Q, W = (torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    gamma, u = 0.7, 2.0**-53
    e2, k2 = dev.lra_error(X, gamma, Q, W, y=y)
    s = (X * X).sum(1)
    K = torch.exp(-gamma * (s[:, None] + s[None, :] - 2.0 * (X @ X.t())).clamp(min=0.0))
    if y is not None:
        K = K * y[:, None] * y[None, :]
    E = K - Q.t().contiguous() @ W
    kerr = (4.0 * gamma * float(s.max()) * (d + 4) + 4) * u
    D = 2 * ((l + 2) * u * (Q.abs().t().contiguous() @ W.abs()) + kerr * K.abs())
    ref_e, ref_k = float((E * E).sum()), float((K * K).sum())
    assert abs(e2 - ref_e) <= 2 * float(E.norm() * D.norm()) + 1e-14 * ref_e
    assert abs(k2 - ref_k) <= (4 * kerr + 1e-14) * ref_k


@pytest.mark.parametrize("n", [500, 6500])
@pytest.mark.parametrize("what,err,norm", [("inf in W", "inf", "finite"),
                                           ("overflow in W", "inf", "finite"),
                                           ("nan in Q", "nan", "finite"),
                                           ("inf in y", "inf", "inf")])
def test_lra_error_of_non_finite_input(dev, n, what, err, norm):
    """One infinite entry, or one whose square overflows, makes the sum infinite
    and not NaN, on the tiles of the whole matrix and on those of one triangle
    (6500); a NaN stays a NaN, and the other sum is not touched."""
    import math

    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    X = torch.randn((n, 24), dtype=torch.float64, device="cuda", generator=g) / 24**0.5
    Q, W = (torch.randn((20, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    y = torch.ones(n, dtype=torch.float64, device="cuda")
    _, clean = dev.lra_error(X, 0.7, Q, W, y=y)
    if what == "inf in W":
        W[3, n - 2] = -math.inf
    elif what == "overflow in W":
        W[3, n // 2] = 1e200
    elif what == "nan in Q":
        Q[0, 5] = math.nan
    else:
        y[n - 1] = math.inf
    e2, k2 = dev.lra_error(X, 0.7, Q, W, y=y)
    assert math.isnan(e2) if err == "nan" else e2 == math.inf
    assert k2 == (math.inf if norm == "inf" else clean)


@pytest.mark.slow
def test_rbf_project_f64_wide_with_very_many_rows(dev):
    """More than 65535 row tiles of 64 rows, a grid's customary limit in y, at
    d > 256, which few column points allow.  Rows at the ends and around the
    first block's end against plain FP64; an entry's distance product is off by
    at most (d + 4) u 4 s, s the largest squared norm, on either side, which
    the exponential turns into gamma times that, relative."""
    import torch
    m, n, d, l, gamma, u = 64 * 65535 + 100, 3, 257, 2, 0.7, 2.0**-53
    g = torch.Generator(device="cuda").manual_seed(m)
    X = torch.rand((m, d), dtype=torch.float64, device="cuda", generator=g).div_(d**0.5)
    O = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    Y = torch.full((l, m), 7.0, dtype=torch.float64, device="cuda")
    dev.rbf_project_f64(X, X[:n], O, gamma, Y)
    b = 64 * 65535
    rows = torch.tensor([0, 1, 63, 64, b // 2, b - 1, b, b + 1, m - 2, m - 1], device="cuda")
    A, B = X[rows], X[:n]
    K = torch.exp(-gamma * (A[:, None, :] - B[None, :, :]).pow(2).sum(2))
    ref = K @ O.t().contiguous()
    tol = 2 * (gamma * 4 * (d + 4) + n + 4) * u * float(O.abs().sum(1).max())
    assert float((Y[:, rows].t() - ref).abs().max()) <= tol  # s <= 1
    assert bool((Y != 7.0).all())


@pytest.mark.parametrize("m,n,d,l,beta", [(130, 300000, 257, 20, 0.5), (700, 300000, 260, 3, 0.0),
                                          (1, 70000, 300, 17, 1.0), (12000, 11500, 257, 290, 0.0),
                                          (150000, 20, 257, 1000, -0.5)])
def test_rbf_project_f64_wide_row_blocks(dev, m, n, d, l, beta):
    """d > 256 with few and many rows against few and many columns: several row
    blocks, many parts of the j range, partial products in several parts of the
    rows.  Tolerance per element: n products and beta Y in any order, and K from
    distances that are off by at most (d + 4) u 4 s, s <= 1 the largest squared
    norm, on either side."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n)
    Xi, Xj = (torch.rand((c, d), dtype=torch.float64, device="cuda", generator=g).div_(d**0.5)
              for c in (m, n))
    yi, yj = (1.0 - 2.0 * (torch.arange(c, device="cuda") % 3 == 0).double() for c in (m, n))
    O = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    Y = torch.randn((l, m), dtype=torch.float64, device="cuda", generator=g)
    gamma, u = 0.7, 2.0**-53
    Y0 = Y.clone()
    dev.rbf_project_f64(Xi, Xj, O, gamma, Y, yi=yi, yj=yj, beta=beta)
    Ot = O.t().contiguous()
    step = max(1, (1 << 27) // n)
    for i in range(0, m, step):
        A = Xi[i:i + step]
        K = torch.exp(-gamma * ((A * A).sum(1)[:, None] + (Xj * Xj).sum(1)[None, :]
                                - 2.0 * (A @ Xj.t())).clamp(min=0.0))
        K = K * yi[i:i + step, None] * yj[None, :]
        ref = K @ Ot + beta * Y0[:, i:i + step].t()
        size = K.abs() @ Ot.abs() + abs(beta) * Y0[:, i:i + step].t().abs()
        tol = 2 * (gamma * 4 * (d + 4) + n + 6) * u * size
        assert bool(((Y[:, i:i + step].t() - ref).abs() <= tol).all())


def test_rbf_project_f64_wide_fills_the_gpu_with_few_rows():
    """The pass over a wide K (300 x 500000) does the work of the pass over its
    transpose; with the j range split enough it takes about as long.  Partial
    products (4.8 GB if they were held for all 600000 x 1000) and blocks of K stay
    within 1 GiB each, and an eighth of headroom."""
    import torch
    h = dh.Handle(0)

    def best(m, n, l):
        Xi, Xj = (torch.rand((c, 300), dtype=torch.float64, device="cuda") for c in (m, n))
        O = torch.rand((l, n), dtype=torch.float64, device="cuda")
        Y = torch.zeros((l, m), dtype=torch.float64, device="cuda")
        ts = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda.synchronize()
            a.record()
            h.rbf_project_f64(Xi, Xj, O, 0.01, Y, beta=0.5)
            h.synchronize()
            b.record()
            torch.cuda.synchronize()
            ts.append(a.elapsed_time(b))
        return min(ts)

    assert best(300, 500000, 74) < 2.0 * best(500000, 300, 74)
    best(600000, 20, 1000)
    assert h.workspace_bytes() < 3 * 2**30
    h.close()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,bs,bad", [(600, 600, 0), (1100, 1024, 0), (1100, 5000, 1090),
                                      (2501, 2501, 0), (2501, 100, 0), (2503, 100, 2301),
                                      (2501, 40, 0)])
def test_potrf_wide_and_odd_panels(dev, n, bs, bad, f32):
    """Panels wider than the kernels take at once, and panel widths that are not
    whole stages of the trailing update's copies at sizes that otherwise use it.
    Backward error as in test_potrf_block_edges."""
    import torch
    dt, u = (torch.float32, 2.0**-24) if f32 else (torch.float64, 2.0**-53)
    g = torch.Generator(device="cuda").manual_seed(n)
    M = torch.randn((n, n + 8), dtype=torch.float64, device="cuda", generator=g)
    A = (M @ M.t() / n + torch.eye(n, dtype=torch.float64, device="cuda")).to(dt)
    K = A.clone()
    if bad:
        K[bad - 1, bad - 1] = -1.0
        assert dev.potrf(K, bs) == bad
        return
    assert dev.potrf(K, bs) == 0
    U = torch.tril(K).double()
    err = (U @ U.t() - A.double()).norm()
    assert float(err) <= (n + 1) * u * float(torch.trace(A.double()))


def test_potrf_with_one_panel_is_as_fast_as_with_several(dev):
    import time

    import torch
    n = 4096
    g = torch.Generator(device="cuda").manual_seed(1)
    M = torch.randn((n, 64), dtype=torch.float64, device="cuda", generator=g)
    A = M @ M.t() + n * torch.eye(n, dtype=torch.float64, device="cuda")
    K = A.clone()

    def best(bs):
        ts = []
        for _ in range(6):
            K.copy_(A)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            assert dev.potrf(K, bs) == 0
            ts.append(time.perf_counter() - t0)
        return min(ts)

    assert best(n) < 1.5 * best(256)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,at", [(50, 20), (50, 48), (50, 49), (64, 15), (200, 0), (200, 63),
                                  (700, 150), (700, 600), (700, 699)])
def test_potrf_with_an_infinite_diagonal_entry(dev, n, at, f32):
    """An infinite pivot is positive: its row of U is zero beside the diagonal (inf /
    inf there) and the other rows are the Cholesky factor of the rest."""
    import torch
    dt, u = (torch.float32, 2.0**-24) if f32 else (torch.float64, 2.0**-53)
    g = torch.Generator(device="cuda").manual_seed(n)
    M = torch.randn((n, n + 8), dtype=torch.float64, device="cuda", generator=g)
    A = (M @ M.t() / n + torch.eye(n, dtype=torch.float64, device="cuda")).to(dt)
    K = A.clone()
    K[at, at] = float("inf")
    assert dev.potrf(K) == 0
    L = torch.tril(K).double()  # U^T
    assert bool(torch.isnan(L[at, at])) and bool((L[at + 1:, at] == 0).all())
    keep = [i for i in range(n) if i != at]
    L, B = L[keep][:, keep], A.double()[keep][:, keep]
    assert float((L @ L.t() - B).norm()) <= (n + 1) * u * float(torch.trace(B))


def test_rbf_project_f64_wide_with_negative_gamma(dev):
    """d > 256 with far but close-lying points: K = exp(+|xi - xj|^2) is finite, and
    the padding of the columns (17 -> 32) must not bring an infinity in.
    Tolerance: distances off by (d + 4) u 4 s on either side, s the largest norm."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    d, n, l, u = 300, 17, 5, 2.0**-53
    X = 1.5 + 0.01 * torch.randn((n, d), dtype=torch.float64, device="cuda", generator=g)
    O = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    Y, Q, W = (torch.empty_like(O) for _ in range(3))
    dev.rbf_project_f64(X, X, O, -1.0, Y)
    K = torch.exp((X[:, None, :] - X[None, :, :]).pow(2).sum(2))
    s = float((X * X).sum(1).max())  # about 700
    tol = 2 * (4 * (d + 4) * s + n + 4) * u * float(K.max() * O.abs().sum(1).max())
    assert float((Y.t() - K @ O.t().contiguous()).abs().max()) <= tol
    assert dev.lra(X, O, -1.0, 0, Q, W) == 0 and bool(torch.isfinite(W).all())


def test_rbf_project_f64_wide_fills_the_gpu_with_few_points():
    """2000 x 2000: 32 row tiles, so the j range goes in eight parts, whose partial
    products (beside K and the packed panel) are held.  n products in any order and
    distances off by (d + 4) u 4 s, s <= 1, on either side."""
    import torch
    h = dh.Handle(0)
    n, d, l, gamma, u = 2000, 300, 272, 0.7, 2.0**-53
    g = torch.Generator(device="cuda").manual_seed(4)
    X = torch.rand((n, d), dtype=torch.float64, device="cuda", generator=g).div_(d**0.5)
    O = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    Y = torch.empty_like(O)
    h.rbf_project_f64(X, X, O, gamma, Y)
    s = (X * X).sum(1)
    K = torch.exp(-gamma * (s[:, None] + s[None, :] - 2.0 * (X @ X.t())).clamp(min=0.0))
    Ot = O.t().contiguous()
    tol = 2 * (gamma * 4 * (d + 4) + n + 4) * u * (K @ Ot.abs())
    assert bool(((Y.t() - K @ Ot).abs() <= tol).all())
    assert h.workspace_bytes() >= 8 * (n * n + n * l + 8 * n * l)
    h.close()
