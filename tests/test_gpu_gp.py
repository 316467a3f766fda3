"""GPU GP log-density caller: partial Cholesky, preconditioner, CG, logpdf.

The reference's own checks (tests/test_low_rank/test_cholesky.py,
tests/test_low_rank/test_preconditioner.py) run through the drop-in API with
``operators.dense_matvec`` as the element function; the kernels are compared
with the oracle's FP32 restatement (oracle/lowrank.py) and with FP64 dense
linear algebra; the log-density with the dense reference of
tutorials/8_gaussian_logpdf.py:55-66 (``scipy.stats``).
"""

import numpy as np
import pytest
import scipy.stats
import torch

from matfree_amd import gp, linalg, low_rank, operators, problems, prng
from oracle import lowrank as olr

pytestmark = pytest.mark.gpu


def sym_from_eigs(eigvals, seed):
    n = len(eigvals)
    Q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))
    return ((Q * np.asarray(eigvals)) @ Q.T).astype(np.float32)


def rbf_dense(X, ls, noise):
    X = np.asarray(X, np.float64)
    d2 = np.sum((X[:, None] - X[None]) ** 2, -1)
    return np.exp(-d2 / (2 * ls**2)) + noise * np.eye(len(X))


@pytest.mark.parametrize("pivot", [False, True])
def test_full_rank_cholesky_reconstructs_matrix(cuda, pivot):
    # test_cholesky.py:16-28 (n = 5, eigenvalues 1 + U(0, 1)); FP32 kernels,
    # tolerance a few FP32 ulps
    n = 5
    cov = sym_from_eigs(1.0 + np.random.default_rng(2).uniform(size=n), 2)
    f = low_rank.cholesky_partial_pivot if pivot else low_rank.cholesky_partial
    L, _ = f(operators.dense_matvec, nrows=n, rank=n)(torch.as_tensor(cov, device=cuda))
    L = L.cpu().numpy().astype(np.float64)
    tol = 8 * np.finfo(np.float32).eps
    assert L.shape == (n, n)
    assert np.allclose(L @ L.T, cov, atol=tol, rtol=tol)


def test_nopivot_matches_cholesky_and_pivot_does_not(cuda):
    # test_cholesky.py:45-62
    n = 10
    cov = sym_from_eigs(0.01 + np.random.default_rng(2).uniform(size=n), 2)
    A = torch.as_tensor(cov, device=cuda)
    reference = np.linalg.cholesky(cov.astype(np.float64))
    Lp, info = low_rank.cholesky_partial_pivot(operators.dense_matvec, nrows=n, rank=n)(A)
    assert bool(info["success"])
    assert not np.allclose(Lp.cpu().numpy(), reference)
    L, _ = low_rank.cholesky_partial(operators.dense_matvec, nrows=n, rank=n)(A)
    assert np.allclose(L.cpu().numpy(), reference, atol=1e-5)


def test_pivoting_improves_the_estimate(cuda):
    # test_cholesky.py:65-81
    n, rank = 10, 5
    cov = sym_from_eigs(0.1 + np.random.default_rng(1).uniform(size=n), 1)
    A = torch.as_tensor(cov, device=cuda)
    nop, _ = low_rank.cholesky_partial(operators.dense_matvec, nrows=n, rank=rank)(A)
    piv, _ = low_rank.cholesky_partial_pivot(operators.dense_matvec, nrows=n, rank=rank)(A)
    nop, piv = nop.cpu().numpy(), piv.cpu().numpy()
    assert np.linalg.norm(cov - piv @ piv.T) < np.linalg.norm(cov - nop @ nop.T)


@pytest.mark.parametrize("n,rank", [(300, 40), (1000, 96)])
def test_pivoted_cholesky_matches_oracle(cuda, n, rank):
    # a dense SPD matrix with well separated residual diagonals: the pivot
    # order is identical and L agrees to FP32 rounding of the sums
    A = problems.dense_spd(n, seed=3, shift=0.1)
    L, success, perm = low_rank.cholesky_partial_pivot(operators.dense_matvec, nrows=n,
                                                       rank=rank).factor(
        torch.as_tensor(A, device=cuda))
    Lo, info, Po = olr.cholesky_partial_pivot(A, rank, np.float32)
    np.testing.assert_array_equal(perm.cpu().numpy(), Po)
    assert bool(success) == info["success"]
    scale = np.abs(Lo).max()
    assert np.abs(L.cpu().numpy() - Lo).max() <= 2e-5 * scale


def test_rbf_pivoted_cholesky_approximates_kernel(cuda):
    # the element function of the RBF operator (noise 0): a rank-r pivoted
    # factor of a smooth kernel; against the oracle on the same matrix (first
    # pivot: all diagonals equal, argmax takes row 0) and by its error
    n, rank = 2048, 64
    X = problems.rbf_points(n, seed=1)
    op = operators.RBF(X)
    L, success, perm = low_rank.cholesky_partial_pivot(op, nrows=n, rank=rank).factor(0.5, 0.0)
    K = rbf_dense(X, 0.5, 0.0)
    Lo, info, Po = olr.cholesky_partial_pivot(K.astype(np.float32), rank, np.float32)
    assert int(perm[0]) == 0 and Po[0] == 0
    assert bool(success) and info["success"]
    Lg = L.cpu().numpy().astype(np.float64)
    err_gpu = np.linalg.norm(K - Lg @ Lg.T)
    err_orc = np.linalg.norm(K - Lo.astype(np.float64) @ Lo.T.astype(np.float64))
    assert err_gpu <= 1.05 * err_orc + 1e-6
    assert err_gpu < 1e-1 * np.linalg.norm(K)


def test_preconditioner_solves_correctly(cuda):
    # test_preconditioner.py:7-40 (rtol 1e-2), and against the FP64 solve
    n = 10
    cov = sym_from_eigs(1.5 ** np.arange(-n // 2, n // 2, step=1.0), 1)
    A = torch.as_tensor(cov, device=cuda)
    cholesky = low_rank.cholesky_partial(operators.dense_matvec, nrows=n, rank=n)
    Lf, _ = cholesky(A)
    assert np.allclose(Lf.cpu().numpy() @ Lf.cpu().numpy().T, cov, atol=1e-5)
    b = np.arange(1.0, 1 + n)
    b /= np.linalg.norm(b)
    expected = np.linalg.solve(cov.astype(np.float64) + 0.1 * np.eye(n), b)
    received, _ = low_rank.preconditioner(cholesky)(torch.as_tensor(b, device=cuda), 0.1, A)
    assert np.allclose(received.cpu().numpy(), expected, rtol=1e-2)
    assert np.allclose(received.cpu().numpy(), expected, rtol=1e-4, atol=1e-5)


def test_woodbury_matches_oracle_low_rank(cuda):
    n, rank, P, s = 3000, 48, 3, 0.05
    rng = np.random.default_rng(5)
    L = (rng.standard_normal((n, rank)) / np.sqrt(n)).astype(np.float32)
    V = rng.standard_normal((P, n)).astype(np.float32)
    out = low_rank.lowrank_solve(torch.as_tensor(L, device=cuda), torch.as_tensor(V, device=cuda),
                                 s).cpu().numpy()
    L64 = L.astype(np.float64)
    exact = np.linalg.solve(s * np.eye(n) + L64 @ L64.T, V.astype(np.float64).T).T
    assert np.abs(out - exact).max() <= 1e-4 * np.abs(exact).max()
    orc = np.stack([olr.preconditioner_solve(L, v, s) for v in V])
    assert np.abs(out - orc).max() <= 1e-4 * np.abs(orc).max()


def test_cg_matches_oracle_and_dense_solve(cuda):
    n, P = 1000, 4
    A = problems.dense_spd(n, seed=2, shift=0.5)
    B = np.random.default_rng(3).standard_normal((P, n)).astype(np.float32)
    X, iters = linalg.cg_batched(operators.dense_matvec, torch.as_tensor(B, device=cuda),
                                 (torch.as_tensor(A, device=cuda),), tol=1e-6)
    Xo, ko = olr.cg(lambda V: V @ A.T, B, tol=1e-6)
    exact = np.linalg.solve(A.astype(np.float64), B.astype(np.float64).T).T
    X = X.cpu().numpy()
    assert np.all(np.abs(iters.cpu().numpy() - ko) <= 1)
    assert np.linalg.norm(X - exact) <= 1e-4 * np.linalg.norm(exact)
    assert np.linalg.norm(X - Xo) <= 1e-4 * np.linalg.norm(Xo)
    # the stopping rule: |b - A x| <= tol |b| up to FP32 rounding of the recurrence
    R = B - X @ A.T
    assert np.all(np.linalg.norm(R, axis=1) <= 5e-6 * np.linalg.norm(B, axis=1))


def test_cg_single_vector_api_and_maxiter(cuda):
    n = 500
    A = torch.as_tensor(problems.dense_spd(n, seed=4, shift=0.2), device=cuda)
    b = torch.ones(n, device=cuda)
    x, info = linalg.cg(operators.dense_matvec, b, A)
    assert info is None and x.shape == (n,)
    _, it = linalg.cg_batched(operators.dense_matvec, b, (A,), tol=1e-12, maxiter=3)
    assert int(it) == 3
    _, it0 = linalg.cg_batched(operators.dense_matvec, torch.zeros(n, device=cuda), (A,))
    assert int(it0) == 0


def test_preconditioned_cg_on_rbf(cuda):
    # K + s I with the pivoted partial Cholesky of K as preconditioner
    # (low_rank.py:7-53): same solution, far fewer iterations
    n, rank, ls, s = 4096, 128, 0.3, 1e-2
    X = problems.rbf_points(n, seed=2)
    op = operators.RBF(X)
    y = torch.as_tensor(np.random.default_rng(0).standard_normal(n).astype(np.float32),
                        device=cuda)
    prec = low_rank.preconditioner(low_rank.cholesky_partial_pivot(op, nrows=n, rank=rank))
    M = prec.bind(s, ls, 0.0)
    x0, k0 = linalg.cg_batched(op, y, (ls, s), tol=1e-5)
    x1, k1 = linalg.cg_batched(op, y, (ls, s), tol=1e-5, M=M)
    A = rbf_dense(X, ls, s)
    exact = np.linalg.solve(A, y.cpu().numpy().astype(np.float64))
    for x in (x0, x1):
        assert np.linalg.norm(x.cpu().numpy() - exact) <= 2e-3 * np.linalg.norm(exact)
    assert int(k1) < int(k0) // 3, (int(k0), int(k1))


def test_quadform_vjp_matches_dense(cuda):
    n, P = 300, 3
    X = problems.rbf_points(n, seed=6)
    V = np.random.default_rng(1).standard_normal((P, n)).astype(np.float32)
    ls = 0.4
    d = linalg.quadform_vjp(operators.RBF(X), torch.as_tensor(V, device=cuda), (ls, 0.1))
    Xd = np.asarray(X, np.float64)
    d2 = np.sum((Xd[:, None] - Xd[None]) ** 2, -1)
    dK = np.exp(-d2 / (2 * ls**2)) * d2 / ls**3
    V64 = V.astype(np.float64)
    assert np.isclose(float(d[0]), np.einsum("pi,ij,pj->", V64, dK, V64), rtol=1e-4)
    assert np.isclose(float(d[1]), np.sum(V64 * V64), rtol=1e-5)
    A = problems.dense_spd(n, seed=1, shift=1.0)
    (D,) = linalg.quadform_vjp(operators.dense_matvec, torch.as_tensor(V, device=cuda),
                               (torch.as_tensor(A, device=cuda),))
    assert np.allclose(D.cpu().numpy(), V64.T @ V64, rtol=1e-4, atol=1e-4)


# The RBF parameter contraction <S, dK/dl>, <S, I> with S = sum_p x_p x_p^T,
# against its FP64 closed form: the FP32 matrix-core form for FP32
# operators, for BF16 operators the derivative kernel applied to the vectors
# as a block matvec in split BF16 (hi*hi + hi*lo + lo*hi, ~2^-16 per
# product) and dotted with them; point dimensions 1-4 (4 in FP32 only),
# unaligned n, one row block (n = 77), split-K slices, several launches of
# 1024 columns with a partial last column block (P = 1100).
@pytest.mark.parametrize("precision,dim,n,P", [
    ("fp32", 1, 300, 3), ("fp32", 4, 301, 5), ("fp32", 4, 1000, 40),
    ("bf16x2", 1, 300, 3), ("bf16x2", 2, 301, 5), ("bf16x2", 3, 1000, 40),
    ("bf16", 3, 517, 17), ("bf16x2", 3, 77, 9), ("bf16x3", 2, 600, 1100)])
def test_quadform_vjp_contraction_forms(cuda, precision, dim, n, P):
    X = problems.rbf_points(n, seed=6, dim=dim)
    V = np.random.default_rng(dim).standard_normal((P, n)).astype(np.float32)
    ls = 0.4
    d = linalg.quadform_vjp(operators.RBF(X, precision=precision),
                            torch.as_tensor(V, device=cuda), (ls, 0.1))
    Xd = np.asarray(X, np.float64)
    d2 = np.sum((Xd[:, None] - Xd[None]) ** 2, -1)
    dK = np.exp(-d2 / (2 * ls**2)) * d2 / ls**3
    V64 = V.astype(np.float64)
    want = np.einsum("pi,ij,pj->", V64, dK, V64)
    # the sum cancels (E[want] = tr dK = 0 for these zero-mean vectors), so
    # besides 1e-4 relative the bound allows 8 x 2^-16 (the representation
    # error of a split-BF16 or FP32 product) of the terms' root sum of squares
    rss = np.sqrt(np.einsum("pi,ij,pj->", V64**2, dK**2, V64**2))
    err = abs(float(d[0]) - want)
    print(f"{precision} dim={dim} n={n} P={P}: rel {err / abs(want):.2e}, "
          f"{err / (2.0**-16 * rss):.2f} x 2^-16 rss", flush=True)
    assert err <= max(1e-4 * abs(want), 8 * 2.0**-16 * rss)
    assert np.isclose(float(d[1]), np.sum(V64 * V64), rtol=1e-4)


def test_gaussian_logpdf_tutorial(cuda):
    # tutorials/8_gaussian_logpdf.py: n = 30 points on [0, 1], log_ell = 0,
    # log_noise = -2, num_matvecs = 6, num_samples = 500; the value against
    # scipy's dense log-density (Monte-Carlo error of the SLQ term: 2%), the
    # gradient against the dense closed form
    #   d logpdf / d theta = (alpha^T dA alpha - tr(A^{-1} dA)) / 2
    n = 30
    xs = np.linspace(0.0, 1.0, n).astype(np.float32)
    op = operators.RBF(xs[:, None])
    logpdf = gp.create_logpdf(op, np.zeros(n, np.float32))
    y = np.random.default_rng(1).standard_normal(n).astype(np.float32)
    log_ell = torch.tensor(0.0, dtype=torch.float64, device=cuda, requires_grad=True)
    log_noise = torch.tensor(-2.0, dtype=torch.float64, device=cuda, requires_grad=True)
    val = logpdf(torch.as_tensor(y, device=cuda), prng.PRNGKey(2), torch.exp(log_ell),
                 torch.exp(log_noise))
    val.backward()
    ell, noise = 1.0, float(np.exp(-2.0))
    A = rbf_dense(xs[:, None], ell, noise)
    ref = scipy.stats.multivariate_normal.logpdf(y.astype(np.float64), mean=np.zeros(n), cov=A)
    v = float(val.detach())
    assert abs(v - ref) <= 2e-2 * abs(ref), (v, ref)
    d2 = (xs[:, None].astype(np.float64) - xs[None].astype(np.float64)) ** 2
    dA_dlogell = np.exp(-d2 / (2 * ell**2)) * d2 / ell**2  # dK/dl * l
    dA_dlognoise = noise * np.eye(n)
    alpha = np.linalg.solve(A, y.astype(np.float64))
    Ainv = np.linalg.inv(A)
    for dA, g in ((dA_dlogell, log_ell.grad), (dA_dlognoise, log_noise.grad)):
        exact = 0.5 * (alpha @ dA @ alpha - np.trace(Ainv @ dA))
        assert abs(float(g) - exact) <= 0.1 * abs(exact) + 0.05, (float(g), exact)


def test_quadform_gradient_is_exact(cuda):
    # the CG part alone: d/dtheta y^T A^{-1} y = -alpha^T dA alpha
    n = 500
    X = problems.rbf_points(n, seed=3)
    op = operators.RBF(X)
    y = torch.as_tensor(np.random.default_rng(2).standard_normal(n).astype(np.float32),
                        device=cuda)
    ls = torch.tensor(0.3, dtype=torch.float64, device=cuda, requires_grad=True)
    s2 = torch.tensor(0.1, dtype=torch.float64, device=cuda, requires_grad=True)
    q = gp.quadform_inverse(op, y, ls, s2, tol=1e-7)
    q.backward()
    A = rbf_dense(X, 0.3, 0.1)
    yd = y.cpu().numpy().astype(np.float64)
    alpha = np.linalg.solve(A, yd)
    assert np.isclose(float(q), yd @ alpha, rtol=1e-4)
    Xd = np.asarray(X, np.float64)
    d2 = np.sum((Xd[:, None] - Xd[None]) ** 2, -1)
    dK = np.exp(-d2 / (2 * 0.3**2)) * d2 / 0.3**3
    assert np.isclose(float(ls.grad), -alpha @ dK @ alpha, rtol=1e-3)
    assert np.isclose(float(s2.grad), -alpha @ alpha, rtol=1e-3)


def test_gaussian_logpdf_with_only_the_lengthscale_learned(cuda):
    # a requires-grad lengthscale and a plain float noise: the gradient of the
    # log-density in the lengthscale alone, against the dense closed form
    n = 40
    xs = np.linspace(0.0, 1.0, n).astype(np.float32)
    op = operators.RBF(xs[:, None])
    logpdf = gp.create_logpdf(op, np.zeros(n, np.float32))
    y = np.random.default_rng(3).standard_normal(n).astype(np.float32)
    ell = torch.tensor(0.8, dtype=torch.float64, device=cuda, requires_grad=True)
    noise = 0.1
    logpdf(torch.as_tensor(y, device=cuda), prng.PRNGKey(4), ell, noise).backward()
    A = rbf_dense(xs[:, None], 0.8, noise)
    d2 = (xs[:, None].astype(np.float64) - xs[None].astype(np.float64)) ** 2
    dA = np.exp(-d2 / (2 * 0.8**2)) * d2 / 0.8**3
    alpha = np.linalg.solve(A, y.astype(np.float64))
    exact = 0.5 * (alpha @ dA @ alpha - np.trace(np.linalg.solve(A, dA)))
    assert abs(float(ell.grad) - exact) <= 0.1 * abs(exact) + 0.05, (float(ell.grad), exact)


@pytest.mark.parametrize("n", [5, 700, 1024, 2047, 2048, 2049, 4096, 4097, 6145, 8192, 8193])
def test_cg_column_kernels(cuda, n):
    # an iteration of a column in one workgroup (n <= 8192), with the split-K sum (n <= 4096)
    # and without, at the chunk edges; a zero right-hand side beside the others stays at zero.
    # A stored matrix with eigenvalues in [1, 5]: the recurrence stops at 1e-6 |b|, and its
    # residual and the true one part by sum_t |alpha_t A d_t| times the products' 2e-6, at most
    # 2e-6 |A| 2 |x| = 2e-5 |b|.  Together with the sums' own rounding 3e-5.
    gen = torch.Generator(device="cuda").manual_seed(n)
    G = torch.randn((n, n), generator=gen, device="cuda")
    A = G @ G.T / n
    A = 0.5 * (A + A.T)
    A.diagonal().add_(1.0)
    B = torch.randn((3, n), generator=gen, device="cuda")
    B[1] = 0.0
    x, iters = linalg.cg_batched(operators.dense_matvec, B, (A,), tol=1e-6)
    residual = (B.double() - x.double() @ A.double()).norm(dim=1)
    assert float(x[1].abs().max()) == 0.0 and int(iters[1]) == 0
    assert int(iters[0]) > 0 and int(iters[2]) > 0
    for p in (0, 2):
        assert float(residual[p] / B[p].double().norm()) < 3e-5
