"""FP32 block products of more than 32 vectors on both sides of the line
between the wave form in blocks of 32 vectors and the workgroup form (run on an
MI355X), against an FP64 product: partial tiles, last blocks of one vector and
of 32, slices, infinities and NaN, small and large operands.

Tolerances as for the other FP32 products: 2e-6 normwise (products and sums of
random sign round by at most 2^-24 of a partial sum); for unit vectors on RBF
entries down to 2^-126, 1e-4 entry by entry (FP32 exponents up to 126)."""

import numpy as np
import pytest
import torch

from matfree_amd import operators, problems

pytestmark = pytest.mark.gpu


def rel(got, ref):
    return float(np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref))


# up to n^2 ceil(P / 32) = 2^25 and n < 4096 the wave form, else the workgroup form
@pytest.mark.parametrize("n,P", [
    (2048, 256), (2048, 257), (2049, 256), (1023, 1024), (3340, 96), (3347, 96), (4095, 33),
    (4095, 64), (4096, 33), (4096, 64), (4097, 65), (4127, 40), (4128, 130), (4129, 64),
    (5003, 100), (5984, 33)])
def test_stored_matrix_against_fp64(cuda, n, P):
    gen = torch.Generator(device="cuda").manual_seed(n + P)
    A = torch.randn((n, n), generator=gen, device=cuda)
    A = A + A.T
    V = torch.randn((P, n), generator=gen, device=cuda)
    ref = (V.double() @ A.double()).cpu().numpy()
    assert rel(operators.dense_matvec(V, A), ref) < 2e-6


@pytest.mark.parametrize("dim", [1, 2, 3, 4])
@pytest.mark.parametrize("n,P", [(2048, 256), (2049, 256), (3347, 96), (4095, 33), (4096, 64),
                                 (4097, 65), (4129, 130)])
def test_rbf_against_fp64(cuda, n, P, dim):
    X = problems.rbf_points(n, seed=n, dim=dim)
    V = np.random.default_rng(P).standard_normal((P, n)).astype(np.float32)
    K = torch.as_tensor(problems.rbf_dense64(X, 0.5, 1e-2), device=cuda)
    ref = (torch.as_tensor(V, device=cuda).double() @ K).cpu().numpy()
    op = operators.RBF(torch.as_tensor(X, device=cuda))
    assert rel(op(torch.as_tensor(V, device=cuda), 0.5, 1e-2), ref) < 2e-6


@pytest.mark.parametrize("n,P", [(301, 64), (301, 97), (4127, 64), (4127, 97)])
def test_non_finite_and_huge_values(cuda, n, P):
    rng = np.random.default_rng(5)
    A = rng.uniform(0.5, 1.0, (n, n)).astype(np.float32)
    A = 0.5 * (A + A.T)
    V = rng.uniform(0.5, 1.0, (P, n)).astype(np.float32)
    V[0, 7] = np.inf
    V[1, 8] = -np.inf
    V[2, 9] = np.nan
    V[3, 10], V[3, n - 1] = np.inf, -np.inf
    V[4] = 0.0
    V[4, 12] = np.float32(3.4e38)  # rounds to infinity in BF16
    V[P - 1, n - 1] = np.inf
    V[P - 2] *= np.float32(1e33)  # sums of the scaled operands overflow
    W = operators.dense_matvec(torch.as_tensor(V, device=cuda), torch.as_tensor(A, device=cuda))
    W = W.cpu().numpy().astype(np.float64)
    assert np.all(W[0] == np.inf) and np.all(W[1] == -np.inf) and np.all(W[P - 1] == np.inf)
    assert np.all(np.isnan(W[2])) and np.all(np.isnan(W[3]))
    ref = V[4:P - 1].astype(np.float64) @ A.astype(np.float64)
    np.testing.assert_allclose(W[4:P - 1], ref, rtol=2e-6)


@pytest.mark.parametrize("n,P", [(300, 28), (300, 40), (4127, 28), (4127, 40), (4127, 100)])
@pytest.mark.parametrize("matrix,vectors", [(1e18, 1e14), (1e-3, 1e36), (1e36, 1e-3)])
def test_large_operands(cuda, n, P, matrix, vectors):
    rng = np.random.default_rng(n + P)
    A = (matrix * rng.uniform(0.5, 1.0, (n, n))).astype(np.float32)
    V = (vectors * rng.uniform(0.6, 1.0, (P, n))).astype(np.float32)
    W = operators.dense_matvec(torch.as_tensor(V, device=cuda), torch.as_tensor(A, device=cuda))
    ref = (V.astype(np.float64) / vectors) @ (A.T.astype(np.float64) / matrix)
    assert rel(W.double() / (matrix * vectors), ref) < 2e-6


@pytest.mark.parametrize("P", [40, 100])
def test_rbf_columns_of_small_entries_workgroup_form(cuda, P):
    n = 4127
    rng = np.random.default_rng(n)
    X = rng.uniform(-0.1, 0.1, (n, 3)).astype(np.float32)
    X[P:] += np.float32(13.0 / np.sqrt(3.0))
    V = np.zeros((P, n), np.float32)
    V[np.arange(P), np.arange(P)] = 1.0
    W = operators.RBF(torch.as_tensor(X, device=cuda))(torch.as_tensor(V, device=cuda), 1.0, 0.0)
    W = W.double().cpu().numpy()
    X64 = X.astype(np.float64)
    ref = np.exp(-0.5 * ((X64[:P, None] - X64[None]) ** 2).sum(-1))
    normal = ref > 2.0**-125
    assert np.max(np.abs(W[normal] / ref[normal] - 1.0)) < 1e-4
