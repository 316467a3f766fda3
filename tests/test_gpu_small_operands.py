"""FP32 block products of operands near the end of the normal range (run on an
MI355X): every form (stored matrix and RBF, up to 32 vectors, 33-64, more)
keeps FP32's significant bits there.

Tolerances: 2e-6 normwise for products of full operands (the bound of the FP32
matvec tests).  A column of the RBF matrix has entries down to 2^-126, whose
base-2 exponents up to 126 are FP32 sums of three squares of differences: each
of the eight operations rounds by 2^-24, so an entry by at most 126 ln 2 8 2^-24
= 4e-5; 1e-4.
"""

import numpy as np
import pytest
import torch

from matfree_amd import operators, problems

pytestmark = pytest.mark.gpu


def rel(got, ref):
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("n,P", [(300, 5), (300, 32), (300, 33), (300, 128), (4127, 32),
                                 (4127, 40), (9001, 28)])
@pytest.mark.parametrize("matrix,vectors", [(1.0, 1e-35), (1e-35, 1.0), (1e-36, 1e10),
                                            (1e12, 2e-38)])
def test_stored_matrix(cuda, n, P, matrix, vectors):
    rng = np.random.default_rng(n + P)
    A = (matrix * rng.uniform(0.5, 1.0, (n, n))).astype(np.float32)
    V = (vectors * rng.uniform(0.6, 1.0, (P, n))).astype(np.float32)
    W = operators.dense_matvec(torch.as_tensor(V, device=cuda), torch.as_tensor(A, device=cuda))
    scale = 1.0 / (matrix * vectors)
    ref = (V.astype(np.float64) / vectors) @ (A.T.astype(np.float64) / matrix)
    assert rel(W.double().cpu().numpy() * scale, ref) < 2e-6


@pytest.mark.parametrize("n,P", [(300, 5), (300, 32), (300, 33), (300, 100), (4127, 32)])
def test_rbf_small_vectors(cuda, n, P):
    X = problems.rbf_points(n, seed=n)
    V = (1e-35 * np.random.default_rng(P).uniform(0.6, 1.0, (P, n))).astype(np.float32)
    W = operators.RBF(torch.as_tensor(X, device=cuda))(torch.as_tensor(V, device=cuda), 0.5, 1e-2)
    ref = (V.astype(np.float64) * 1e35) @ problems.rbf_dense64(X, 0.5, 1e-2)
    assert rel(W.double().cpu().numpy() * 1e35, ref) < 2e-6


@pytest.mark.parametrize("n,P", [(300, 32), (300, 33), (300, 100), (4127, 32)])
def test_rbf_columns_of_small_entries(cuda, n, P):
    # unit vectors: entry by entry, one point at the origin and the others 13 lengthscales away
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
    assert np.count_nonzero(normal[:, P:] & (ref[:, P:] < 2.0**-118)) > 100
    assert np.max(np.abs(W[normal] / ref[normal] - 1.0)) < 1e-4
