"""The Gram-Schmidt passes and the planes of the reverse pass at the sizes where
their rules change (run on an MI355X).  Rows longer than a chunk (2048), so that
no step runs in one workgroup:

* columns a block of the dots (8, 16, 32 or 64, as many as leave 512 blocks),
  aligned rows and rows of odd length;
* the projection with a batch of columns ahead (below 640 blocks) and without;
* passes that alternate in direction (from 1024 blocks on);
* the projection's output as one and two BF16 planes and as the FP32 products'
  three (n % 4 == 0, more than four probes).

Tolerances: a matrix with spectrum in [1, 2], FP32 products good to 1e-6, the
recurrence at these depths grows an error by less than 100 (1e-4 normwise), two
classical passes keep the basis orthonormal to a few roundings of sums over n
(1e-5).  Reverse pass at depth 6 of operators of condition number below ten: 1e-4
for FP32 (products to 1e-6, growth below 100), 1.5e-3 for bf16x3 (2^-16).
"""

import numpy as np
import pytest
import torch

from matfree_amd import decomp, operators, problems
from oracle import slq as oslq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2052, 2053])
@pytest.mark.parametrize("P,k", [(32, 20), (200, 20), (300, 30), (300, 41), (319, 12), (320, 12),
                                 (512, 12)])
def test_columns_of_a_block(cuda, n, P, k):
    rng = np.random.default_rng(n + P + k)
    B = rng.standard_normal((n, n)) / np.sqrt(n)
    A = (0.17 * (B + B.T) + 1.5 * np.eye(n)).astype(np.float32)
    V = rng.standard_normal((P, n)).astype(np.float32)
    out = decomp.hessenberg(k, reortho="full").batched(
        operators.dense_matvec, torch.tensor(V, device=cuda), torch.tensor(A, device=cuda))
    H = out.J_small.double().cpu().numpy()
    picks = [0, 1, P // 2, P - 1]
    _, Href, _, _ = oslq.hessenberg_forward(oslq.DenseOperator(A, np.float64), k, V[picks],
                                            np.float64)
    for i, p in enumerate(picks):
        assert np.linalg.norm(H[p] - Href[i]) <= 1e-4 * np.linalg.norm(Href[i])
    Q = out.Q_tall.double()
    gram = Q @ Q.transpose(1, 2)
    assert float((gram - torch.eye(k, device=cuda, dtype=torch.float64)).abs().max()) <= 1e-5


@pytest.mark.parametrize("precision,n,P,tol", [
    ("bf16x3", 2052, 6, 1.5e-3), ("bf16x3", 2052, 40, 1.5e-3), ("bf16x3", 2053, 40, 1.5e-3),
    ("fp32", 2052, 6, 1e-4), ("fp32", 4100, 6, 1e-4), ("fp32", 4100, 40, 1e-4)])
def test_reverse_pass_planes(cuda, precision, n, P, tol):
    k = 6
    rng = np.random.default_rng(n + P)
    V = rng.standard_normal((P, n)).astype(np.float32)
    dQ, dH = rng.standard_normal((P, k, n)), rng.standard_normal((P, k, k))

    def t(x, grad=False):
        return torch.tensor(np.asarray(x, np.float32), device=cuda, requires_grad=grad)

    # about four neighbours within a lengthscale at n = 2052
    X = problems.rbf_points(n, seed=n)
    oracle = oslq.RBFOperator(X, 0.05, 1.0, np.float64)
    params = tuple(torch.tensor(x, dtype=torch.float64, device=cuda, requires_grad=True)
                   for x in (0.05, 1.0))
    Vt = t(V, True)
    out = decomp.hessenberg(k, reortho="full").batched(operators.RBF(X, precision=precision), Vt,
                                                       *params)
    ((out.Q_tall * t(dQ)).sum() + (out.J_small * t(dH)).sum()).backward()
    Q, H, r, c = oslq.hessenberg_forward(oracle, k, V, np.float64)
    dv, g = np.empty((P, n)), 0.0
    for p in range(P):
        dv[p], gp = oslq.hessenberg_adjoint(oracle, Q[p], H[p], r[p], float(c[p]), dQ[p].T, dH[p],
                                            np.zeros(n), 0.0)
        g = g + np.asarray(gp)
    got = np.asarray([float(x.grad) for x in params])
    assert np.linalg.norm(Vt.grad.double().cpu().numpy() - dv) <= tol * np.linalg.norm(dv)
    assert np.linalg.norm(got - g) <= tol * np.linalg.norm(g)
