"""The reverse scan's operator products at the sizes where their route changes.

The projection that forms a product's input writes the product's planes when
the rows are whole groups of four (n % 4 == 0), the product's split-K sum is
formed by the dots that read it, and the rows of dQ^T Q are done together
unless the rows of dQ differ in alignment (P n not a multiple of 4).  Random
cotangents on every output of ``hessenberg`` against the FP64 restatement of
decomp.py:480-600, one chunk of a probe's vector (a step in one workgroup a
probe) and two, more than 32 probes and fewer.  The planes from the projection
of longer rows: test_gpu_pass_rules.py.  Tolerances: 1e-4 normwise for FP32 operators of
condition number below ten at depth 6 (products to 1e-6, growth through the
scan below 100); for bf16x3, whose products are good to 2^-16, the same growth
gives 1.5e-3.
"""

import numpy as np
import pytest
import torch

from matfree_amd import decomp, operators, problems
from oracle import slq as oslq

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("kind,n,P,tol", [
    ("dense", 131, 3, 1e-4), ("dense", 131, 4, 1e-4), ("dense", 132, 33, 1e-4),
    ("fp32", 132, 5, 1e-4), ("fp32", 133, 33, 1e-4), ("fp32", 2052, 33, 1e-4),
    ("bf16x3", 132, 33, 1.5e-3), ("bf16x3", 2052, 3, 1.5e-3), ("bf16x3", 2053, 6, 1.5e-3)])
def test_reverse_pass_routes(cuda, kind, n, P, tol):
    k = 6
    rng = np.random.default_rng(n + P)
    V = rng.standard_normal((P, n)).astype(np.float32)
    dQ, dH = rng.standard_normal((P, k, n)), rng.standard_normal((P, k, k))
    dr, dc = rng.standard_normal((P, n)), rng.standard_normal(P)

    def t(x, grad=False):
        return torch.tensor(np.asarray(x, np.float32), device=cuda, requires_grad=grad)

    Vt = t(V, True)
    if kind == "dense":
        B = rng.standard_normal((n, n)) / np.sqrt(n)
        A = (0.2 * (B + B.T) + 2.0 * np.eye(n)).astype(np.float32)
        op, params = oslq.DenseOperator(A, np.float64), (t(A, True),)
        mv = operators.dense_matvec
    else:
        # about four neighbours within a lengthscale at n = 2052
        X = problems.rbf_points(n, seed=n)
        op = oslq.RBFOperator(X, 0.05, 1.0, np.float64)
        params = tuple(torch.tensor(x, dtype=torch.float64, device=cuda, requires_grad=True)
                       for x in (0.05, 1.0))
        mv = operators.RBF(X, precision=kind)
    out = decomp.hessenberg(k, reortho="full").batched(mv, Vt, *params)
    loss = ((out.Q_tall * t(dQ)).sum() + (out.J_small * t(dH)).sum()
            + (out.residual * t(dr)).sum() + (out.init_length_inv * t(dc)).sum())
    loss.backward()
    Q, H, r, c = oslq.hessenberg_forward(op, k, V, np.float64)
    dv, g = np.empty((P, n)), 0.0
    for p in range(P):
        dv[p], gp = oslq.hessenberg_adjoint(op, Q[p], H[p], r[p], float(c[p]), dQ[p].T, dH[p],
                                            dr[p], dc[p])
        g = g + np.asarray(gp)
    assert rel(Vt.grad.cpu(), dv) <= tol
    got = params[0].grad.cpu() if kind == "dense" else [float(x.grad) for x in params]
    assert rel(got, g) <= tol
