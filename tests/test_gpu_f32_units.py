"""Decompositions of a stored matrix on the FP32 matrix cores (those that are
differentiated) at the edges of the products' tiles (run on an MI355X): the
Arnoldi relation to 1e-5 of |A| (products to 1e-6 of it, two projections of up
to eight columns)."""

import pytest
import torch

from matfree_amd import decomp, operators

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 31, 32, 33, 63, 65, 127, 128, 129, 257, 1001])
@pytest.mark.parametrize("P", [1, 32, 33, 65])
def test_relation_of_the_matrix_cores_products(cuda, n, P):
    k = min(n, 8)
    gen = torch.Generator().manual_seed(n + P)
    B = torch.randn((n, n), generator=gen, dtype=torch.float64)
    A = B @ B.T / n + 0.5 * torch.eye(n, dtype=torch.float64)
    A = (0.5 * (A + A.T)).float()
    V = torch.randn((P, n), generator=gen)
    out = decomp.hessenberg(k, reortho="full").batched(
        operators.dense_matvec, V.to(cuda), A.to(cuda).requires_grad_())
    Q, H, r = (x.detach().double().cpu() for x in (out.Q_tall, out.J_small, out.residual))
    norm = torch.linalg.matrix_norm(A.double(), 2)
    rhs = H.transpose(1, 2) @ Q
    rhs[:, -1] += r
    assert float((Q @ A.double() - rhs).norm(dim=2).max() / norm) < 1e-5
