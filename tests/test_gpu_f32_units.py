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


# one, a few, eight, nine and fifteen tiles a slice; 1 to 8 slices; up to 2048
# dealt to waves for up to 32 probes and not beyond, or with more probes
@pytest.mark.parametrize("n", [1, 31, 96, 255, 257, 480, 511, 513, 991, 1500, 2047, 2048])
@pytest.mark.parametrize("P", [1, 31, 32])
def test_few_probes_take_the_same_sums(cuda, n, P):
    """A probe's decomposition does not depend on how many there are: the tiles'
    sums are added in one order, bit for bit."""
    gen = torch.Generator().manual_seed(n)
    A = (torch.randn((n, n), generator=gen) / n**0.5).to(cuda).requires_grad_()
    V = torch.randn((33, n), generator=gen).to(cuda)
    many, few = (decomp.hessenberg(min(n, 3), reortho="full").batched(
        operators.dense_matvec, x, A) for x in (V, V[:P]))
    for a, b in zip(few, many):
        assert torch.isfinite(a).all()
        assert torch.equal(a, b[:P])
