"""Gram-Schmidt steps of rows of one chunk (n <= 2048), one workgroup a probe.

The Arnoldi relation and the orthogonality of the basis at the sizes where the
kernel's groups end: the shortest row it takes and the one below, rows that end
inside a group of two and of four, one and two rounds of column batches, the
whole chunk and one element more (the kernels with a launch per pass).

Tolerances: one FP32 operation rounds by 2^-24 = 6e-8; a dot of 2048 terms in a
tree of 8-term chains stays below 20 of them, and so does the projection over
up to 41 columns.  The relation collects the product's error (1e-6 of |A|) and
the two projections' (2 x 1.2e-6): 1e-5 |A|.  Twice-orthogonalised columns keep
the second pass's rounding, 1.2e-6 a pair before normalisation: 1e-5.
"""

import pytest
import torch

from matfree_amd import decomp, operators

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,P,k", [
    (3, 2, 3), (4, 1, 4), (5, 3, 5), (7, 2, 6), (66, 5, 9), (255, 2, 8), (1023, 3, 33),
    (1025, 2, 41), (2046, 2, 12), (2047, 33, 10), (2048, 3, 34), (2049, 3, 12)])
def test_relation_and_orthogonality(cuda, n, P, k):
    gen = torch.Generator().manual_seed(n)
    B = torch.randn((n, n), generator=gen, dtype=torch.float64)
    A = B @ B.T / n + 0.5 * torch.eye(n, dtype=torch.float64)
    A = (0.5 * (A + A.T)).float()
    V = torch.randn((P, n), generator=gen)
    out = decomp.hessenberg(k, reortho="full").batched(operators.dense_matvec, V.to(cuda),
                                                       A.to(cuda))
    Q, H = out.Q_tall.double().cpu(), out.J_small.double().cpu()  # P k n, P k k
    r, c = out.residual.double().cpu(), out.init_length_inv.double().cpu()
    if Q.shape[1] != k:
        Q = Q.transpose(1, 2)
    norm = torch.linalg.matrix_norm(A.double(), 2)
    lhs = Q @ A.double()
    rhs = H.transpose(1, 2) @ Q
    rhs[:, -1] += r
    assert float((lhs - rhs).norm(dim=2).max() / norm) < 1e-5
    gram = Q @ Q.transpose(1, 2) - torch.eye(k, dtype=torch.float64)
    assert float(gram.abs().max()) < 1e-5
    first = V.double() * c[:, None]
    assert float((Q[:, 0] - first).norm(dim=1).max()) < 1e-6
