"""Stored-matrix FP32 products of up to 32 vectors beyond n = 4096, whose blocks
are split evenly over the workgroups (run on an MI355X): row blocks of one to
three segments, the last block a partial tile alone, sizes on both sides of the
split's range, against an FP64 product, with the scratch full of NaN from the
call before (planes without a segment are written too).

Tolerance: 2e-6 normwise, as for the other FP32 products."""

import pytest
import torch

from matfree_amd import decomp, operators

pytestmark = pytest.mark.gpu


def rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


# one row block more than 4096's; 4225 and 8193 end in a partial tile of its own block; 7360 /
# 7361 and 8192 / 8193: a row block a workgroup in between; 8960, 10413, 12289: two segments
@pytest.mark.parametrize("n", [96, 97, 4096, 4097, 4128, 4225, 5003, 6144, 7360, 7361, 8192, 8193,
                               8960, 10413, 12289])
def test_against_fp64(cuda, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, n), generator=gen, device=cuda)
    A = A + A.T
    A64 = A.double()
    nan = torch.full((32, n), float("nan"), device=cuda)
    for P in (1, 7, 25, 32):
        V = torch.randn((P, n), generator=gen, device=cuda)
        assert bool(operators.dense_matvec(nan, A).isnan().all())
        assert rel(operators.dense_matvec(V, A), V.double() @ A64) < 2e-6, (n, P)


@pytest.mark.parametrize("n,P", [(4225, 5), (5003, 28), (8193, 3), (8961, 31)])
def test_split_sums_left_to_the_dots(cuda, n, P):
    # A q_j = Q h_j: the products' sums are formed by the Gram-Schmidt dots (2e-6 of the
    # product and as much of two projections of three columns: 5e-6)
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, n), generator=gen, device=cuda)
    A = (A + A.T) / (2 * n) ** 0.5
    V = torch.randn((P, n), generator=gen, device=cuda)
    out = decomp.hessenberg(3, reortho="full").batched(operators.dense_matvec, V, A)
    Q, H = out.Q_tall.double(), out.J_small.double()
    image = H.transpose(1, 2) @ Q
    image[:, -1] += out.residual.double()
    assert rel(image, Q @ A.double()) < 5e-6
