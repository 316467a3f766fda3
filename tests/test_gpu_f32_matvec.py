"""The FP32 block matvec's forms (run on an MI355X): up to 32 vectors (stream
and wave forms), 33-64 and more (workgroup form), at the edges of their tiles,
blocks and slices, against an FP64 product; infinities, NaN and values beyond
BF16's range as FP32 arithmetic has them; the probes split in groups when the
scratch is the least size.

Tolerance: each of the n products and sums of an output rounds by at most
2^-24 of a partial sum; over sums of random sign the normwise error stays
under 2e-6 for n <= 16384 (the bound of the FP32 matvec tests)."""

import ctypes

import numpy as np
import pytest
import torch

from matfree_amd import _lib, _runtime, decomp, operators, problems

pytestmark = pytest.mark.gpu

# tile (32), row-block (32, 128), load-block (128 columns) and slice edges
SIZES = [1, 3, 31, 32, 33, 127, 129, 160, 257, 1001, 4095, 4097]
PROBES = [5, 16, 32, 33, 64, 65, 128, 130]


def rel(got, ref):
    return float(np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("n", SIZES)
def test_stored_matrix_against_fp64(cuda, n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)).astype(np.float32)
    A = A + A.T
    for P in [1] + PROBES:
        V = rng.standard_normal((P, n)).astype(np.float32)
        W = operators.dense_matvec(torch.as_tensor(V, device=cuda), torch.as_tensor(A, device=cuda))
        assert rel(W, V.astype(np.float64) @ A.astype(np.float64)) < 2e-6, (n, P)


@pytest.mark.parametrize("dim", [1, 2, 3, 4])
def test_rbf_against_fp64(cuda, dim):
    for n in SIZES:
        X = problems.rbf_points(n, seed=n, dim=dim)
        K = problems.rbf_dense64(X, 0.5, 1e-2)
        op = operators.RBF(torch.as_tensor(X, device=cuda))
        for P in PROBES if n < 4000 else (32, 65):
            V = np.random.default_rng(P).standard_normal((P, n)).astype(np.float32)
            W = op(torch.as_tensor(V, device=cuda), 0.5, 1e-2)
            assert rel(W, V.astype(np.float64) @ K) < 2e-6, (n, dim, P)


@pytest.mark.parametrize("P", [32, 64, 100])
def test_non_finite_and_huge_values(cuda, P):
    n = 300
    rng = np.random.default_rng(5)
    A = rng.uniform(0.5, 1.0, (n, n)).astype(np.float32)
    A = 0.5 * (A + A.T)
    V = rng.uniform(0.5, 1.0, (P, n)).astype(np.float32)
    V[0, 7] = np.inf
    V[1, 8] = -np.inf
    V[2, 9] = np.nan
    V[3, 10], V[3, 11] = np.inf, -np.inf
    big = np.float32(3.4e38)  # rounds to infinity in BF16
    V[4] = 0.0
    V[4, 12] = big
    V[5] *= np.float32(1e-30)  # low parts near the end of the normal range
    W = operators.dense_matvec(torch.as_tensor(V, device=cuda), torch.as_tensor(A, device=cuda))
    W = W.cpu().numpy().astype(np.float64)
    ref = V.astype(np.float64) @ A.astype(np.float64)
    assert np.all(W[0] == np.inf) and np.all(W[1] == -np.inf)
    assert np.all(np.isnan(W[2])) and np.all(np.isnan(W[3]))
    for p in range(4, P):
        np.testing.assert_allclose(W[p], ref[p], rtol=2e-6)


def test_decomposition_writes_the_planes(cuda):
    # P > 32: the normalisation writes the next matvec's planes (odd n, n % 4 = 2, n % 4 = 0)
    for n in (301, 302, 304):
        A = torch.as_tensor(problems.dense_spd(n, seed=1, shift=0.5), device=cuda)
        V = torch.randn((40, n), generator=torch.Generator(device="cuda").manual_seed(1),
                        device=cuda)
        all_at_once = decomp.tridiag_sym(8).batched(operators.dense_matvec, V, A)
        few = [decomp.tridiag_sym(8).batched(operators.dense_matvec, V[s:s + 20], A)
               for s in (0, 20)]
        J = torch.cat([f.J_small for f in few])
        assert float((all_at_once.J_small - J).abs().max()) < 1e-5 * float(J.abs().max())


def test_least_scratch_gives_the_same_results(cuda):
    # a call that fits slq_logdet_noalloc's scratch only with the planes of part of its probes
    P, k = 128, 100
    limit = _lib.NOALLOC_SCRATCH_BYTES
    ctx = _runtime.context(cuda)
    for n in range(4400, 4000, -1):
        X = torch.as_tensor(problems.rbf_points(n, seed=3), device=cuda)
        op = operators.RBF(X)
        desc, keep = op.descriptor(n, (0.5, 1e-1), cuda)
        need = ctx.workspace_bytes("logdet", desc, P, k)
        if need <= limit + 4 * 40 * n:  # the third plane takes 4 x 48 n bytes
            break
    assert limit < need <= limit + 160 * n
    Z = torch.as_tensor(np.random.default_rng(0).choice([-1.0, 1.0], (P, n)).astype(np.float32),
                        device=cuda)
    out = []
    for entry in ("slq_logdet", "slq_logdet_noalloc"):
        per = torch.zeros((P,), dtype=torch.float64, device=cuda)
        ctx.call(entry, ctypes.byref(desc), _runtime.ptr(Z), P, k, _runtime.ptr(per), None, None,
                 None)
        out.append(per.cpu().numpy())
    del keep
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("n,P", [(8961, 25), (8963, 32), (9024, 31), (10413, 32)])
def test_probe_tiles_of_the_stream_form(cuda, n, P):
    # vectors read in the order of the fragments: the first row that takes it, no whole last
    # tile, and the tiles written by the normalisation (the three vectors' relation
    # A q_j = Q h_j, whose last columns have few terms: 2e-6 as for the product)
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, n), generator=gen, device="cuda")
    A = (A + A.T) / (2 * n) ** 0.5
    V = torch.randn((P, n), generator=gen, device="cuda")
    A64 = A.double()
    W = operators.dense_matvec(V, A)
    assert rel(W, (V.double() @ A64).cpu().numpy()) < 2e-6
    out = decomp.hessenberg(3, reortho="full").batched(operators.dense_matvec, V, A)
    Q, H = out.Q_tall.double(), out.J_small.double()
    if Q.shape[1] != 3:
        Q = Q.transpose(1, 2)
    image = H.transpose(1, 2) @ Q
    image[:, -1] += out.residual.double()
    for j in range(3):
        assert rel(image[:, j], (Q[:, j] @ A64).cpu().numpy()) < 2e-6
