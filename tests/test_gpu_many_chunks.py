"""The Gram-Schmidt passes of many blocks (chunks of 2048 elements times probes).

From 1024 blocks the passes over the basis take the probes in alternating order
(n = 2052 and 2050 here; rows of one chunk, n = 131 and 132, take a step in one
workgroup a probe).  ``tridiag_sym`` of a stored matrix with spectrum in [1, 2]
against the FP64 restatement, rows of whole float4 groups and others.  The
columns a block of the dots takes and the projection's rule:
test_gpu_pass_rules.py.  Tolerances:
the FP32 products are good to 1e-6 and the recurrence at these depths grows an
error by less than 100 (1e-4 normwise); two classical passes keep the basis
orthonormal to a few FP32 roundings of sums over n (1e-5).
"""

import numpy as np
import pytest
import torch

from matfree_amd import decomp, operators
from oracle import slq as oslq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,P,k", [(2052, 511, 9), (2052, 512, 17), (2050, 513, 33),
                                   (131, 1024, 8), (132, 1023, 34)])
def test_tridiag_few_and_many_blocks(cuda, n, P, k):
    rng = np.random.default_rng(n + P)
    B = rng.standard_normal((n, n)) / np.sqrt(n)
    A = (0.17 * (B + B.T) + 1.5 * np.eye(n)).astype(np.float32)
    V = rng.standard_normal((P, n)).astype(np.float32)
    out = decomp.hessenberg(k, reortho="full").batched(
        operators.dense_matvec, torch.tensor(V, device=cuda), torch.tensor(A, device=cuda))
    Q = out.Q_tall.double().cpu().numpy()
    H = out.J_small.double().cpu().numpy()
    picks = [0, 1, P // 2, P - 2, P - 1]
    _, Href, _, _ = oslq.hessenberg_forward(oslq.DenseOperator(A, np.float64), k, V[picks],
                                            np.float64)
    for i, p in enumerate(picks):
        assert np.linalg.norm(H[p] - Href[i]) <= 1e-4 * np.linalg.norm(Href[i])
    G = np.einsum("pkn,pln->pkl", Q, Q) if Q.shape[1] == k else np.einsum("pnk,pnl->pkl", Q, Q)
    assert np.abs(G - np.eye(k)).max() <= 1e-5
