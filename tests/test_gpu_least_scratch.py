"""``slq_logdet_noalloc`` with the least matvec scratch (run on an MI355X).

A call that fits the static scratch only with the FP32 matvec's planes in
passes over the columns runs the kernels, slices and sums of ``slq_logdet``:
the same bits, for probe counts that fill no whole block of 32, 64 or 128 and
for a stored matrix on both sides of n = 8960, where up to 32 vectors of their
own would be read in another layout."""

import ctypes

import numpy as np
import pytest
import torch

from matfree_amd import _lib, _runtime, operators, problems

pytestmark = pytest.mark.gpu

LIMIT = _lib.NOALLOC_SCRATCH_BYTES


def saving(P, n):
    """Bytes the least scratch does without: half of a plane pair less 16 floats a column."""
    pad = -(-P // 64) * 64 if P <= 64 else -(-P // 128) * 128
    return 4 * (-(-n // 32) * 32) * (pad // 2 - 16)


def both_entries(ctx, desc, P, n, k, cuda):
    Z = torch.as_tensor(np.random.default_rng(P).choice([-1.0, 1.0], (P, n)).astype(np.float32),
                        device=cuda)
    out = []
    for entry in ("slq_logdet", "slq_logdet_noalloc"):
        per = torch.zeros((P,), dtype=torch.float64, device=cuda)
        ctx.call(entry, ctypes.byref(desc), _runtime.ptr(Z), P, k, _runtime.ptr(per), None, None,
                 None)
        out.append(per.cpu().numpy())
    return out


@pytest.mark.parametrize("n,P,k", [(16384, 34, 108), (16257, 96, 33), (16257, 160, 18)])
def test_stored_matrix(cuda, n, P, k):
    gen = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn((n, n), generator=gen, device=cuda)
    A = 0.1 * (A + A.T) / n**0.5
    A.diagonal().add_(1.0)
    ctx = _runtime.context(cuda)
    desc, keep = operators.dense_matvec.descriptor(n, (A,), cuda)
    need = ctx.workspace_bytes("logdet", desc, P, k)
    assert LIMIT < need <= LIMIT + saving(P, n)
    full, least = both_entries(ctx, desc, P, n, k, cuda)
    del keep
    assert np.all(np.isfinite(full))
    np.testing.assert_array_equal(full, least)


@pytest.mark.parametrize("P,k", [(40, 150), (64, 90), (96, 70), (160, 40), (200, 30)])
def test_rbf(cuda, P, k):
    ctx = _runtime.context(cuda)
    n = int(LIMIT / (4 * P * k))
    while n > 1000:  # the largest n that fits without half of the saving
        X = torch.as_tensor(problems.rbf_points(n, seed=3), device=cuda)
        desc, keep = operators.RBF(X).descriptor(n, (0.5, 1e-1), cuda)
        need = ctx.workspace_bytes("logdet", desc, P, k)
        if need <= LIMIT + saving(P, n) // 2:
            break
        n -= 3
    assert LIMIT < need
    full, least = both_entries(ctx, desc, P, n, k, cuda)
    del keep
    np.testing.assert_array_equal(full, least)
