"""The decomposition a reverse pass is taken at is the one that was returned
(run on an MI355X).

The columns of a basis stay orthonormal, so the cotangents dQ_j = sum_i S_ij
q_i with a symmetric S (of the constant loss sum_ij S_ij q_i . q_j / 2) give
zero at the basis that the q_i come from.  With the same bits only the rounding
of the dots and of the sums over k columns is left, 2^-24 times less than a
hundred of the gradient of a random loss of the same size: 1e-5.  At the basis
of other products the gradient moves with the difference of the two: a
stored matrix with one eigenvalue far from the others has one of 4e-4 and more.
"""

import ctypes

import numpy as np
import pytest
import torch

from matfree_amd import _lib, _runtime, decomp, operators

pytestmark = pytest.mark.gpu

SIZES = [(300, 4, 20), (300, 40, 20), (1500, 4, 40), (2500, 3, 30), (2500, 66, 12)]


def problem(n, P, k, cuda):
    rng = np.random.default_rng(n + P)
    U, _ = np.linalg.qr(rng.standard_normal((n, n)))
    ev = rng.uniform(0.5, 1.5, n)
    ev[0] = 1e3
    A = (U * ev) @ U.T
    A = 0.5 * (A + A.T)
    S = rng.standard_normal((P, k, k))
    S = (S + S.transpose(0, 2, 1)) / np.sqrt(2.0 * k)
    V, G = rng.standard_normal((P, n)), rng.standard_normal((P, k, n))
    return (torch.tensor(x, dtype=torch.float32, device=cuda) for x in (A, V, S, G))


@pytest.mark.parametrize("n,P,k", SIZES)
def test_differentiated_call(cuda, n, P, k):
    A, V, S, G = problem(n, P, k, cuda)
    norms = []
    for constant in (True, False):
        Ag, Vg = A.clone().requires_grad_(), V.clone().requires_grad_()
        out = decomp.hessenberg(k, reortho="full").batched(operators.dense_matvec, Vg, Ag)
        SQ = S @ out.Q_tall.detach()
        dQ = SQ if constant else G * (SQ.norm() / G.norm())
        (out.Q_tall * dQ).sum().backward()
        norms.append((float(Ag.grad.norm()), float(Vg.grad.norm())))
    for zero, one in zip(*norms):
        assert zero < 1e-5 * one


@pytest.mark.parametrize("n,P,k", SIZES)
@pytest.mark.parametrize("units", [0, _lib.ARNOLDI_FP32_UNITS])
def test_c_entries(cuda, n, P, k, units):
    A, V, S, G = problem(n, P, k, cuda)
    ctx = _runtime.context(cuda)
    desc, keep = operators.dense_matvec.descriptor(n, (A,), cuda)
    ptr = _runtime.ptr
    Q, H = torch.empty((k, P, n), device=cuda), torch.empty((P, k, k), device=cuda)
    r, c = torch.empty((P, n), device=cuda), torch.empty((P,), device=cuda)
    ctx.call("slq_arnoldi", ctypes.byref(desc), ptr(V), P, k, 1 | units, ptr(Q), ptr(H), ptr(r),
             ptr(c))
    SQ = S @ Q.transpose(0, 1)
    norms = []
    for dQ in (SQ, G * (SQ.norm() / G.norm())):
        dQ = dQ.transpose(0, 1).contiguous()
        dA, dv = torch.empty((n, n), device=cuda), torch.empty((P, n), device=cuda)
        ctx.call("slq_arnoldi_vjp", ctypes.byref(desc), ptr(V), P, k, 1 | units, 1, ptr(dQ), None,
                 None, None, ptr(dv), None, ptr(dA))
        norms.append((float(dA.norm()), float(dv.norm())))
    del keep
    for zero, one in zip(*norms):
        assert zero < 1e-5 * one
