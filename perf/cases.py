"""Performance cases of the stochastic-Lanczos path: what programs on top of this package call.

Five kinds of call, each through a public entry point:

* ``matvec``  -- ``op(V, *params)``: the block matvec of every operator form;
* ``tridiag`` -- ``decomp.tridiag_sym(k).batched(op, V, A)``: the decomposition
  of a stored matrix, all of its outputs;
* ``vjp``     -- the reverse pass through that decomposition (cotangents of the
  start vectors and of the matrix for a loss on the tridiagonals);
* ``logdet``  -- a whole log-determinant request on probes in memory:
  decomposition and quadrature; with ``grad`` the parameter cotangents too;
* ``cg``      -- a Gaussian-process solve by conjugate gradients.

Spectra matter for the decompositions: a Krylov basis of an RBF kernel matrix
amplifies any change of rounding by orders of magnitude once its few large
eigenvalues have converged, so FP32 decompositions are taken on stored
matrices with a Wishart spectrum and the FP32 RBF operator is taken by its
block matvec; the two log-determinant requests run the RBF operator whole.
"""

import math

import torch

from matfree_amd import decomp, funm, linalg, operators

LENGTHSCALE = 0.5
NOISE = 1e-2
SHIFT = 0.1  # of the Wishart matrices B B^T / n + SHIFT I


def listed():
    return [
        # one iteration of a user's own block method on a few thousand points
        dict(name="matvec rbf fp32 small", call="matvec", form="rbf", precision="fp32",
             n=2048, dim=3, P=16),
        # the default operator on an ordinary ragged data set
        dict(name="matvec rbf fp32 ragged", call="matvec", form="rbf", precision="fp32",
             n=10413, dim=2, P=32),
        # the default operator at the full benchmark size
        dict(name="matvec rbf fp32 large", call="matvec", form="rbf", precision="fp32",
             n=32768, dim=3, P=128),
        # the block matvec of the headline log-determinant
        dict(name="matvec rbf bf16x2 large", call="matvec", form="rbf", precision="bf16x2",
             n=32768, dim=3, P=128),
        # a matrix packed once and applied many times
        dict(name="matvec packed bf16x2", call="matvec", form="packed", precision="bf16x2",
             n=16384, dim=0, P=256),
        # a small decomposition: latency and launches
        dict(name="tridiag small", call="tridiag", n=1001, P=16, k=20),
        # an ordinary serving request on a stored matrix, every row misaligned
        dict(name="tridiag ragged", call="tridiag", n=10413, P=32, k=37),
        # the stored-matrix benchmark's matrix and probes (at depths beyond about 40 FP32
        # rounding alone moves the last vectors by more than 2e-5)
        dict(name="tridiag large", call="tridiag", n=16384, P=256, k=40),
        # one training step through a decomposition
        dict(name="vjp", call="vjp", n=4096, P=32, k=32),
        # the headline benchmark: one whole request
        dict(name="logdet", call="logdet", n=32768, P=128, k=64, grad=False),
        # a hyper-parameter step of an ordinary size: value and gradient
        dict(name="logdet gradient", call="logdet", n=8192, P=32, k=32, grad=True),
        # the linear solve of a GP posterior mean
        dict(name="cg", call="cg", n=8192, dim=3),
    ]


def _size(rng, lo, hi):
    """Log-uniform; one in two as it falls (mostly odd or ragged), one in two a multiple of 64."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else max(lo, n // 64 * 64)


def _probes(rng, hi):
    if rng.random() < 0.6:
        return rng.choice([p for p in (16, 32, 64, 128, 256) if p <= hi])
    return int(round(math.exp(rng.uniform(0.0, math.log(hi)))))


def draw(rng):
    call = rng.choice(["matvec", "matvec", "matvec", "tridiag", "tridiag", "vjp", "logdet",
                       "logdet", "cg"])
    if call == "matvec":
        form, precision = rng.choice([("rbf", "fp32"), ("rbf", "fp32"), ("rbf", "bf16x2"),
                                      ("dense", "fp32"), ("dense", "fp32"),
                                      ("packed", "bf16x2"), ("packed", "bf16")])
        n = _size(rng, 512, 32768 if form == "rbf" else 16384)
        dim = rng.choice([1, 2, 3]) if form == "rbf" else 0
        return dict(call=call, form=form, precision=precision, n=n, dim=dim,
                    P=_probes(rng, 128 if form == "rbf" else 256))
    if call == "tridiag":
        return dict(call=call, n=_size(rng, 512, 16384), P=_probes(rng, 256),
                    k=rng.randint(8, 40))
    if call == "vjp":
        return dict(call=call, n=_size(rng, 512, 6000), P=_probes(rng, 64), k=rng.randint(8, 32))
    if call == "logdet":
        grad = rng.random() < 0.5
        return dict(call=call, n=_size(rng, 2048, 12288 if grad else 32768),
                    P=rng.choice([16, 32, 64, 128]), k=rng.randint(16, 64), grad=grad)
    return dict(call=call, n=_size(rng, 1024, 16384), dim=rng.choice([2, 3]))


# ---- inputs ------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _points(case, gen):
    return torch.rand((case["n"], case.get("dim", 3)), generator=gen, device="cuda")


def _wishart(n, gen):
    B = torch.randn((n, n), generator=gen, device="cuda")
    A = B @ B.T / n
    A = 0.5 * (A + A.T)
    A.diagonal().add_(SHIFT)
    return A


def _inputs(case, seed):
    """The tensors of a case, the same for ``prepare`` and ``exact``."""
    gen = _generator(seed)
    call, n = case["call"], case["n"]
    if call == "cg":
        X = _points(case, gen)
        f = torch.sin(6.0 * X).sum(dim=1)
        y = f + math.sqrt(NOISE) * torch.randn((n,), generator=gen, device="cuda")
        return dict(X=X, y=y)
    if call == "logdet":
        bits = torch.randint(0, 2, (case["P"], n), generator=gen, device="cuda")
        return dict(X=_points(case, gen), Z=(2 * bits - 1).to(torch.float32))
    if call == "matvec" and case["form"] == "rbf":
        X = _points(case, gen)
        return dict(X=X, V=torch.randn((case["P"], n), generator=gen, device="cuda"))
    A = _wishart(n, gen)
    V = torch.randn((case["P"], n), generator=gen, device="cuda")
    if call == "vjp":
        k, P = case["k"], case["P"]
        return dict(A=A, V=V, G=torch.randn((P, k, k), generator=gen, device="cuda"))
    return dict(A=A, V=V)


def prepare(case, seed):
    s = dict(case=case, **_inputs(case, seed))
    call = case["call"]
    if call == "matvec":
        if case["form"] == "rbf":
            s["op"] = operators.RBF(s["X"], precision=case["precision"])
            s["params"] = (LENGTHSCALE, NOISE)
        elif case["form"] == "dense":
            s["op"], s["params"] = operators.dense_matvec, (s["A"],)
        else:
            s["op"] = operators.packed_matvec
            s["params"] = (operators.pack(s.pop("A"), case["precision"]),)
    elif call in ("tridiag", "vjp"):
        s["decompose"] = decomp.tridiag_sym(case["k"])
        if call == "vjp":
            s["A"].requires_grad_()
            s["V"].requires_grad_()
    elif call == "logdet":
        s["op"] = operators.RBF(s["X"], precision="bf16x2")
    else:
        s["op"] = operators.RBF(s["X"])
    return s


def run(state):
    case = state["case"]
    call = case["call"]
    if call == "matvec":
        return state["op"](state["V"], *state["params"])
    if call == "tridiag":
        out = state["decompose"].batched(operators.dense_matvec, state["V"], state["A"])
        return dict(Q=out.Q_tall, T=out.J_small, residual=out.residual, length=out.init_length_inv)
    if call == "vjp":
        out = state["decompose"].batched(operators.dense_matvec, state["V"], state["A"])
        dV, dA = torch.autograd.grad(out.J_small, (state["V"], state["A"]), state["G"])
        return dict(T=out.J_small.detach(), dV=dV, dA=dA)
    if call == "logdet":
        Z, params = state["Z"], (LENGTHSCALE, NOISE)
        if not case["grad"]:
            per_probe, mean = funm.logdet_per_probe(state["op"], Z, case["k"], params)
            return dict(per_probe=per_probe, mean=mean)
        per_probe, mean, grads = funm.logdet_value_and_grad(state["op"], Z, case["k"], params)
        return dict(per_probe=per_probe, mean=mean, dlengthscale=grads[0], dnoise=grads[1])
    x, _ = linalg.cg(state["op"], state["y"], LENGTHSCALE, NOISE)
    return x


# ---- the work a pass cannot do without ------------------------------------------


def work(case):
    n, call = case["n"], case["call"]
    if call == "cg":
        # one pass over the kernel per iteration; about sqrt(condition) iterations
        return dict(bytes=4.0 * n * (case["dim"] + 2), flops=2.0 * n * n * 400)
    P = case["P"]
    if call == "matvec":
        if case["form"] == "rbf":
            operand = 4.0 * n * case["dim"]
        else:
            per_entry = {"fp32": 4.0, "bf16x2": 4.0, "bf16": 2.0}[case["precision"]]
            operand = per_entry * n * n
        return dict(bytes=operand + 8.0 * n * P, flops=2.0 * n * n * P)
    k = case["k"]
    steps = 2.0 * n * n * P * k + 8.0 * n * P * k * (k + 1) / 2
    if call == "tridiag":
        return dict(bytes=4.0 * n * n + 4.0 * n * P * (k + 2) + 4.0 * P * k * k, flops=steps)
    if call == "vjp":
        # forward, reverse recursion and the outer products of the matrix cotangent
        return dict(bytes=8.0 * n * n + 8.0 * n * P + 8.0 * P * k * k,
                    flops=2.0 * steps + 2.0 * n * n * P * k)
    flops = 2.0 * steps + 2.0 * n * n * P * k if case["grad"] else steps
    return dict(bytes=12.0 * n + 8.0 * P, flops=flops)


# ---- the same in 64 bits, by plain torch -------------------------------------------


def _kernel64(X, lengthscale, noise):
    """Dense FP64 RBF matrix in blocks of rows (direct differences)."""
    n = X.shape[0]
    X = X.to(torch.float64)
    K = torch.empty((n, n), dtype=torch.float64, device=X.device)
    rows = max(1, (1 << 26) // n)
    for s in range(0, n, rows):
        d2 = ((X[s:s + rows, None, :] - X[None, :, :]) ** 2).sum(-1)
        K[s:s + rows] = torch.exp(d2 * (-0.5 / lengthscale**2))
    K.diagonal().add_(noise)
    return K


def _arnoldi64(matvec, V, k):
    """Arnoldi with Gram-Schmidt twice on the rows of V: basis (k, P, n), the
    diagonals and both off-diagonals of H, the residual and the lengths."""
    length0 = torch.linalg.vector_norm(V, dim=1)
    v, w = V / length0[:, None], V
    Q, diag, upper, lower = [], [], [], []
    for j in range(k):
        if j:
            length = torch.linalg.vector_norm(w, dim=1)
            lower.append(length)
            v = w / length[:, None]
        Q.append(v)
        B = torch.stack(Q, dim=1)  # P, j + 1, n
        w = matvec(v)
        h = (B @ w[:, :, None])[:, :, 0]
        diag.append(h[:, j])
        if j:
            upper.append(h[:, j - 1])
        w = w - (h[:, None, :] @ B)[:, 0]
        w = w - ((B @ w[:, :, None]).transpose(1, 2) @ B)[:, 0]
    empty = V.new_zeros((V.shape[0], 0))
    off = 0.5 * (torch.stack(upper, 1) + torch.stack(lower, 1)) if k > 1 else empty
    return torch.stack(Q, dim=1), torch.stack(diag, 1), off, w, length0


def _tridiagonal(diag, off):
    return torch.diag_embed(diag) + torch.diag_embed(off, 1) + torch.diag_embed(off, -1)


def _logdet64(diag, off, length0):
    theta, U = torch.linalg.eigh(_tridiagonal(diag, off).cpu())
    per_probe = length0**2 * (U[:, 0, :] ** 2 * torch.log(theta)).sum(1).to(length0.device)
    return per_probe


class _KernelMatvec(torch.autograd.Function):
    """``v -> K v`` with the cotangents of v and the noise."""

    @staticmethod
    def forward(ctx, K, v, noise):
        ctx.save_for_backward(K, v)
        return v @ K

    @staticmethod
    def backward(ctx, g):
        K, v = ctx.saved_tensors
        return None, g @ K, (g * v).sum()


def exact(case, seed):
    s = _inputs(case, seed)
    call, n = case["call"], case["n"]
    f64 = torch.float64
    if call == "cg":
        K = _kernel64(s["X"], LENGTHSCALE, NOISE)
        L = torch.linalg.cholesky(K)
        return torch.cholesky_solve(s["y"].to(f64)[:, None], L)[:, 0]
    if call == "matvec":
        V = s["V"].to(f64)
        if case["form"] == "rbf":
            return V @ _kernel64(s["X"], LENGTHSCALE, NOISE)
        return V @ s["A"].to(f64)
    k = case["k"]
    if call == "tridiag":
        A = s["A"].to(f64)
        Q, diag, off, w, length0 = _arnoldi64(lambda v: v @ A, s["V"].to(f64), k)
        return dict(Q=Q, T=_tridiagonal(diag, off), residual=w, length=length0)
    if call == "vjp":
        A = s["A"].to(f64).requires_grad_()
        V = s["V"].to(f64).requires_grad_()
        # (v A^T)_i = sum_m A_im v_m: the cotangent of A is sum lambda q^T
        _, diag, off, _, _ = _arnoldi64(lambda v: v @ A.T, V, k)
        T = _tridiagonal(diag, off)
        dV, dA = torch.autograd.grad(T, (V, A), s["G"].to(f64))
        return dict(T=T.detach(), dV=dV, dA=dA)
    Z = s["Z"].to(f64)
    K = _kernel64(s["X"], LENGTHSCALE, NOISE)
    if not case["grad"]:
        _, diag, off, _, length0 = _arnoldi64(lambda v: v @ K, Z, k)
        per_probe = _logdet64(diag, off, length0)
        return dict(per_probe=per_probe, mean=per_probe.mean())
    s2 = torch.tensor(NOISE, dtype=f64, device="cuda", requires_grad=True)
    _, diag, off, _, length0 = _arnoldi64(lambda v: _KernelMatvec.apply(K, v, s2), Z, k)
    per_probe = _logdet64(diag, off, length0)
    (ds2,) = torch.autograd.grad(per_probe.mean(), (s2,))
    # no value for d/d lengthscale: its terms cancel, and what the BF16 operator's own
    # representation leaves of the sum is not near the exact kernel's
    return dict(per_probe=per_probe.detach(), mean=per_probe.mean().detach(), dlengthscale=None,
                dnoise=ds2)
