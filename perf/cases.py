"""Performance cases of cholesky_gpu_amd: what a program asks of it, through
its public entry points (cholesky_gpu_amd.solver), from the smallest systems to
a 60000-point kernel matrix.

    listed()             the cases that are always measured
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the matrix, right-hand sides, options and handle that
                         a program holds before the call, on the GPU
    run(state)           one pass through the public entry points
    work(case)           bytes and flops that no implementation can avoid
    exact(case, seed)    what run returns, computed in FP64 with plain torch

A case is a dict of plain values:
    op      "solve"   factor + PCG from A (precond_cg)
            "resolve" PCG with a factor that the program kept (pcg)
            "block"   block PCG with a kept factor (block_pcg)
            "grad"    differentiable solve, forward and backward (spd_solve)
            "factor"  the mixed-precision factor itself (factor)
            "gp"      GP loss and all its gradients (gp_loss_grad)
    matrix  "hh"      conditioned SPD, H Lambda H^T with log-spaced Lambda
            "rbf"     RBF kernel of N(0, I_d) points plus a nugget
            "image"   RBF kernel of image-shaped points (d coordinates, 80 %
                      zero), lengthscale = median distance of a subsample
    n, nb, nrhs, d    sizes; nb is the factor's block
    update            "switch" over `ladder`, or one format for every tile
"""
import math

import numpy as np
import torch

from cholesky_gpu_amd import _lib as L
from cholesky_gpu_amd import solver as S

FORMATS = {"fp32": L.PREC_FP32, "bf16": L.PREC_BF16, "fp16": L.PREC_FP16, "e5m2": L.PREC_E5M2,
           "e4m3": L.PREC_E4M3, "mxe4m3": L.PREC_MXE4M3, "mxe5m2": L.PREC_MXE5M2}
# every tolerance is the 1e-10 FP64 true residual that the solver is used at
# (1e-11 for the GP gradient, whose entries are wanted to 1e-6 and better)
TOL, TOL_GP = 1e-10, 1e-11
ROWS = 4096          # rows of a matrix made (or factored in FP64) at a time


def _case(name, op, matrix, n, nb=256, nrhs=1, update="switch", ladder="e4m3,fp32", eps=0.125, d=16):
    c = {"op": op, "matrix": matrix, "n": n, "nb": nb, "nrhs": nrhs, "update": update,
         "ladder": ladder, "eps": eps, "d": d}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small kernel system solved once: launches and synchronisations
        _case("solve-rbf-500", "solve", "rbf", 500, nb=64, d=8),
        # 2048 points, block 128, FP16 update: the small kernel workload
        _case("solve-rbf-2048-fp16", "solve", "rbf", 2048, nb=128, update="fp16", ladder="fp16"),
        # an ordinary system of a size that is no multiple of anything, with a
        # few right-hand sides and the default switching ladder
        _case("solve-hh-3001-r4", "solve", "hh", 3001, nrhs=4, eps=0.25),
        # the headline solve: n = 16384, cond 1e6, E4M3 with FP32 switching
        _case("solve-hh-16384-e4m3", "solve", "hh", 16384),
        # the same solve with FP32 updates, for users who want a plain factor
        _case("solve-hh-16384-fp32", "solve", "hh", 16384, update="fp32", ladder="fp32"),
        # the largest: 60000 image-shaped points, MXFP8 with FP32 switching
        _case("solve-image-60000-r4", "solve", "image", 60000, nrhs=4, ladder="mxe4m3,fp32", d=784),
        # one more right-hand side on a factor kept from before (time
        # stepping, a new target vector); odd size, unaligned columns
        _case("resolve-hh-9001", "resolve", "hh", 9001),
        # sixteen related right-hand sides solved together
        _case("block-hh-6000-r16", "block", "hh", 6000, nrhs=16),
        # training through the solve: the forward PCG and the adjoint one,
        # with the four-format ladder
        _case("grad-hh-8192-r16", "grad", "hh", 8192, nrhs=16, ladder="e5m2,mxe4m3,bf16,fp32"),
        # the factor for its own sake (a caller's own preconditioner)
        _case("factor-hh-4000-fp32", "factor", "hh", 4000, nb=128, update="fp32", ladder="fp32"),
        # GP hyperparameter step at full size: 8192 points, ARD, 32 probes
        _case("gp-8192-ard", "gp", "rbf", 8192, nrhs=32, d=8, eps=0.25),
        # and a small one, as in a hyperparameter search
        _case("gp-777-ard", "gp", "rbf", 777, nb=128, nrhs=8, d=4, eps=0.25),
    ]


def _size(rng, lo, hi):
    """log-uniform over [lo, hi]; one in three a multiple of 256 (of 64 below 1024)"""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 1 / 3:
        q = 256 if n >= 1024 else 64
        n = max(q, n // q * q)
    return min(max(n, lo), hi)


def draw(rng):
    op = rng.choice(("solve", "solve", "solve", "resolve", "block", "grad", "factor", "gp"))
    nb = rng.choice((64, 128, 256, 256))
    if op == "gp":
        return _case(None, op, "rbf", _size(rng, 300, 8192), nb=nb, nrhs=rng.choice((4, 8, 16, 32)),
                     d=rng.randint(2, 8), eps=0.25)
    if op == "factor":
        update = rng.choice(("fp32", "fp32", "bf16"))
        return _case(None, op, "hh" if update == "fp32" else "rbf", _size(rng, 300, 12000), nb=nb,
                     update=update, ladder=update)
    if op != "solve":
        return _case(None, op, "hh", _size(rng, 500, 12000), nb=nb,
                     nrhs=rng.randint(2, 16) if op == "block" else rng.choice((1, 2, 3, 5, 8, 16)),
                     ladder=rng.choice(("e4m3,fp32", "mxe4m3,fp32", "e5m2,mxe4m3,bf16,fp32")))
    matrix = rng.choice(("hh", "hh", "rbf", "image"))
    update, ladder = "switch", rng.choice(("e4m3,fp32", "mxe4m3,fp32", "e4m3,bf16,fp32"))
    if rng.random() < 0.4:
        update = ladder = "fp32" if matrix == "hh" else rng.choice(("fp32", "fp16"))
    return _case(None, op, matrix, _size(rng, 300, 30000), nb=nb, nrhs=rng.choice((1, 1, 2, 4, 7, 16)),
                 update=update, ladder=ladder, d=784 if matrix == "image" else rng.randint(4, 16))


# ---------------------------------------------------------------- inputs
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _by_rows(n, rows, device):
    """FP32 n x n, exactly symmetric, from rows(r0, r1) = its FP64 rows r0..r1
    and columns 0..r1."""
    A = torch.empty(n, n, dtype=torch.float32, device=device)
    for r0 in range(0, n, ROWS):
        r1 = min(n, r0 + ROWS)
        P = rows(r0, r1).to(torch.float32)
        D = torch.tril(P[:, r0:])
        P[:, r0:] = D + torch.tril(D, -1).T
        A[r0:r1, :r1] = P
        A[:r0, r0:r1] = P[:, :r0].T
    return A


def _householder(n, g, device, cond=1e6, lam_max=1e6, reflectors=4):
    """H Lambda H^T, Lambda log-spaced up to lam_max: reflecting A by w gives
    A - w v^T - v w^T with v = 2 (A w - (w^T A w) w)."""
    lam = torch.logspace(math.log10(lam_max / cond), math.log10(lam_max), n, dtype=torch.float64,
                         device=device)
    W = torch.empty(n, 0, dtype=torch.float64, device=device)
    V = torch.empty(n, 0, dtype=torch.float64, device=device)
    for _ in range(reflectors):
        w = torch.randn(n, generator=g, dtype=torch.float64, device=device)
        w /= w.norm()
        Aw = lam * w - W @ (V.T @ w) - V @ (W.T @ w)
        v = 2 * (Aw - (w @ Aw) * w)
        W, V = torch.cat([W, w[:, None]], 1), torch.cat([V, v[:, None]], 1)
    F, G = torch.cat([W, V], 1), torch.cat([V, W], 1)

    def rows(r0, r1):
        P = -(F[r0:r1] @ G[:r1].T.contiguous())
        P[:, r0:].diagonal().add_(lam[r0:r1])
        return P
    return _by_rows(n, rows, device)


def _points(case, g, device):
    n, d = case["n"], case["d"]
    if case["matrix"] == "image":
        X = 1.0 - torch.rand(n, d, generator=g, dtype=torch.float32, device=device)
        return X * (torch.rand(n, d, generator=g, dtype=torch.float32, device=device) >= 0.8)
    return torch.randn(n, d, generator=g, dtype=torch.float32, device=device)


def _kernel(X, ls, nugget, device):
    """exp(-|x - y|^2 / (2 ls^2)) + nugget I; ls one number or one per dimension"""
    Y = X.to(torch.float64) / ls
    q = (Y * Y).sum(1)

    def rows(r0, r1):
        P = Y[r0:r1] @ Y[:r1].T.contiguous()
        P = torch.exp(-0.5 * (q[r0:r1, None] + q[None, :r1] - 2 * P).clamp_(min=0))
        P[:, r0:].diagonal().fill_(1.0 + nugget)
        return P
    return rows


def _inputs(case, seed, device):
    """(A or None, B, points, lengthscales)"""
    g = torch.Generator(device=device).manual_seed(seed)
    n = case["n"]
    if case["op"] == "gp":
        X = _points(case, g, device)
        ls = (0.5 + 1.5 * torch.rand(case["d"], generator=g, dtype=torch.float64, device=device)).cpu().numpy()
        return None, torch.randn(n, generator=g, dtype=torch.float64, device=device), X, ls
    if case["matrix"] == "hh":
        A = _householder(n, g, device)
    else:
        X = _points(case, g, device)
        if case["matrix"] == "image":
            sub = X[torch.randperm(n, generator=g, device=device)[:1024]].to(torch.float64)
            ls, nugget = float(torch.nn.functional.pdist(sub).median()), 1e-3
        else:
            ls, nugget = math.sqrt(case["d"]), 1e-2
        A = _by_rows(n, _kernel(X, ls, nugget, device), device)
    return A, torch.randn(case["nrhs"], n, generator=g, dtype=torch.float64, device=device), None, None


def prepare(case, seed):
    A, B, X, ls = _inputs(case, seed, _device())
    ladder = tuple(FORMATS[f] for f in case["ladder"].split(","))
    update = L.PREC_SWITCH if case["update"] == "switch" else FORMATS[case["update"]]
    fo = S.factor_opts(nb=case["nb"], update_prec=update, ladder=ladder, eps_prime=case["eps"])
    st = {"op": case["op"], "nb": case["nb"], "handle": S.Handle(0), "A": A, "B": B, "fo": fo,
          "po": S.pcg_opts(tol=TOL, maxit=500)}
    if case["op"] in ("resolve", "block", "grad"):
        Lf = A.clone()
        rc, _, _, _ = S.factor(st["handle"], Lf, fo, want_map=False)
        if rc != 0:
            raise RuntimeError(f"the factor broke down in column {rc}")
        st["Lf"] = Lf
    elif case["op"] == "gp":
        st.update(X=X, ls=ls, go=S.gp_opts(n_probes=case["nrhs"], probe_seed=seed, factor=fo,
                                           pcg=S.pcg_opts(tol=TOL_GP, maxit=500)))
    return st


# ---------------------------------------------------------------- one pass
def run(state):
    s, h, op = state, state["handle"], state["op"]
    if op == "solve":
        return S.precond_cg(h, s["A"], s["B"], s["fo"], s["po"])[0]
    if op == "resolve":
        return S.pcg(h, s["A"], s["Lf"], s["B"], nb=s["nb"], opts=s["po"])[0]
    if op == "block":
        return S.block_pcg(h, s["A"], s["Lf"], s["B"], nb=s["nb"], opts=s["po"])[0]
    if op == "factor":
        T = s["A"].clone()               # the factor is made in place
        S.factor(h, T, s["fo"])
        return T
    if op == "grad":
        B = s["B"].detach().requires_grad_(True)
        X = S.spd_solve(B, s["A"], s["Lf"], h, nb=s["nb"], opts=s["po"])
        (0.5 * (B * X).sum()).backward()
        return {"X": X.detach(), "grad_B": B.grad}
    loss, gb, gls, gvar, gnoise, _ = S.gp_loss_grad(h, s["X"], s["ls"], 1.0, 1e-2, s["B"], s["go"])
    return {"loss": loss, "grad_b": gb, "grad_ls": gls, "grad_variance": gvar, "grad_noise": gnoise}


def work(case):
    """A symmetric A is n (n + 1) / 2 FP32 values, and so is a factor; a solve
    from A is one Cholesky and two triangular solves a column, one with a kept
    factor a product with A and two triangular solves.  The GP step: Cholesky,
    the probes' and the target's solves, and the contraction of the weights
    U V^T with the derivatives of every entry."""
    n, r = case["n"], case["nrhs"]
    tri = n * (n + 1) / 2
    if case["op"] == "gp":
        d = case["d"]
        return {"bytes": 4.0 * n * d + 16.0 * n,
                "flops": n ** 3 / 3 + 4.0 * tri * (r + 1) + tri * (4.0 * (r + 1) + 5.0 * d)}
    if case["op"] == "factor":
        return {"bytes": 8.0 * tri, "flops": n ** 3 / 3}
    if case["op"] == "solve":
        return {"bytes": 4.0 * tri + 16.0 * n * r, "flops": n ** 3 / 3 + 4.0 * tri * r}
    passes = 2 if case["op"] == "grad" else 1
    return {"bytes": passes * (8.0 * tri + 16.0 * n * r), "flops": passes * 8.0 * tri * r}


# ---------------------------------------------------------------- FP64 values
def _cholesky(rows, n):
    """Blocks L[i][j] of ROWS of the FP64 Cholesky factor of the symmetric
    matrix whose rows r0..r1, columns 0..r1 are rows(r0, r1)."""
    blk = []
    for r0 in range(0, n, ROWS):
        r1 = min(n, r0 + ROWS)
        P = rows(r0, r1).to(torch.float64)
        own = []
        for j, Lj in enumerate(blk):
            T = P[:, j * ROWS:(j + 1) * ROWS].contiguous()
            for k in range(j):
                T -= own[k] @ Lj[k].T.contiguous()
            own.append(torch.linalg.solve_triangular(Lj[j], T.T.contiguous(), upper=False).T.contiguous())
        T = P[:, r0:].contiguous()
        for k in range(len(own)):
            T -= own[k] @ own[k].T.contiguous()
        blk.append(own + [torch.linalg.cholesky(T)])
    return blk


def _solve(blk, n, B):
    """(L L^T)^-1 B^T, returned like B: (nrhs, n)"""
    Y = [b.T.contiguous() for b in B.split(ROWS, 1)]
    for i, Li in enumerate(blk):
        for k in range(i):
            Y[i] = Y[i] - Li[k] @ Y[k]
        Y[i] = torch.linalg.solve_triangular(Li[i], Y[i], upper=False)
    for i in reversed(range(len(blk))):
        for k in range(i + 1, len(blk)):
            Y[i] = Y[i] - blk[k][i].T.contiguous() @ Y[k]
        Y[i] = torch.linalg.solve_triangular(blk[i][i].T.contiguous(), Y[i], upper=True)
    return torch.cat(Y).T.contiguous()


def _probes(n, nprobe, seed):
    """The Rademacher probes of the GP step: -1 where the first word of
    Philox4x32-10 (counter: index p n + i, stream 3, the tag of the uniform
    generator; key: the seed) is below 2^31, else +1."""
    idx = np.arange(n * nprobe, dtype=np.uint64)
    m32 = np.uint64(0xFFFFFFFF)
    c = [idx & m32, idx >> np.uint64(32), np.full_like(idx, 3), np.full_like(idx, 0x554E4946)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & m32,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & m32]
    return torch.from_numpy(np.where(c[0] < 2 ** 31, -1.0, 1.0).reshape(nprobe, n))


def _exact_gp(case, seed, X, ls, b, device):
    n, P = case["n"], case["nrhs"]
    lst = torch.from_numpy(ls).to(device)
    K = _kernel(X, lst, 0.0, device)(0, n)          # noise-free, rows 0..n in one
    A = K.clone()
    A.diagonal().add_(1e-2)
    blk = _cholesky(lambda r0, r1: A[r0:r1, :r1], n)
    del A
    Z = _probes(n, P, seed).to(device)
    sol = _solve(blk, n, torch.cat([b[None, :], Z]))
    M = (0.5 / P) * (sol[1:].T.contiguous() @ Z) - 0.5 * torch.outer(sol[0], sol[0])
    gnoise = float(M.diagonal().sum())
    M *= K
    Y = X.to(torch.float64) / lst
    gls = [float((M * (Y[:, c, None] - Y[None, :, c]) ** 2).sum() / ls[c]) for c in range(case["d"])]
    # the loss holds the mixed-precision factor's logdet, an estimate: no value
    return {"loss": None, "grad_b": sol[0], "grad_ls": np.array(gls), "grad_variance": float(M.sum()),
            "grad_noise": gnoise}


def exact(case, seed):
    device = _device()
    A, B, X, ls = _inputs(case, seed, device)
    n = case["n"]
    if case["op"] == "gp":
        return _exact_gp(case, seed, X, ls, B, device)
    blk = _cholesky(lambda r0, r1: A[r0:r1, :r1], n)
    if case["op"] == "factor":                       # column-major: the tensor holds L^T
        T = A.to(torch.float64)
        for i, row in enumerate(blk):
            for j, Lij in enumerate(row):
                r, c = slice(i * ROWS, (i + 1) * ROWS), slice(j * ROWS, (j + 1) * ROWS)
                T[c, r] = Lij.T if i != j else torch.triu(Lij.T) + torch.tril(T[c, r], -1)
        return T
    Y = _solve(blk, n, B)
    return {"X": Y, "grad_B": Y} if case["op"] == "grad" else Y
