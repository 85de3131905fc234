"""GPU tests of the products with blocks of right-hand sides (libmpchol through
the C ABI) at the edges of their tiles, chunks and passes."""
import numpy as np
import pytest
import torch

from cholesky_gpu_amd import _lib as L
from cholesky_gpu_amd import solver as S

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("n", [1, 63, 65, 257, 1000, 4609, 14337])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 16, 21])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_symmetric_product(handle, n, nrhs, dtype):
    """The operator's product A X, read off the true residual of a PCG that
    starts at X and takes no step (B the exact product to FP64, L = I): an
    FP64 sum of n exact products is within n u |A| |X| of it, and B too."""
    say("product", n, nrhs, dtype)
    if n > 10000 and (nrhs in (2, 3, 21) or dtype is torch.float64):
        pytest.skip("one large size per kernel is enough")
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn(n, n, generator=g, device="cuda", dtype=torch.float32).to(dtype)
    A = torch.tril(A) + torch.tril(A, -1).T.contiguous()
    X = torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64)
    Xt = X.T.contiguous()
    rows = [A[r:r + 2048].to(torch.float64) for r in range(0, n, 2048)]
    B = torch.cat([R @ Xt for R in rows]).T.contiguous()
    mag = torch.cat([R.abs() @ Xt.abs() for R in rows]).T
    bound = float((2 * n * 2.0 ** -53 * mag.norm(dim=1) / B.norm(dim=1)).max())
    eye = torch.eye(n, device="cuda", dtype=torch.float32)
    f = S.pcg if dtype is torch.float32 else S.pcg64
    _, pi, _ = f(handle, A, eye, B, nb=64, X=X.clone(), opts=S.pcg_opts(x0_mode=2, maxit=0))
    assert pi.relres <= bound, (pi.relres, bound)


@pytest.mark.parametrize("n", [65, 256, 1000, 2049, 4200, 8300])
@pytest.mark.parametrize("nrhs", [1, 4, 5, 16, 21])
def test_apply_precond_blocks(handle, n, nrhs):
    """z = (L L^T)^-1 r for the sizes and passes of the blocked sweeps against
    FP64 triangular solves with the same L (diagonally dominant, cond <= 3, so
    that the FP32 block inverses are within a few hundred u32 of exact)."""
    say("apply_precond", n, nrhs)
    g = torch.Generator(device="cuda").manual_seed(n + nrhs)
    T = torch.randn(n, n, generator=g, device="cuda") * (0.25 / n ** 0.5)
    T = torch.triu(T, 1) + torch.eye(n, device="cuda")            # tensor = L^T
    T = T + torch.tril(torch.full_like(T, float("nan")), -1)      # A's upper part is not read
    R = torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64)
    Z = S.apply_precond(handle, T.contiguous(), R)
    L64 = torch.triu(T).nan_to_num(0.0).to(torch.float64).T.contiguous()
    Y = torch.linalg.solve_triangular(L64, R.T.contiguous(), upper=False)
    X = torch.linalg.solve_triangular(L64.T.contiguous(), Y, upper=True).T
    assert float((Z - X).norm() / X.norm()) < 256 * 2.0 ** -24


@pytest.mark.parametrize("n", [1, 127, 255, 257, 2047, 2050, 2051, 2052, 3073, 4097, 5121])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 6])
def test_apply_precond_edges(handle, n, nrhs):
    """The sweeps where a column ends: one to four rows below a big block, one
    past 1024 (the backward products' step), pieces of 256 that are not full,
    last row blocks of 1 to 63 rows.  Tolerance as above."""
    test_apply_precond_blocks(handle, n, nrhs)


@pytest.mark.parametrize("n,nb", [(300, 64), (500, 64), (512, 128), (513, 256), (777, 128), (1100, 128),
                                  (2047, 256), (2048, 128), (2500, 256), (3001, 256), (3600, 128)])
def test_inverses_built_in_stages(handle, n, nb):
    """The last big block's inverse built in stages during the factor (half,
    three quarters, the end; whole and ragged blocks) is the one built at once
    from a finished factor: the solutions agree bit for bit."""
    say("staged inverses", n, nb)
    A, _ = S.matgen_householder(handle, n, cond=1e3, lam_max=1e3, seed=n)
    B = torch.from_numpy(np.random.default_rng(n).standard_normal((2, n))).cuda()
    fo = S.factor_opts(nb=nb, update_prec=L.PREC_FP32, fallback=0)
    po = S.pcg_opts(tol=1e-10, maxit=100)
    X1, _, pi1, rc1 = S.precond_cg(handle, A, B, fo, po)
    Lf = A.clone()
    rc, _, _, _ = S.factor(handle, Lf, fo)
    X2, pi2, rc2 = S.pcg(handle, A, Lf, B, nb=nb, opts=po)
    assert rc == 0 and rc1 == 0 and rc2 == 0 and pi1.iters == pi2.iters
    assert torch.equal(X1, X2)


@pytest.mark.parametrize("n", [1, 63, 65, 130, 777, 4609])
@pytest.mark.parametrize("nrhs", [4, 5, 16, 21])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_product_reads_upper_triangle(handle, n, nrhs, dtype):
    """The operator's product takes A from its upper triangle (column-major) for
    any number of right-hand sides: with NaN below the diagonal the residual is,
    bit for bit, that of the full matrix."""
    say("upper triangle", n, nrhs, dtype)
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn(n, n, generator=g, device="cuda", dtype=torch.float32).to(dtype)
    A = torch.tril(A) + torch.tril(A, -1).T.contiguous()
    half = torch.tril(A) + torch.triu(torch.full_like(A, float("nan")), 1)   # tensor = transpose
    X = torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64)
    B = torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64)
    eye = torch.eye(n, device="cuda", dtype=torch.float32)
    f = S.pcg if dtype is torch.float32 else S.pcg64
    res = [f(handle, M.contiguous(), eye, B, nb=64, X=X.clone(),
             opts=S.pcg_opts(x0_mode=2, maxit=0))[1].relres for M in (A, half)]
    assert res[0] == res[1], res


@pytest.mark.parametrize("n", [63, 256, 257, 2100, 4500])
@pytest.mark.parametrize("nrhs", [6, 33, 64, 65, 70])
def test_apply_precond_many(handle, n, nrhs):
    """More right-hand sides than one product takes and than one pass takes, by
    column dots (up to 256 rows) and on the matrix cores.  Tolerance as above."""
    test_apply_precond_blocks(handle, n, nrhs)
