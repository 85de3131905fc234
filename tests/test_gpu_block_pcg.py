"""Block PCG's small kernels (Gram matrix, s x s solve, block update) at the
edges of their splits: rows that end inside a wave's 64 and a workgroup's 256,
more than 32 workgroups' worth of rows, 1, 2, 15 and 16 columns."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholesky_gpu_amd import solver as S  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [48, 63, 65, 256, 257, 8191, 8193])
@pytest.mark.parametrize("s", [1, 2, 15, 16])
def test_three_eigenvalues(handle, n, s):
    """A diagonal matrix with three distinct eigenvalues and the identity as
    preconditioner: CG ends after three steps in exact arithmetic (fewer where
    s columns span more), with x = b / lambda; cond(A) = 4, so the stopping rule
    ||r|| <= 1e-12 ||b|| bounds the error by 4e-12 of ||x||."""
    print("[case]", n, s, flush=True)
    lam = torch.tensor([1.0, 2.0, 4.0]).repeat(n // 3 + 1)[:n].cuda()
    B = torch.from_numpy(np.random.default_rng(n + s).standard_normal((s, n))).cuda()
    X, pi, rc = S.block_pcg(handle, torch.diag(lam).contiguous(), torch.eye(n, device="cuda"), B, nb=64,
                            opts=S.pcg_opts(tol=1e-12, maxit=50, x0_mode=1))
    assert rc == 0 and 0 < pi.iters <= 4, (rc, pi.iters)
    want = B / lam.to(torch.float64)[None, :]
    err = (X - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= 4e-12, float(err.max())


@pytest.mark.parametrize("n", [1, 1023, 8193, 16384, 16385])
@pytest.mark.parametrize("s", [1, 3])
def test_dots_where_they_split(handle, n, s):
    """Independent PCGs on the same kind of matrix at the sizes where a dot
    takes a second batch of rows and a second launch: same bounds as above."""
    print("[case]", n, s, flush=True)
    lam = torch.tensor([1.0, 2.0, 4.0]).repeat(n // 3 + 1)[:n].cuda()
    B = torch.from_numpy(np.random.default_rng(n + s).standard_normal((s, n))).cuda()
    X, pi, rc = S.pcg(handle, torch.diag(lam).contiguous(), torch.eye(n, device="cuda"), B, nb=64,
                      opts=S.pcg_opts(tol=1e-12, maxit=50, x0_mode=1))
    assert rc == 0 and 0 < pi.iters <= 4, (rc, pi.iters)
    want = B / lam.to(torch.float64)[None, :]
    err = (X - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= 4e-12, float(err.max())
