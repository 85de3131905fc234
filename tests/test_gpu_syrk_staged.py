"""GPU tests of the staged update kernels (libmpchol through the C ABI) at
the edges of their tiles and K chunks."""
import numpy as np
import pytest
import torch

from cholesky_gpu_amd import _lib as L
from cholesky_gpu_amd import solver as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(1, 64), (63, 64), (128, 192), (129, 64), (257, 320), (700, 256)])
@pytest.mark.parametrize("first", [L.PREC_FP32, L.PREC_BF16, L.PREC_FP16, L.PREC_E4M3])
@pytest.mark.parametrize("other", [L.PREC_FP32, L.PREC_E4M3, L.PREC_MXE5M2, L.PREC_BF16, L.PREC_FP16])
def test_staged_updates(handle, oracle, m, k, first, other):
    """C -= Q Q^T with tiles of `first` and `other` alternating: every element
    within k u32 of the FP64 result, relative to |C| + |Q| |Q|^T (exact
    products, FP32 sums; pairs of two 8-bit tiles, 1e-4 as measured for the
    8-bit op).  Nothing above the diagonal is written."""
    print("[case]", m, k, L.PREC_NAMES[first], L.PREC_NAMES[other], flush=True)
    if {first, other} & {L.PREC_FP16} and {first, other} - {L.PREC_FP16, L.PREC_FP32}:
        pytest.skip("FP16 is combined with FP32 only")
    rng = np.random.default_rng(m + k)
    P = rng.standard_normal((m, k)).astype(np.float32)
    Cm = rng.standard_normal((m, m)).astype(np.float32)
    nt = (m + 127) // 128
    precs = [first if t % 2 == 0 else other for t in range(nt)]
    pay, sc, pt = S.quantize_panel(handle, torch.from_numpy(P.T.copy()).cuda(), precs, 128)
    deq = oracle.quantize_panel(P, precs, 128)[2].astype(np.float64)
    Cd = torch.from_numpy(Cm.T.copy()).cuda()
    S.syrk(handle, Cd, pay, sc, k, 128, pt)
    got = Cd.cpu().numpy().T
    ref = Cm - deq @ deq.T
    err = np.abs(got - ref) / (np.abs(Cm) + np.abs(deq) @ np.abs(deq).T)
    low8 = np.repeat([p >= L.PREC_E5M2 for p in precs], 128)[:m]
    pair8 = low8[:, None] & low8[None, :]
    low = np.tril(np.ones((m, m), bool))
    assert err[low & ~pair8].max(initial=0.0) <= k * 2.0 ** -24
    assert err[low & pair8].max(initial=0.0) < 1e-4
    assert np.array_equal(np.triu(got, 1), np.triu(Cm, 1))


@pytest.mark.parametrize("n", [1024, 1280, 1600, 2304, 2816])
@pytest.mark.parametrize("prec", [L.PREC_BF16, L.PREC_MXE4M3])
def test_factor_group_pairs(handle, n, prec):
    """Two-group far updates (4 to 11 block columns of 256: groups without,
    with one and with several pairs, full and partial last ones): the backward
    error of the factor is that of the per-panel updates (agg_panels = 1) up
    to 10 %, and two runs agree bit for bit."""
    print("[case]", n, L.PREC_NAMES[prec], flush=True)
    A, _ = S.matgen_householder(handle, n, cond=20.0, lam_max=20.0, seed=n)
    err, outs = {}, []
    for agg in (1, 2, 2):
        T = A.clone()
        rc, _, _, _ = S.factor(handle, T, S.factor_opts(nb=256, update_prec=prec, ladder=(prec,),
                                                        fallback=0, agg_panels=agg))
        assert rc == 0
        L64 = torch.triu(T).to(torch.float64).T.contiguous()
        err[agg] = float((L64 @ L64.T.contiguous() - A.to(torch.float64)).norm() / A.to(torch.float64).norm())
        outs.append(T)
    assert torch.equal(outs[1], outs[2])
    assert err[2] <= 1.1 * err[1], err


@pytest.mark.parametrize("n,nb", [(65, 64), (2303, 128), (4096, 256), (4097, 256), (4352, 256),
                                  (5000, 128), (5120, 256), (4480, 64)])
@pytest.mark.parametrize("prec", [L.PREC_FP32, L.PREC_SWITCH])
def test_factor_one_stream_tail(handle, n, nb, prec):
    """The last 4096 columns on one stream (whole factors and the ends of
    larger ones, from a group's start on): the backward error is that of the
    phase-by-phase schedule up to 10 %, and two runs agree bit for bit."""
    print("[case]", n, nb, prec, flush=True)
    A, _ = S.matgen_householder(handle, n, cond=20.0, lam_max=20.0, seed=n)
    err, outs = [], []
    for prof in (1, 0, 0):
        T = A.clone()
        rc, _, _, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=prec, eps_prime=0.125,
                                                        ladder=(L.PREC_E4M3, L.PREC_FP32),
                                                        fallback=0, profile=prof))
        assert rc == 0
        L64 = torch.triu(T).to(torch.float64).T.contiguous()
        err.append(float((L64 @ L64.T.contiguous() - A.to(torch.float64)).norm() / A.to(torch.float64).norm()))
        outs.append(T)
    assert torch.equal(outs[1], outs[2])
    assert err[1] <= 1.1 * err[0], err


@pytest.mark.parametrize("n,nb", [(130, 64), (517, 128), (1031, 256), (4101, 256)])
def test_factor_restored_after_breakdown(handle, n, nb):
    """E4M3 updates break down on a kernel matrix with eigenvalues down to
    1e-5; the fallback restores A (its lower triangle, 16-byte pieces, ragged
    ends) and ends with FP32 updates: the outcome is that of an FP32 run on A,
    the same factor bit for bit or (4101 points: cond 1e8) the same failing
    column, and the strict upper triangle is A's."""
    print("[case]", n, nb, flush=True)
    x = torch.linspace(0, 8, n, device="cuda")
    A = torch.exp(-0.5 * (x[:, None] - x[None, :]) ** 2) + 1e-5 * torch.eye(n, device="cuda")
    T1, T2 = A.clone(), A.clone()
    rc1, fi, _, _ = S.factor(handle, T1, S.factor_opts(nb=nb, update_prec=L.PREC_E4M3, fallback=1))
    rc2, _, _, _ = S.factor(handle, T2, S.factor_opts(nb=nb, update_prec=L.PREC_FP32, fallback=0))
    assert fi.retries == 1 and rc1 == rc2
    assert rc1 or torch.equal(T1, T2)
    assert torch.equal(torch.tril(T1, -1), torch.tril(A, -1))      # (the tensor is the transpose)


@pytest.mark.parametrize("n,nb", [(8447, 256), (8448, 256), (8750, 256), (4225, 128), (5000, 128)])
@pytest.mark.parametrize("prec", [L.PREC_BF16, L.PREC_MXE4M3])
def test_factor_group_pairs_large(handle, n, nb, prec):
    """The sizes from which two groups' panels go into one far update, before
    the one-stream tail: the backward error of the factor is that of the
    per-panel updates (agg_panels = 1) up to 10 %, and two runs agree bit for
    bit."""
    print("[case]", n, nb, L.PREC_NAMES[prec], flush=True)
    A, _ = S.matgen_householder(handle, n, cond=20.0, lam_max=20.0, seed=n)
    err, outs = {}, []
    for agg in (1, 2, 2):
        T = A.clone()
        rc, _, _, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=prec, ladder=(prec,),
                                                        fallback=0, agg_panels=agg))
        assert rc == 0
        L64 = torch.triu(T).to(torch.float64).T.contiguous()
        err[agg] = float((L64 @ L64.T.contiguous() - A.to(torch.float64)).norm()
                         / A.to(torch.float64).norm())
        outs.append(T)
    print("backward errors", err, flush=True)
    assert err[2] <= 1.1 * err[1]
    assert torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("n,nb", [(15359, 256), (15360, 256), (16001, 256), (15487, 128)])
@pytest.mark.parametrize("prec", [L.PREC_BF16, L.PREC_SWITCH])
def test_factor_group_quads(handle, n, nb, prec):
    """The size from which four groups' panels go into one far update: the
    backward error of the factor, on random vectors, is that of the per-panel
    updates (agg_panels = 1) up to 10 %, two runs agree bit for bit, and the
    solve that factors a partly copied matrix equals factor and solve."""
    print("[case]", n, nb, prec, flush=True)
    A, _ = S.matgen_householder(handle, n, cond=20.0, lam_max=20.0, seed=n)
    V = torch.randn(n, 8, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda()
    ladder = (L.PREC_E4M3, L.PREC_FP32) if prec == L.PREC_SWITCH else (prec,)

    def product(M):                  # M V by row blocks, in FP64
        return torch.cat([M[r:r + 2048].to(torch.float64) @ V for r in range(0, n, 2048)])

    ref = product(A)
    err, outs = {}, []
    for agg in (1, 2, 2):
        T = A.clone()
        fo = S.factor_opts(nb=nb, update_prec=prec, ladder=ladder, eps_prime=0.125, fallback=0,
                           agg_panels=agg)
        rc, _, _, _ = S.factor(handle, T, fo)
        assert rc == 0
        Lt = torch.triu(T)
        w = product(Lt)
        y = sum(Lt[r:r + 2048].to(torch.float64).T.contiguous() @ w[r:r + 2048]
                for r in range(0, n, 2048))
        err[agg] = float((y - ref).norm() / ref.norm())
        outs.append(T)
    print("backward errors", err, flush=True)
    assert err[2] <= 1.1 * err[1]
    assert torch.equal(outs[1], outs[2])
    B = V[:, :1].T.contiguous()
    po = S.pcg_opts(tol=1e-10)
    # (first the solve with the handle's last factor, whose 32x32 inverses it
    # still has; for another factor it computes them again, in other bits)
    X2 = S.pcg(handle, A, outs[2], B, nb=nb, opts=po)[0]
    X1 = S.precond_cg(handle, A, B, fo, po)[0]
    assert torch.equal(X1, X2)


@pytest.mark.parametrize("m,k", [(129, 64), (257, 192), (640, 256)])
def test_staged_bf16_with_fp16(handle, oracle, m, k):
    """BF16 and FP16 tiles alternating: a pair of one of each is computed in
    BF16, the FP16 values cut to their leading 8 bits, a pair of two FP16 tiles
    from the values themselves: every element within k u32 of the FP64 result on
    these operands, relative to |C| + |Q| |Q|^T."""
    print("[case]", m, k, flush=True)
    rng = np.random.default_rng(m + k)
    P = rng.standard_normal((m, k)).astype(np.float32)
    Cm = rng.standard_normal((m, m)).astype(np.float32)
    precs = [L.PREC_FP16 if t % 2 else L.PREC_BF16 for t in range((m + 127) // 128)]
    pay, sc, pt = S.quantize_panel(handle, torch.from_numpy(P.T.copy()).cuda(), precs, 128)
    Q = np.ascontiguousarray(oracle.quantize_panel(P, precs, 128)[2], dtype=np.float32)
    cut = (Q.view(np.uint32) & np.uint32(0xffff0000)).view(np.float32).astype(np.float64)
    Q = Q.astype(np.float64)
    Cd = torch.from_numpy(Cm.T.copy()).cuda()
    S.syrk(handle, Cd, pay, sc, k, 128, pt)
    got = Cd.cpu().numpy().T
    half = np.repeat([p == L.PREC_FP16 for p in precs], 128)[:m]
    ref = Cm - np.where(half[:, None] & half[None, :], Q @ Q.T, cut @ cut.T)
    err = np.abs(got - ref) / (np.abs(Cm) + np.abs(Q) @ np.abs(Q).T)
    assert err[np.tril(np.ones((m, m), bool))].max() <= k * 2.0 ** -24
    assert np.array_equal(np.triu(got, 1), np.triu(Cm, 1))


@pytest.mark.parametrize("n,nb", [(640, 128), (1111, 128), (1500, 256), (4096, 256), (4864, 128), (6000, 256)])
@pytest.mark.parametrize("agg", [1, 2, 3, 4])
def test_factor_group_sums(handle, n, nb, agg):
    """The products of a group's panels are added before C takes them, in whole
    factors of any size and in the last columns of larger ones.  I in front, then
    rows of constant b: a panel adds nb b^2, less than half the spacing of the
    floats below 1, to every entry of C.  Entries of C that are 1 stay 1 when
    panels are subtracted one by one and become fl(1 - agg nb b^2), one or two
    spacings less, in groups; divided by a pivot of 4 they come out halved.  All
    of it is exact in FP32."""
    print("[case]", n, nb, agg, flush=True)
    b = 0.875 * 2.0 ** -16 if nb == 128 else 1.25 * 2.0 ** -17
    last = max(k for k in range(1, 200) if k * agg * nb + nb // 2 < n)    # the last group with rows below
    for group in {1, last}:
        e, p = group * agg * nb, (group - 1) * agg * nb
        T = torch.eye(n, device="cuda")
        T[p:e, e:] = b                           # the tensor is the transpose
        T[torch.arange(e, n), torch.arange(e, n)] = 4.0
        rows = sorted({e + 1, (e + n) // 2, n - 1} - {e})
        T[e, rows] = 1.0
        T = torch.triu(T) + torch.triu(T, 1).T.contiguous()
        rc, _, _, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=L.PREC_FP32, fallback=0,
                                                        agg_panels=agg))
        assert rc == 0
        want = 0.5 * float(np.float32(1.0 - agg * nb * b * b))
        got = T[e, rows].cpu().numpy()
        assert (got == want).all(), (group, rows, got - 0.5, want - 0.5)


@pytest.mark.parametrize("n,nb,ladder", [(15360, 256, (L.PREC_FP32,)), (8500, 256, (L.PREC_E4M3, L.PREC_FP32)),
                                         (15400, 256, (L.PREC_E4M3, L.PREC_FP32)),
                                         (15500, 128, (L.PREC_E4M3, L.PREC_FP32))])
def test_factor_fp32_sums_per_group(handle, n, nb, ladder):
    """A switching factor that keeps every tile FP32, with a ladder that has
    nothing else or on a matrix whose rows grow by sqrt(2) per 128 (so that no
    tile is small beside the first pivots: the first panel's next tile has row
    sums of squares of about a tenth of them, E4M3 takes 1/16 at this eps'), is
    the fixed FP32 factor bit for bit: updates with several groups' panels add
    FP32 products group by group."""
    print("[case]", n, nb, ladder, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    G = torch.randn(n, n // 32, generator=g, device="cuda")
    d = torch.exp2(torch.arange(n, device="cuda").div(128, rounding_mode="floor") / 2 - 30)
    A = G @ G.T / (n // 32) + torch.eye(n, device="cuda")
    A = torch.tril(A) + torch.tril(A, -1).T
    A = (A * d[:, None] * d[None, :]).contiguous()
    outs = []
    for prec, lad in ((L.PREC_FP32, (L.PREC_FP32,)), (L.PREC_SWITCH, ladder)):
        T = A.clone()
        rc, _, mp, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=prec, ladder=lad,
                                                         eps_prime=1 / 256, fallback=0), want_map=True)
        assert rc == 0
        low = np.tril(np.ones(tuple(mp.shape), bool), -1)
        assert (mp.cpu().numpy().T[low] == L.PREC_FP32).all()
        outs.append(T)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("n,nb", [(1111, 128), (1500, 256), (4000, 128), (4096, 256), (6000, 256)])
@pytest.mark.parametrize("agg", [2, 3, 4])
def test_factor_panel_sums(handle, n, nb, agg):
    """Each panel's products are added apart from the other panels of the group:
    where the group's first panel gives 1 and every product of the others is
    2^-25, a quarter of the spacing of the floats there, one chain would stay at
    1; apart they give 1 + (agg - 1) nb 2^-25 exactly.  The pivot beside it is 4
    exactly when its sum is right, and halves the entries."""
    print("[case]", n, nb, agg, flush=True)
    last = max(k for k in range(1, 200) if k * agg * nb + nb // 2 < n)    # the last group with rows below
    for group in {1, last}:
        e, p = group * agg * nb, (group - 1) * agg * nb
        T = torch.eye(n, device="cuda")
        T[torch.arange(e, n), torch.arange(e, n)] = 8.0
        rows = sorted({e + 1, (e + n) // 2, n - 1} - {e})
        small = (agg - 1) * nb * 2.0 ** -25
        T[p, e] = 1.0                            # (the tensor is the transpose)
        T[p, rows] = 1.0
        T[p + nb:e, e] = 2.0 ** -13
        T[p + nb:e, rows] = 2.0 ** -12
        T[e, e] = 5.0 + 0.5 * small
        T[e, rows] = 2.0
        T = torch.triu(T) + torch.triu(T, 1).T.contiguous()
        rc, _, _, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=L.PREC_FP32, fallback=0,
                                                        agg_panels=agg))
        assert rc == 0
        assert float(T[e, e]) == 2.0
        got = T[e, rows].cpu().numpy()
        assert (got == 0.5 * (1.0 - small)).all(), (group, rows, got - 0.5, -0.5 * small)
