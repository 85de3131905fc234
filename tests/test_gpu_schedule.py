"""GPU tests of the factor's overlapped schedule (more than 4096 columns: panels,
group columns and far updates on streams of their own), on matrices whose factor
is whole numbers, and of the solve that copies its matrix with the first update."""
import numpy as np
import pytest
import torch

from cholesky_gpu_amd import _lib as L
from cholesky_gpu_amd import solver as S

pytestmark = pytest.mark.gpu

E4, BF, F32, F16 = L.PREC_E4M3, L.PREC_BF16, L.PREC_FP32, L.PREC_FP16
MIXED = (E4, BF, F32)


def whole_factor(n, nb):
    """L (as its transpose) with 8 on the diagonal, zeros elsewhere in the 32 x 32
    diagonal blocks and whole numbers below: a third of the (row tile, panel)
    blocks each 1/16 full of +-1, half full of +-2 and full of +-16.  Every entry
    is a value of every format, every product and sum of the factorisation a
    whole number below 2^24 and every pivot 64: the factor of L L^T is L, whatever
    the formats, the grouping and the order of the updates."""
    g = torch.Generator(device="cuda").manual_seed(n + nb)
    T = torch.zeros(n, n, device="cuda")
    tile = max(nb, 128)
    for j in range(0, n, nb):
        w = min(nb, n - j)
        i = torch.arange(n, device="cuda")
        sign = torch.randint(0, 2, (w, n), generator=g, device="cuda") * 2.0 - 1.0
        u = torch.rand(w, n, generator=g, device="cuda")
        kind = ((i - j - nb).div(tile, rounding_mode="floor") * 7 + j // nb * 3).remainder(3)
        amp = torch.tensor([1.0, 2.0, 16.0], device="cuda")[kind]
        fill = torch.tensor([1 / 16, 0.5, 1.0], device="cuda")[kind]
        inside = i < j + nb                       # the diagonal block: sparse +-1
        amp, fill = torch.where(inside, 1.0, amp), torch.where(inside, 1 / 16, fill)
        block = torch.where(u < fill, sign * amp, 0.0)
        below = i[None, :].div(32, rounding_mode="floor") > (j + torch.arange(w, device="cuda"))[:, None].div(
            32, rounding_mode="floor")
        T[j:j + w] = torch.where(below, block, 0.0)
    T.diagonal().fill_(8.0)
    return T


@pytest.mark.parametrize("n,nb,agg,prec,ladder,rule,eps", [
    # per panel; groups of 2, 3 and 4, whole and ragged at the end
    (4500, 64, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (4353, 256, 1, L.PREC_SWITCH, MIXED, 0, 0.125),
    (5633, 256, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (6401, 256, 3, L.PREC_SWITCH, MIXED, 0, 0.125),
    (7169, 256, 4, L.PREC_SWITCH, MIXED, 0, 0.125),
    (4900, 128, 3, L.PREC_SWITCH, MIXED, 0, 0.125),
    (5250, 128, 4, L.PREC_SWITCH, (L.PREC_MXE5M2, L.PREC_MXE4M3, BF, F32), 0, 0.125),
    (5900, 256, 2, L.PREC_SWITCH, (F16, F32), 0, 0.125),
    (5633, 256, 2, L.PREC_SWITCH, MIXED, L.RULE_FROBENIUS, 0.125),
    (4900, 128, 3, L.PREC_SWITCH, MIXED, L.RULE_FROBENIUS, 0.125),
    (5633, 256, 2, L.PREC_SWITCH, (E4, F32), L.RULE_SCHUR, 0.03),
    # two groups in a far update
    (5377, 128, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (8448, 256, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (9001, 256, 2, L.PREC_SWITCH, (F16, F32), 0, 0.125),
    (9001, 256, 2, E4, (E4,), 0, 0.125),
    # four
    (15360, 256, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (15487, 128, 2, L.PREC_SWITCH, MIXED, 0, 0.125),
    (16001, 256, 2, L.PREC_SWITCH, (F16, F32), 0, 0.125),
    (16001, 256, 2, BF, (BF,), 0, 0.125),
    (16001, 256, 2, F32, (F32,), 0, 0.125),
])
def test_whole_number_factor(handle, n, nb, agg, prec, ladder, rule, eps):
    """The factor is exact, so any update that is missed, done twice, taken from
    the wrong panel, format or copy of C, or not waited for shows as a wrong
    entry; a switching ladder leaves tiles of more than one format."""
    print("[case]", n, nb, agg, prec, ladder, rule, flush=True)
    Lt = whole_factor(n, nb)
    A = torch.empty(n, n, device="cuda")
    for r in range(0, n, 2048):                  # L L^T, exact in FP64 and in FP32
        A[r:r + 2048] = Lt[:, r:r + 2048].to(torch.float64).T.contiguous() @ Lt.to(torch.float64)
    assert float(A.abs().max()) < 2.0 ** 24
    for _ in range(2):
        T = A.clone()
        rc, _, mp, _ = S.factor(handle, T, S.factor_opts(nb=nb, update_prec=prec, ladder=ladder, eps_prime=eps,
                                                         fallback=0, agg_panels=agg, rule=rule), want_map=True)
        assert rc == 0
        low = np.tril(np.ones(tuple(mp.shape), bool), -1)
        kinds = np.unique(mp.cpu().numpy().T[low])
        assert len(kinds) > 1 if prec == L.PREC_SWITCH else list(kinds) == [prec], kinds
        wrong = (torch.triu(T) != Lt).nonzero()
        assert len(wrong) == 0, (len(wrong), wrong[0].tolist(), wrong[-1].tolist())
        assert torch.equal(torch.tril(T, -1), torch.tril(A, -1))


@pytest.mark.parametrize("n,nb,agg,eps,fallback", [(5633, 256, 2, 0.125, 0), (6401, 256, 3, 0.125, 0),
                                                   (7169, 256, 4, 0.125, 0), (5377, 128, 2, 0.125, 0),
                                                   (8600, 256, 2, 0.125, 0), (15400, 256, 2, 0.125, 0),
                                                   (5633, 256, 2, 1e12, 1), (8600, 256, 2, 1e12, 1)])
def test_deferred_copy_overlapped(handle, n, nb, agg, eps, fallback):
    """precond_cg, which copies the first group's columns and lets the first
    update of every other column read A, gives bit for bit what factor on a full
    copy and pcg give, with tiles of two formats; also when the first attempt
    breaks down (eps' = 1e12: E4M3 everywhere) and A is copied again."""
    print("[case]", n, nb, agg, eps, flush=True)
    A, _ = S.matgen_householder(handle, n, cond=1e6, lam_max=1e6, seed=n)
    B = torch.from_numpy(np.random.default_rng(n).standard_normal((2, n))).cuda()
    fo = S.factor_opts(nb=nb, update_prec=L.PREC_SWITCH, ladder=(E4, F32), eps_prime=eps, fallback=fallback,
                       agg_panels=agg)
    po = S.pcg_opts(tol=1e-10, maxit=300)
    keep = A.clone()
    Lf = A.clone()
    rc, fi2, _, _ = S.factor(handle, Lf, fo)
    assert rc == 0 and (fi2.retries > 0) == bool(fallback)
    # (with the handle's last factor, whose 32x32 inverses it still has)
    X2, pi2, rc2 = S.pcg(handle, A, Lf, B, nb=nb, opts=po)
    X1, fi1, pi1, rc1 = S.precond_cg(handle, A, B, fo, po)
    assert rc1 == 0 and rc2 == 0 and pi1.iters == pi2.iters and fi1.retries == fi2.retries
    assert list(fi1.syrk_flops) == list(fi2.syrk_flops)
    if not fallback:
        assert fi1.syrk_flops[E4] > 0 and fi1.syrk_flops[F32] > 0
    assert torch.equal(X1, X2)
    assert torch.equal(A, keep)
