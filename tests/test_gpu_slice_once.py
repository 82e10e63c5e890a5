"""Slicing of real operands in one pass (K up to 2048) against the two-pass form:
the same product with zeros appended along K until the two-pass form takes it
must have the same bits (digits and row exponents are equal, the digit products
are exact, zeros add nothing). Row and K remainders, both storage orders,
several row and K modes, rows of zeros, of Inf / NaN and of tiny values, and
plans whose blocks take both forms with either operand's digits kept.
"""
import numpy as np
import pytest

from test_gpu_split import PREC, SPLIT_RTOL

pytestmark = pytest.mark.gpu
LONG = 2049  # the first K of the two-pass form


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import _lib
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, _lib, ND


def _equal(torch, a, b):
    return torch.equal(a.contiguous().view(torch.int64), b.contiguous().view(torch.int64))


def _product(ND, A, B, kfirst):
    """(R x K) (K x N), operands stored as they are or transposed."""
    ka = ((-1, 1), A.T) if kfirst else ((1, -1), A)
    kb = ((-1, 2), B) if kfirst else ((2, -1), B.T)
    a, b = (ND.DenseTensor.from_numpy(np.asfortranarray(x)) for x in (ka[1], kb[1]))
    return ND.contract(a, ka[0], b, kb[0], (1, 2), prec=PREC)


@pytest.mark.parametrize("K", [24, 31, 32, 33, 100, 500, 512, 513, 1023, 1040, 2017, 2048])
@pytest.mark.parametrize("R", [30, 64, 259])
@pytest.mark.parametrize("kfirst", [False, True])
def test_same_bits_as_two_passes(env, R, K, kfirst):
    torch, itg, _lib, ND = env
    rng = np.random.default_rng(R + K)
    A, B = rng.standard_normal((R, K)), rng.standard_normal((K, 70))
    A *= 2.0 ** rng.integers(-40, 40, (R, 1))
    A[3] = 0.0
    A[5] *= 1e-300
    A[:, 7] = 0.0
    zA, zB = np.zeros((R, LONG - K)), np.zeros((LONG - K, 70))
    got = _product(ND, A, B, kfirst)
    want = _product(ND, np.hstack([A, zA]), np.vstack([B, zB]), kfirst)
    torch.cuda.synchronize()
    assert _equal(torch, got.data, want.data)
    ref = A @ B
    ok = np.linalg.norm(ref, axis=1) > 0
    err = np.linalg.norm(got.to_numpy() - ref, axis=1)[ok] / np.linalg.norm(ref, axis=1)[ok]
    assert err[np.flatnonzero(ok) != 5].max() < 10 * SPLIT_RTOL


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_rows(env, bad):
    torch, itg, _lib, ND = env
    rng = np.random.default_rng(1)
    R, K = 90, 300
    A, B = rng.standard_normal((R, K)), rng.standard_normal((K, 70))
    A[11, 0], A[12, K - 1], A[80, 150] = bad, bad, bad
    out = _product(ND, A, B, False).to_numpy()
    want = _product(ND, np.hstack([A, np.zeros((R, LONG - K))]),
                    np.vstack([B, np.zeros((LONG - K, 70))]), False).to_numpy()
    rows = [11, 12, 80]
    assert not np.isfinite(out[rows]).any()
    assert np.isfinite(np.delete(out, rows, axis=0)).all()
    np.testing.assert_array_equal(out, want)


@pytest.mark.parametrize("la,da", [((1, -1, 2, -2), (7, 5, 11, 40)), ((-2, 2, 1, -1), (40, 11, 7, 5)),
                                   ((-1, 1, -2, 2), (5, 7, 40, 11))])
def test_several_modes(env, la, da):
    torch, itg, _lib, ND = env
    rng = np.random.default_rng(2)
    A, B = rng.standard_normal(da), rng.standard_normal((5, 40, 64))
    ax = la.index(-2)
    pa, pb = [(0, 0)] * 4, [(0, 0), (0, LONG // 5 + 1 - 40), (0, 0)]
    pa[ax] = (0, LONG // 5 + 1 - 40)
    out = []
    for X, Y in ((A, B), (np.pad(A, pa), np.pad(B, pb))):
        a, b = (ND.DenseTensor.from_numpy(np.asfortranarray(x)) for x in (X, Y))
        out.append(ND.contract(a, la, b, (-1, -2, 3), (1, 2, 3), prec=PREC).data)
    torch.cuda.synchronize()
    assert _equal(torch, *out)


def test_both_forms_in_one_plan_and_kept_digits(env):
    """Blocks of K = 100 and 2100 in each operand; either or both kept."""
    torch, itg, _lib, ND = env
    QN, Index = itg.QN, itg.Index
    sp = lambda s: [(QN(("Sz", q)), n) for q, n in s]
    rng = np.random.default_rng(3)
    i = Index(sp([(0, 72), (1, 48), (2, 66)]), "i", dir=itg.Out)
    j = Index(sp([(0, 2100), (1, 100), (2, 2048)]), "j", dir=itg.In)
    l = Index(sp([(0, 65), (1, 90), (2, 30)]), "l", dir=itg.In)
    A = itg.random_itensor(QN(("Sz", 0)), i, j, rng=rng)
    B = itg.random_itensor(QN(("Sz", 0)), j.dag(), l, rng=rng)
    la, lb = itg.compute_contraction_labels(A.inds, B.inds)
    p = ND.bs_plan(A.tensor, la, B.tensor, lb, ND.contract_labels(la, lb))
    a, b = A.tensor.data, B.tensor.data
    ref = torch.empty(p.nnzR, dtype=torch.float64, device="cuda")
    plain = torch.empty_like(ref)
    p.execute(ref, a, b)
    p.execute(plain, a, b, prec=PREC)
    torch.cuda.synchronize()
    assert (plain - ref).norm() / ref.norm() < SPLIT_RTOL
    k1, k2 = _lib.ITG_FLAG_KEEP_SLICES_1, _lib.ITG_FLAG_KEEP_SLICES_2
    r1, r2 = _lib.ITG_FLAG_REUSE_SLICES_1, _lib.ITG_FLAG_REUSE_SLICES_2
    for keep, reuse in ((k1, r1), (k2, r2), (k1 | k2, r1 | r2)):
        for flags in (keep, reuse):
            out = torch.full_like(ref, float("nan"))
            p.execute(out, a, b, prec=PREC, flags=flags)
            torch.cuda.synchronize()
            assert _equal(torch, out, plain)
