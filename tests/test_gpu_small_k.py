"""Contractions over few values (2 to 23): GEMM, strided or fiber kernels by the
plan's estimate. Every storage order of both operands and of the result, real
and complex with conjugations, dense and block-sparse, against numpy and
against the strided kernel (gemm backend Generic); split precision gives the
FP64 bits; a plan's first run may be inside a capture; a run in the fixed
scratch buffer needs no run before it.

Sums of at most 23 products per block pair: 64 eps times the sum of magnitudes
covers any order of addition on both sides.
"""
import itertools

import numpy as np
import pytest

from helpers import rand

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


def einsum(X, l1, Y, l2, lR):
    name = {x: chr(97 + i) for i, x in enumerate(dict.fromkeys(l1 + l2))}
    f = "".join
    return np.einsum("%s,%s->%s" % (f(name[x] for x in l1), f(name[x] for x in l2),
                                    f(name[x] for x in lR)), X, Y, optimize=True)


# free dims of T1, contracted dims, free dims of T2
SHAPES = [((300,), (12,), (400,)), ((50,), (20,), (60,)), ((1000,), (4,), (999,)),
          ((65, 3), (2, 5), (130,)), ((40, 41), (5, 3), (50,)), ((129,), (23,), (7, 33)),
          ((200,), (10,), (3000,)), ((3,), (20,), (5000,)), ((17, 13), (6,), (40,))]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("cplx", [False, True], ids=["f64", "c128"])
def test_dense_orders(env, shape, cplx):
    torch, itg, ND = env
    m, k, n = SHAPES[shape]
    rng = np.random.default_rng(shape)
    lm = tuple(range(1, 1 + len(m)))
    ln = tuple(range(10, 10 + len(n)))
    lk = tuple(range(-1, -1 - len(k), -1))
    dim = dict(zip(lm + ln + lk, m + n + k))
    p1 = list(itertools.permutations(lm + lk))
    p2 = list(itertools.permutations(lk + ln))
    pR = list(itertools.permutations(lm + ln))
    for i in range(max(len(p1), len(p2), len(pR))):
        l1, l2, lR = p1[i % len(p1)], p2[(2 * i + 1) % len(p2)], pR[(i + shape) % len(pR)]
        X = rand(rng, tuple(dim[x] for x in l1), cplx)
        Y = rand(rng, tuple(dim[x] for x in l2), cplx)
        c1, c2 = (bool(i & 1), bool(i & 2)) if cplx else (False, False)
        a, b = ND.DenseTensor.from_numpy(X), ND.DenseTensor.from_numpy(Y)
        kw = dict(conj1=c1, conj2=c2)
        T = ND.contract(a, l1, b, l2, lR, **kw)
        S = ND.contract(a, l1, b, l2, lR, prec="split_int8", **kw)
        C = rand(rng, tuple(dim[x] for x in lR), cplx)
        U = ND.DenseTensor.from_numpy(C)
        ND.contract_(U, lR, a, l1, b, l2, -1.5, 0.5, **kw)
        torch.cuda.synchronize()
        ref = einsum(np.conj(X) if c1 else X, l1, np.conj(Y) if c2 else Y, l2, lR)
        mag = einsum(np.abs(X), l1, np.abs(Y), l2, lR)
        tol = 64 * EPS * mag * (2 if cplx else 1)
        assert np.all(np.abs(T.to_numpy() - ref) <= tol), (l1, l2, lR)
        assert np.array_equal(S.to_numpy(), T.to_numpy())
        assert np.all(np.abs(U.to_numpy() - (-1.5 * ref + 0.5 * C)) <=
                      2 * tol + 4 * EPS * np.abs(C))


def u1(ND, torch, sectors, rng, cplx):
    """Rank-3 tensor of the blocks (i, j, k) with k = (i + j) mod n."""
    offs, o = {}, 0
    s0, s1, s2 = sectors
    for k in range(len(s2)):
        for j in range(len(s1)):
            for i in range(len(s0)):
                if (i + j) % len(s2) == k:
                    offs[(i + 1, j + 1, k + 1)] = o
                    o += s0[i] * s1[j] * s2[k]
    return ND.BlockSparseTensor(torch.from_numpy(rand(rng, (o,), cplx)).cuda(), offs, sectors)


SECTORS = [(40, 5, 17), (1, 9), (12, 3, 20)], [(90, 64, 70), (2, 3), (23, 6, 11)]


@pytest.mark.parametrize("sec", range(len(SECTORS)))
@pytest.mark.parametrize("cplx", [False, True], ids=["f64", "c128"])
def test_block_sparse(env, sec, cplx):
    torch, itg, ND = env
    rng = np.random.default_rng(sec)
    s0, s1, s2 = SECTORS[sec]
    A, B = u1(ND, torch, (s0, s1, s2), rng, cplx), u1(ND, torch, (s2, s1, s0), rng, cplx)
    for l1, l2, lR in [((1, 2, -1), (-1, 3, 4), (1, 2, 3, 4)), ((1, 2, -1), (-1, 3, 4), (3, 1, 4, 2)),
                       ((1, -2, -1), (-1, -2, 4), (4, 1)), ((1, -2, -1), (-1, -2, 4), (1, 4))]:
        name = ND.gemm_backend()
        p = ND.bs_plan(A, l1, B, l2, lR)
        R = torch.full((p.nnzR,), float("nan"), dtype=A.data.dtype, device="cuda")
        # the first run of the plan inside a capture (an ordinary GEMM plan,
        # such as those that contract two modes here, must run once before)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        if -2 not in l1:
            with torch.cuda.graph(g):
                p.execute(R, A.data, B.data)
            for _ in range(3):
                R.fill_(float("nan"))
                g.replay()
                torch.cuda.synchronize()
            first = R.clone()
            R.fill_(float("nan"))
            p.execute(R, A.data, B.data)
            torch.cuda.synchronize()
            assert torch.equal(first, R)
        else:
            p.execute(R, A.data, B.data)
        S = torch.full_like(R, float("nan"))
        p.execute(S, A.data, B.data, prec="split_int8")
        try:
            ND._set_backend("Generic")
            q = ND.bs_plan(A, l1, B, l2, lR)
            G, M = torch.empty_like(R), torch.empty(R.shape, dtype=torch.float64, device="cuda")
            q.execute(G, A.data, B.data)
            q.execute(M, A.data.abs(), B.data.abs())
        finally:
            ND._set_backend(name)
        torch.cuda.synchronize()
        assert bool(torch.all((R - G).abs() <= 128 * EPS * M))
        if -2 not in l1:  # few values: FP64 in split precision too
            assert torch.equal(S, R)
