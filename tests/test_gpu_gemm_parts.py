"""FP64 products whose last tiles are computed in parts along K: plain shapes
that leave part of the chip idle at the end, with edge tiles, K not a multiple
of a slice, both storage orders of either operand, complex data with
conjugations, alpha / beta, an output that is permuted afterwards, block
pairs of different K in one block, and graph replay.

A sum of K products in any order differs from another by at most about
2 K eps sum |a b|; against a long-double reference the bound below uses
K eps (the part sums and their join are sums of the same K terms).
"""
import numpy as np
import pytest

from helpers import rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


def check(got, A, B, scale=1.0, extra=0.0):
    rows = np.linspace(0, A.shape[0] - 1, 24).astype(int)
    cols = np.linspace(0, B.shape[1] - 1, 24).astype(int)
    wide = np.clongdouble if np.iscomplexobj(A) else np.longdouble
    ref = scale * (A[rows].astype(wide) @ B[:, cols].astype(wide))
    if np.ndim(extra):
        ref = ref + extra[np.ix_(rows, cols)]
    mag = abs(scale) * (np.abs(A[rows]) @ np.abs(B[:, cols])) + 1.0
    tol = 4 * (A.shape[1] + 8) * np.finfo(np.float64).eps * mag
    assert np.all(np.abs(got[np.ix_(rows, cols)] - ref) <= tol)


def kernels(ND, torch, f):
    with ND.timer() as t:
        r = f()
        torch.cuda.synchronize()
    return r, list(t.results)


@pytest.mark.parametrize("mnk", [(1500, 1500, 1500), (1601, 1333, 777), (2240, 1024, 515),
                                 (4800, 495, 2100), (700, 1900, 300)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_real(env, mnk, ta, tb):
    torch, itg, ND = env
    M, N, K = mnk
    rng = np.random.default_rng(M + 2 * ta + tb)
    A, B = rand(rng, (M, K)), rand(rng, (K, N))
    a = ND.DenseTensor.from_numpy(np.ascontiguousarray(A.T) if ta else A)
    b = ND.DenseTensor.from_numpy(np.ascontiguousarray(B.T) if tb else B)
    la, lb = ((-1, 1) if ta else (1, -1)), ((2, -1) if tb else (-1, 2))
    T, _k = kernels(ND, torch, lambda: ND.contract(a, la, b, lb, (1, 2)))
    check(T.to_numpy(), A, B)
    C = rand(rng, (N, M))  # the permuted output order
    T = ND.DenseTensor.from_numpy(C)
    ND.contract_(T, (2, 1), a, la, b, lb, -0.75, 0.5)
    torch.cuda.synchronize()
    check(T.to_numpy().T, A, B, -0.75, 0.5 * C.T)


@pytest.mark.parametrize("mnk", [(1100, 900, 700), (901, 1303, 333)])
def test_complex(env, mnk):
    torch, itg, ND = env
    M, N, K = mnk
    rng = np.random.default_rng(K)
    A, B, C = rand(rng, (M, K), True), rand(rng, (K, N), True), rand(rng, (M, N), True)
    a, b = ND.DenseTensor.from_numpy(A), ND.DenseTensor.from_numpy(B)
    for c1, c2 in [(False, False), (True, False), (False, True), (True, True)]:
        X, Y = (np.conj(A) if c1 else A), (np.conj(B) if c2 else B)
        T = ND.contract(a, (1, -1), b, (-1, 2), (1, 2), conj1=c1, conj2=c2)
        check(T.to_numpy(), X, Y)
        T = ND.DenseTensor.from_numpy(C)
        al, be = 0.5 - 1.5j, -0.25 + 2.0j
        ND.contract_(T, (1, 2), a, (1, -1), b, (-1, 2), al, be, conj1=c1, conj2=c2)
        torch.cuda.synchronize()
        check(T.to_numpy(), X, Y, al, be * C)


def test_part_form_runs(env):
    torch, itg, ND = env
    rng = np.random.default_rng(1)
    a = ND.DenseTensor.from_numpy(rand(rng, (1500, 1500)))
    T, k = kernels(ND, torch, lambda: ND.contract(a, (1, -1), a, (-1, 2), (1, 2)))
    assert k == ["gemm_f64_kernel", "gemm_join_kernel"]


@pytest.mark.parametrize("kd", [[300, 5, 470], [129, 1000], [17, 31, 640, 3, 200]])
def test_block_pairs(env, kd):
    """Output blocks summed over pairs of these K: cuts fall inside pairs and
    between them; a captured run gives the eager bits on every replay."""
    torch, itg, ND = env
    rng = np.random.default_rng(sum(kd))
    md, nd = [1000, 330], [500, 700]
    A, B = rand(rng, (sum(md), sum(kd))), rand(rng, (sum(kd), sum(nd)))

    def blocks(X, rows, cols):
        offs, parts, o = {}, [], 0
        r0 = np.concatenate([[0], np.cumsum(rows)])
        c0 = np.concatenate([[0], np.cumsum(cols)])
        for j in range(len(cols)):
            for i in range(len(rows)):
                blk = X[r0[i]:r0[i + 1], c0[j]:c0[j + 1]]
                offs[(i + 1, j + 1)] = o
                o += blk.size
                parts.append(blk.flatten(order="F"))
        data = torch.from_numpy(np.concatenate(parts)).cuda()
        return ND.BlockSparseTensor(data, offs, (tuple(rows), tuple(cols)))

    a, b = blocks(A, md, kd), blocks(B, kd, nd)
    p = ND.bs_plan(a, (1, -1), b, (-1, 2), (1, 2))
    R = torch.full((p.nnzR,), float("nan"), dtype=torch.float64, device="cuda")
    _r, k = kernels(ND, torch, lambda: p.execute(R, a.data, b.data))
    eager = R.clone()
    out, data = np.full((sum(md), sum(nd)), np.nan), eager.cpu().numpy()
    for (i, j), o in zip(p.blocksR, p.offsR):
        m, n = md[i - 1], nd[j - 1]
        r, c = sum(md[:i - 1]), sum(nd[:j - 1])
        out[r:r + m, c:c + n] = data[o:o + m * n].reshape((m, n), order="F")
    check(out, A, B)
    p.execute(R, a.data, b.data)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        p.execute(R, a.data, b.data)
    for _ in range(3):
        R.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(R, eager)
        p.execute(R, a.data, b.data)
        torch.cuda.synchronize()
        assert torch.equal(R, eager)
