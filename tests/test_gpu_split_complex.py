"""Complex split-precision products at the edges of the one-pass kernel: K of
one, two, three and more steps of 32 with and without a remainder, K cut into
chunks at 8192, blocks on both sides of the 64 x 64 tile, every combination of
conjugations, alpha / beta, several block pairs per output block (stages run
on across pairs of different K), empty contracted modes.
"""
import numpy as np
import pytest

from helpers import rand, relerr
from test_gpu_split import PREC, SPLIT_RTOL

pytestmark = pytest.mark.gpu

CONJ = [(False, False), (True, False), (False, True), (True, True)]


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


@pytest.mark.parametrize("K", [24, 31, 32, 33, 64, 65, 96, 97, 128, 500, 8192, 8193, 8256])
@pytest.mark.parametrize("mn", [(64, 64), (65, 63), (33, 130), (200, 31)])
def test_dense_edges(env, mn, K):
    torch, itg, ND = env
    rng = np.random.default_rng(K)
    M, N = mn
    A, B = rand(rng, (M, K), True), rand(rng, (K, N), True)
    a, b = ND.DenseTensor.from_numpy(A), ND.DenseTensor.from_numpy(B)
    for c1, c2 in CONJ:
        T = ND.contract(a, (1, -1), b, (-1, 2), (1, 2), prec=PREC, conj1=c1, conj2=c2)
        torch.cuda.synchronize()
        ref = (np.conj(A) if c1 else A) @ (np.conj(B) if c2 else B)
        assert relerr(T.to_numpy(), ref) < SPLIT_RTOL, (c1, c2)


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.5), (-0.25, 0.0), (0.5 - 2.0j, 0.75 + 0.5j)])
def test_scales(env, alpha, beta):
    torch, itg, ND = env
    rng = np.random.default_rng(5)
    A, B, C = rand(rng, (70, 90), True), rand(rng, (90, 100), True), rand(rng, (70, 100), True)
    for c1, c2 in CONJ:
        T = ND.DenseTensor.from_numpy(C)
        ND.contract_(T, (1, 2), ND.DenseTensor.from_numpy(A), (1, -1), ND.DenseTensor.from_numpy(B),
                     (-1, 2), alpha, beta, prec=PREC, conj1=c1, conj2=c2)
        torch.cuda.synchronize()
        ref = alpha * ((np.conj(A) if c1 else A) @ (np.conj(B) if c2 else B)) + beta * C
        assert relerr(T.to_numpy(), ref) < SPLIT_RTOL, (c1, c2)


@pytest.mark.parametrize("kd", [[40, 96, 32], [7, 33, 64, 161], [0, 50], [30, 0, 1, 200, 0]])
def test_block_pairs(env, kd):
    """One output block summed over pairs of these K."""
    torch, itg, ND = env
    rng = np.random.default_rng(sum(kd))
    md, nd = [70, 20], [100, 64]
    K = sum(kd)
    A, B = rand(rng, (sum(md), K), True), rand(rng, (K, sum(nd)), True)

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
    for c1, c2 in CONJ:
        T = ND.contract(a, (1, -1), b, (-1, 2), (1, 2), prec=PREC, conj1=c1, conj2=c2)
        torch.cuda.synchronize()
        ref = (np.conj(A) if c1 else A) @ (np.conj(B) if c2 else B)
        out, data = np.full_like(ref, np.nan), T.data.cpu().numpy()
        for (i, j), o in T.blockoffsets.items():
            m, n = md[i - 1], nd[j - 1]
            r, c = sum(md[:i - 1]), sum(nd[:j - 1])
            out[r:r + m, c:c + n] = data[o:o + m * n].reshape((m, n), order="F")
        assert relerr(out, ref) < SPLIT_RTOL, (c1, c2)
