"""Real split-precision products at the edges of the kernel's stage ring: K of
one, two, three and more steps of 32 with and without a remainder, K cut into
chunks at 8192, blocks on both sides of the 64 x 64 tile, several block pairs
per output block (stages run on across pairs of different K), alpha / beta.
"""
import numpy as np
import pytest

from helpers import rand, relerr
from test_gpu_split import PREC, SPLIT_RTOL

pytestmark = pytest.mark.gpu


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
    A, B, C = rand(rng, (M, K)), rand(rng, (K, N)), rand(rng, (M, N))
    a, b, T = (ND.DenseTensor.from_numpy(x) for x in (A, B, C))
    ND.contract_(T, (1, 2), a, (1, -1), b, (-1, 2), -0.5, 1.25, prec=PREC)
    T1 = ND.contract(a, (1, -1), b, (-1, 2), (1, 2), prec=PREC)
    torch.cuda.synchronize()
    assert relerr(T.to_numpy(), -0.5 * (A @ B) + 1.25 * C) < SPLIT_RTOL
    assert relerr(T1.to_numpy(), A @ B) < SPLIT_RTOL


@pytest.mark.parametrize("kd", [[40, 96, 32], [7, 33, 64, 161], [0, 50], [30, 0, 1, 200, 0]])
def test_block_pairs(env, kd):
    """One output block summed over pairs of these K."""
    torch, itg, ND = env
    rng = np.random.default_rng(sum(kd))
    md, nd = [70, 20], [100, 64]
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

    T = ND.contract(blocks(A, md, kd), (1, -1), blocks(B, kd, nd), (-1, 2), (1, 2), prec=PREC)
    torch.cuda.synchronize()
    out, data = np.full((sum(md), sum(nd)), np.nan), T.data.cpu().numpy()
    for (i, j), o in T.blockoffsets.items():
        m, n = md[i - 1], nd[j - 1]
        r, c = sum(md[:i - 1]), sum(nd[:j - 1])
        out[r:r + m, c:c + n] = data[o:o + m * n].reshape((m, n), order="F")
    assert relerr(out, A @ B) < SPLIT_RTOL
