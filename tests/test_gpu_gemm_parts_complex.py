"""Products computed in parts along K, complex data: shapes that take this form
(every case asserts that the join ran), with ragged edges, every storage order
and conjugation, alpha / beta, a permuted output, and block pairs; captured and
allocation-free runs give the eager bits.

The bound is the one of the real cases: sums of the same K products in any order
against a long-double reference.
"""
import ctypes

import numpy as np
import pytest

from helpers import rand
from test_gpu_gemm_parts import check, env, kernels  # noqa: F401

pytestmark = pytest.mark.gpu


def joined(k):
    return "gemm_join_kernel" in k


@pytest.mark.parametrize("mnk", [(1500, 1500, 700), (1501, 1437, 701), (333, 901, 1303),
                                 (1500, 700, 900)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_dense(env, mnk, ta, tb):  # noqa: F811
    torch, itg, ND = env
    M, N, K = mnk
    rng = np.random.default_rng(M + 2 * ta + tb)
    A, B, C = rand(rng, (M, K), True), rand(rng, (K, N), True), rand(rng, (N, M), True)
    a = ND.DenseTensor.from_numpy(np.ascontiguousarray(A.T) if ta else A)
    b = ND.DenseTensor.from_numpy(np.ascontiguousarray(B.T) if tb else B)
    la, lb = ((-1, 1) if ta else (1, -1)), ((2, -1) if tb else (-1, 2))
    for c1, c2 in [(False, False), (True, False), (False, True), (True, True)]:
        X, Y = (np.conj(A) if c1 else A), (np.conj(B) if c2 else B)
        T, k = kernels(ND, torch, lambda: ND.contract(a, la, b, lb, (1, 2), conj1=c1, conj2=c2))
        assert joined(k)
        check(T.to_numpy(), X, Y)
        T = ND.DenseTensor.from_numpy(C)
        al, be = 0.5 - 1.5j, -0.25 + 2.0j
        _r, k = kernels(ND, torch, lambda: ND.contract_(T, (2, 1), a, la, b, lb, al, be, conj1=c1,
                                                        conj2=c2))
        assert joined(k) or M != N  # the operands change places
        check(T.to_numpy().T, X, Y, al, be * C.T)


def test_permuted_output(env):  # noqa: F811
    torch, itg, ND = env
    rng = np.random.default_rng(9)
    A, B, C = rand(rng, (1500, 700), True), rand(rng, (700, 1500), True), rand(rng, (30, 1500, 50), True)
    a = ND.DenseTensor.from_numpy(A.reshape((30, 50, 700), order="F"))
    b, T = ND.DenseTensor.from_numpy(B), ND.DenseTensor.from_numpy(C)
    al, be = -1.25 + 0.5j, 0.75 - 1.0j
    _r, k = kernels(ND, torch, lambda: ND.contract_(T, (1, 3, 2), a, (1, 2, -1), b, (-1, 3), al, be))
    assert joined(k) and "permute_kernel" in k
    mat = lambda X: X.transpose(0, 2, 1).reshape((1500, 1500), order="F")
    check(mat(T.to_numpy()), A, B, al, be * mat(C))


@pytest.mark.parametrize("kd", [[400, 329], [17, 31, 640, 3, 9]])
@pytest.mark.parametrize("cplx", [False, True], ids=["f64", "c128"])
def test_block_pairs(env, kd, cplx):  # noqa: F811
    """One output block summed over pairs of these K: eager, captured and
    allocation-free runs have the same bits."""
    torch, itg, ND = env
    from itg import _lib
    rng = np.random.default_rng(sum(kd))
    M, N = 1500, 1500
    A, B = rand(rng, (M, sum(kd)), cplx), rand(rng, (sum(kd), N), cplx)

    def blocks(X, axis):
        cuts = np.cumsum(kd)[:-1]
        parts = np.split(X, cuts, axis=axis)
        offs, o = {}, 0
        for i, x in enumerate(parts, 1):
            offs[(1, i) if axis == 1 else (i, 1)] = o
            o += x.size
        data = torch.from_numpy(np.concatenate([x.flatten(order="F") for x in parts])).cuda()
        return ND.BlockSparseTensor(data, offs, ((M,), tuple(kd)) if axis == 1 else (tuple(kd), (N,)))

    a, b = blocks(A, 1), blocks(B, 0)
    p = ND.bs_plan(a, (1, -1), b, (-1, 2), (1, 2))
    R = torch.full((p.nnzR,), float("nan"), dtype=a.data.dtype, device="cuda")
    _r, k = kernels(ND, torch, lambda: p.execute(R, a.data, b.data))
    assert joined(k)
    eager = R.clone()
    check(eager.cpu().numpy().reshape((M, N), order="F"), A, B)
    for _ in range(2):
        R.fill_(float("nan"))
        ptr = [ctypes.c_void_p(x.data_ptr()) for x in (R, a.data, b.data)]
        h = ND._handle(R.device)
        h.check(_lib.lib().itg_bs_execute_noalloc(h.h, p.plan, ND._dtype_code(R.dtype), *ptr,
                                                  _lib.scalar2(1.0)[0], None, _lib.PREC["fp64"], 0))
        torch.cuda.synchronize()
        assert torch.equal(R, eager)
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
