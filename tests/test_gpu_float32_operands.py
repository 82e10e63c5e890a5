"""Float32 / ComplexF32 operands that a product permutes first are widened by the
permutation itself; the result must have the bits of the FP64 contraction of
the widened operands, rounded once. Shapes: tiled and streamed permutations
of T1, T2, both and neither, both operand orders, edges of the 32-wide tiles,
dense and block-sparse.
"""
import numpy as np
import pytest

from helpers import rand

pytestmark = pytest.mark.gpu

# (labels and dims of T1, of T2)
CASES = [
    (((1, 40), (-1, 33), (2, 17), (-2, 9)), ((-2, 9), (3, 31), (-1, 33), (4, 5))),
    (((1, 64), (-1, 32), (2, 32), (-2, 2)), ((-1, 32), (-2, 2), (3, 50))),
    (((1, 50), (-1, 70)), ((-1, 70), (2, 3), (4, 1), (3, 40))),
    (((-1, 8), (1, 65), (-2, 8), (2, 3)), ((3, 66), (-2, 8), (4, 2), (-1, 8))),
    (((1, 128), (-1, 64)), ((-1, 64), (2, 96))),
    (((-1, 31), (1, 200), (-2, 3)), ((-2, 3), (2, 7), (-1, 31))),
]


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


def split(case):
    return [tuple(x[i] for x in case) for i in (0, 1)]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("cplx", [False, True], ids=["f32", "c64"])
@pytest.mark.parametrize("swap", [False, True])
def test_dense(env, case, cplx, swap):
    torch, itg, ND = env
    rng = np.random.default_rng(case)
    narrow = np.complex64 if cplx else np.float32
    c1, c2 = CASES[case][::-1] if swap else CASES[case]
    (l1, d1), (l2, d2) = split(c1), split(c2)
    A, B = rand(rng, d1, cplx).astype(narrow), rand(rng, d2, cplx).astype(narrow)
    lR = ND.contract_labels(l1, l2)
    for conj in (False, True) if cplx else (False,):
        T = ND.contract(ND.DenseTensor.from_numpy(A), l1, ND.DenseTensor.from_numpy(B), l2, lR,
                        conj1=conj)
        W = ND.contract(ND.DenseTensor.from_numpy(A.astype(np.complex128 if cplx else np.float64)),
                        l1, ND.DenseTensor.from_numpy(B.astype(np.complex128 if cplx else
                                                               np.float64)), l2, lR, conj1=conj)
        torch.cuda.synchronize()
        assert T.to_numpy().dtype == narrow
        assert np.array_equal(T.to_numpy(), W.to_numpy().astype(narrow))


@pytest.mark.parametrize("cplx", [False, True], ids=["f32", "c64"])
def test_block_sparse(env, cplx):
    torch, itg, ND = env
    rng = np.random.default_rng(3)
    d1, d2 = ((20, 33), (5, 40), (30, 7)), ((30, 7), (20, 33), (64,))
    narrow = torch.complex64 if cplx else torch.float32
    wide = torch.complex128 if cplx else torch.float64

    def tensor(dims):
        offs, o = {}, 0
        for b in np.ndindex(*[len(d) for d in dims]):
            if sum(b) % 2:
                continue
            offs[tuple(x + 1 for x in b)] = o
            o += int(np.prod([d[x] for d, x in zip(dims, b)]))
        data = torch.from_numpy(rand(rng, (o,), cplx)).cuda().to(narrow)
        return ND.BlockSparseTensor(data, offs, dims)

    # T1[a, m, k] T2[k, a, n]: both operands hold the contracted modes apart
    a, b = tensor(d1), tensor(d2)
    aw = ND.BlockSparseTensor(a.data.to(wide), dict(a.blockoffsets), d1)
    bw = ND.BlockSparseTensor(b.data.to(wide), dict(b.blockoffsets), d2)
    l1, l2, lR = (-1, 1, -2), (-2, -1, 2), (1, 2)
    T, W = ND.contract(a, l1, b, l2, lR), ND.contract(aw, l1, bw, l2, lR)
    torch.cuda.synchronize()
    assert list(T.blockoffsets.items()) == list(W.blockoffsets.items())
    assert T.data.dtype == narrow and torch.equal(T.data, W.data.to(narrow))
