"""Complex data with infinities through permuted copies: a permutation moves values
as they are, and a contraction of few values whose plan permutes its operands or
its output gives the infinities of the products, not NaN.
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


SPECIAL = (complex(np.inf, 0.0), complex(-np.inf, 2.0), complex(0.0, np.inf), complex(np.nan, 1.0),
           complex(1.0, -np.inf), complex(-0.0, 0.0))


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("dims,perm", [((7,), (1,)), ((40, 50), (2, 1)), ((5, 33, 6), (3, 1, 2)),
                                       ((64, 3, 70), (1, 3, 2))])
def test_permutedims_copies(env, dtype, dims, perm):
    torch, itg, ND = env
    x = rand(np.random.default_rng(0), dims, True).astype(dtype)
    flat = x.reshape(-1)
    flat[:6] = np.array(SPECIAL, dtype=dtype)
    T = ND.permutedims(ND.DenseTensor.from_numpy(np.asfortranarray(x)), perm)
    torch.cuda.synchronize()
    want = np.ascontiguousarray(np.transpose(x, [p - 1 for p in perm]))
    part = np.float64 if dtype is np.complex128 else np.float32
    assert np.array_equal(np.ascontiguousarray(T.to_numpy()).view(part), want.view(part), equal_nan=True)


# A (m1, k1, m2, k2) B (n, k2, k1) -> R: the operands, or the output too, are permuted
@pytest.mark.parametrize("lR", [(1, 2, 3), (1, 3, 2)])
@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_few_values(env, lR, dtype):
    torch, itg, ND = env
    rng = np.random.default_rng(1)
    dims = {1: 40, 2: 30, -1: 5, -2: 4, 3: 300}
    la, lb = (1, -1, 2, -2), (3, -2, -1)
    A = rand(rng, tuple(dims[x] for x in la), True).astype(dtype)
    B = rand(rng, tuple(dims[x] for x in lb), True).astype(dtype)
    A[3, 2, 7, 1] = complex(np.inf, 0.0)
    a, b = ND.DenseTensor.from_numpy(A), ND.DenseTensor.from_numpy(B)
    with ND.timer() as t:
        T = ND.contract(a, la, b, lb, lR)
        torch.cuda.synchronize()
    assert "permute_kernel" in t.results
    got = T.to_numpy()
    got = got if lR == (1, 2, 3) else got.transpose(0, 2, 1)
    row = got[3, 7]
    v = B[:, 1, 2]  # the values the infinity is multiplied with
    assert np.array_equal(row.real, np.sign(v.real) * np.inf)
    assert np.array_equal(row.imag, np.sign(v.imag) * np.inf)
    got[3, 7] = 0.0
    assert np.isfinite(got).all()
