"""FP64 grouped GEMM at the sizes where it changes form: tile and slice
remainders, every number of live 16-row and 16-column blocks of a tile, one
row or column, one slice or less, pairs with different K, few tiles (run as
quarters) and many (run whole, several strips of tile columns), operands in
every storage order, blocks at odd element offsets, alpha and conj; and
leading dimensions whose slices do not fit 32-bit offsets.

Tolerance: a sum of K products in any order is within K * eps of the exact
one, relative to the sum of the products' magnitudes (real; a complex product
is four real ones, two per part). Reference and result each carry that bound,
alpha and the final rounding add three more units."""
import numpy as np
import pytest

import helpers  # noqa: F401

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _device(x):
    """x (column-major) on the device at an odd element offset."""
    import torch
    flat = torch.from_numpy(np.concatenate([[np.nan], x.reshape(-1, order="F")]).astype(x.dtype))
    return flat.to("cuda")[1:]


@pytest.fixture
def blas():
    from itg import ndtensors as ND
    ND.backend_blas()
    yield ND
    ND.backend_auto()


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 70, 17), (70, 1, 16), (2, 3, 40), (16, 17, 15),
                                   (33, 48, 31), (64, 64, 64), (65, 63, 33), (81, 129, 100),
                                   (257, 31, 47), (70, 1100, 40), (1030, 1100, 33),
                                   (2100, 2055, 20)])
def test_shapes_and_orders(blas, m, n, k, ta, tb, cplx):
    ND = blas
    rng = np.random.default_rng(m * 1000003 + n * 1009 + k)

    def draw(*s):
        x = rng.standard_normal(s)
        return x + 1j * rng.standard_normal(s) if cplx else x

    A, B = draw(m, k), draw(k, n)
    alpha = (0.75 - 0.5j) if cplx else -1.25
    lA, lB = ((-1, 1) if ta else (1, -1)), ((2, -1) if tb else (-1, 2))
    TA = ND.DenseTensor(_device(A.T if ta else A), (k, m) if ta else (m, k))
    TB = ND.DenseTensor(_device(B.T if tb else B), (n, k) if tb else (k, n))
    for al, conj in ((1.0, False), (alpha, cplx)):
        R = ND.DenseTensor(_device(np.full((m, n), np.nan, dtype=A.dtype)), (m, n))
        ND.contract_(R, (1, 2), TA, lA, TB, lB, al, 0.0, conj1=conj, conj2=conj)
        X, Y = (A.conj(), B.conj()) if conj else (A, B)
        ref = al * (X @ Y)
        bound = 2 * ((2 if cplx else 1) * k + 3) * EPS * (2 if cplx else 1) * abs(al) * (
            np.abs(A) @ np.abs(B))
        assert np.all(np.abs(R.to_numpy() - ref) <= bound)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("m,n", [((37, 66), 70), ((370, 666), 2100)])
def test_pairs_of_different_length(m, n, cplx):
    """Output blocks summing over blocks of 5, 16, 33 and 100 values of k."""
    import itg
    from itg import ndtensors as ND
    rng = np.random.default_rng(3)
    q = [itg.QN(("Sz", i)) for i in range(4)]
    i = itg.Index([(itg.QN(("Sz", 0)), m[0]), (itg.QN(("Sz", 1)), m[1])], "i", dir=itg.Out)
    j = itg.Index([(itg.QN(("Sz", 0)), n)], "j", dir=itg.In)
    k = itg.Index(list(zip(q, (5, 16, 33, 100))), "k", dir=itg.Out)
    s = itg.Index([(itg.QN(("Sz", -x)), 1) for x in range(4)], "s", dir=itg.Out)
    dt = np.complex128 if cplx else np.float64
    A = itg.random_itensor(itg.QN(("Sz", 0)), i, s, k, dtype=dt, rng=rng)
    B = itg.random_itensor(itg.QN(("Sz", 0)), k.dag(), s.dag(), j, dtype=dt, rng=rng)
    R = A * B
    a, b, got = (x.tensor.to_numpy_dense() for x in (A, B, R))
    ref = np.tensordot(a, b, axes=([1, 2], [1, 0]))
    mag = np.tensordot(np.abs(a), np.abs(b), axes=([1, 2], [1, 0]))
    assert R.tensor.nnzblocks() >= 1
    assert ND.bs_plan(A.tensor, (1, -1, -2), B.tensor, (-2, -1, 2), (1, 2)).info()[
        "strategy"] == "gemm"
    assert np.all(np.abs(got - ref) <= 2 * (2 * 154 + 3) * EPS * (2 if cplx else 1) * mag)


@pytest.mark.parametrize("shape", ["rows", "contracted"])
def test_leading_dimension_beyond_32_bit_offsets(blas, shape):
    import torch
    ND = blas
    g = torch.Generator(device="cuda").manual_seed(5)

    def draw(*s):
        return torch.randn(*s, generator=g, dtype=torch.float64, device="cuda")

    if shape == "rows":  # A column-major m x 2: 16 columns of 2^24 + 1 rows exceed 2^31 bytes
        m, n, k = (1 << 24) + 1, 3, 2
        A, B = draw(k, m), draw(n, k)  # row-major images of the column-major arrays
        R = ND.DenseTensor(torch.empty(m * n, dtype=torch.float64, device="cuda"), (m, n))
        ND.contract_(R, (1, 2), ND.DenseTensor(A.reshape(-1), (m, k)), (1, -1),
                     ND.DenseTensor(B.reshape(-1), (k, n)), (-1, 2), 1.0, 0.0)
        got, ref = R.data.reshape(n, m), B @ A
        bound = 2 * (k + 3) * EPS * (B.abs() @ A.abs())
    else:  # A stored k x m: 64 rows of 2^22 + 7 values exceed 2^31 bytes
        m, n, k = 64, 5, (1 << 22) + 7
        A, B = draw(m, k), draw(n, k)
        R = ND.DenseTensor(torch.empty(m * n, dtype=torch.float64, device="cuda"), (m, n))
        ND.contract_(R, (1, 2), ND.DenseTensor(A.reshape(-1), (k, m)), (-1, 1),
                     ND.DenseTensor(B.reshape(-1), (k, n)), (-1, 2), 1.0, 0.0)
        got, ref = R.data.reshape(n, m), B @ A.T
        # a sum of 2^22 values in 2048-value slices and library blocks: both
        # orders stay within the bound of a plain sum of that length
        bound = 2 * (k + 3) * EPS * (B.abs() @ A.abs().T)
    assert bool(((got - ref).abs() <= bound).all())
