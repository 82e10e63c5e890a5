"""The split product's bits against the digit arithmetic itself, on the CPU: row
exponents, radix-254 digits and level sums in exact integers, the recombination
with exactly rounded fused multiply-adds. Every element is compared, so every wave
and fragment of a tile, edge tiles, K steps and the pairs of an output block are.
"""
from fractions import Fraction

import numpy as np
import pytest

from test_gpu_split import PREC

pytestmark = pytest.mark.gpu
S = 6  # digits
INV_RADIX, INV_LEAD2 = 1.0 / 254.0, 1.0 / (127.0 * 127.0)


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def row_exponents(*parts):
    m = np.max([np.abs(x).max(axis=1) for x in parts], axis=0)
    return np.where(m > 0, np.frexp(m)[1], 0)


def digits(X, e):
    """S arrays of integers: the digits of each value of X under its row's scale."""
    y = np.ldexp(X, -e[:, None]) * 127.0
    out = []
    for _ in range(S):
        v = np.rint(y)
        y = (y - v) * 254.0
        out.append(v.astype(np.int64))
    return out


def levels(dA, dB, sign=1):
    lev = [0] * S
    for i in range(S):
        for j in range(S - i):
            lev[i + j] = lev[i + j] + sign * (dA[i] @ dB[j].T)
    return lev


def recombined(lev, ea, eb):
    out = np.empty(lev[0].shape)
    for m, n in np.ndindex(*out.shape):
        h = float(lev[S - 1][m, n])
        for L in range(S - 2, -1, -1):
            h = fma(h, INV_RADIX, float(lev[L][m, n]))
        out[m, n] = np.ldexp(h * INV_LEAD2, int(ea[m] + eb[n]))
    return out


def product(A, B, conja=False, conjb=False):
    """The split product of (M x K) (K x N) before scaling and accumulation."""
    if not np.iscomplexobj(A):
        ea, eb = row_exponents(A), row_exponents(B.T)
        return recombined(levels(digits(A, ea), digits(B.T, eb)), ea, eb)
    A, B = (np.conj(A) if conja else A), (np.conj(B) if conjb else B)
    ea, eb = row_exponents(A.real, A.imag), row_exponents(B.T.real, B.T.imag)
    ar, ai, br, bi = (digits(np.ascontiguousarray(x), e) for x, e in
                      ((A.real, ea), (A.imag, ea), (B.T.real, eb), (B.T.imag, eb)))
    add = lambda x, y: [p + q for p, q in zip(x, y)]
    re = add(levels(ar, br), levels(ai, bi, -1))
    im = add(levels(ar, bi), levels(ai, br))
    return recombined(re, ea, eb) + 1j * recombined(im, ea, eb)


def values(rng, shape, cplx, axis):
    """Rows (along `axis`) of very different magnitude, one of zeros. Values are
    multiples of 2^-40 of their row's scale: forming their digits then rounds
    nowhere, whether or not a product and a difference are fused."""
    def part():
        x = rng.standard_normal(shape) * 2.0 ** rng.integers(-8, 9, shape)
        x = np.moveaxis(x, axis, 0)
        x = np.rint(x * 2.0 ** 30) * 2.0 ** -30  # below 2^12: at most 42 bits
        x *= 2.0 ** rng.integers(-60, 60, (x.shape[0], 1))
        if x.shape[0] > 40:
            x[7] = 0.0
        return np.ascontiguousarray(np.moveaxis(x, 0, axis))
    return part() + 1j * part() if cplx else part()


def bits(x):
    # a negated zero equals a zero
    return (np.ascontiguousarray(x) + 0.0).view(np.int64)


@pytest.mark.parametrize("mnk", [(64, 64, 32), (130, 70, 24), (33, 129, 100), (97, 65, 515), (5, 200, 1111)])
@pytest.mark.parametrize("kfirst", [False, True])
def test_real(env, mnk, kfirst):
    torch, itg, ND = env
    M, N, K = mnk
    rng = np.random.default_rng(M + N + K)
    A, B = values(rng, (M, K), False, 0), values(rng, (K, N), False, 1)
    a = ND.DenseTensor.from_numpy(np.ascontiguousarray(A.T) if kfirst else A)
    b = ND.DenseTensor.from_numpy(B if kfirst else np.ascontiguousarray(B.T))
    T = ND.contract(a, (-1, 1) if kfirst else (1, -1), b, (-1, 2) if kfirst else (2, -1), (1, 2),
                    prec=PREC)
    torch.cuda.synchronize()
    assert np.array_equal(bits(T.to_numpy()), bits(product(A, B)))


@pytest.mark.parametrize("mnk", [(64, 64, 32), (70, 65, 100), (33, 97, 321)])
@pytest.mark.parametrize("conja,conjb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_complex(env, mnk, conja, conjb):
    torch, itg, ND = env
    M, N, K = mnk
    rng = np.random.default_rng(M + N + K)
    A, B = values(rng, (M, K), True, 0), values(rng, (K, N), True, 1)
    a, b = ND.DenseTensor.from_numpy(A), ND.DenseTensor.from_numpy(B)
    T = ND.contract(a, (1, -1), b, (-1, 2), (1, 2), prec=PREC, conj1=bool(conja), conj2=bool(conjb))
    torch.cuda.synchronize()
    got, want = T.to_numpy(), product(A, B, conja, conjb)
    assert np.array_equal(bits(got.real), bits(want.real))
    assert np.array_equal(bits(got.imag), bits(want.imag))


def test_block_pairs(env):
    """Output blocks summed over three pairs, in plan order."""
    torch, itg, ND = env
    rng = np.random.default_rng(5)
    md, kd, nd = (70, 33), (40, 129, 31), (65, 20)
    A = {(i, k): values(rng, (m, q), False, 0) for k, q in enumerate(kd, 1) for i, m in enumerate(md, 1)}
    B = {(k, j): values(rng, (q, n), False, 1) for j, n in enumerate(nd, 1) for k, q in enumerate(kd, 1)}

    def tensor(X, dims):
        offs, o = {}, 0
        for b, x in X.items():
            offs[b] = o
            o += x.size
        data = np.concatenate([x.flatten(order="F") for x in X.values()])
        return ND.BlockSparseTensor(torch.from_numpy(data).cuda(), offs, dims)

    a, b = tensor(A, (md, kd)), tensor(B, (kd, nd))
    p = ND.bs_plan(a, (1, -1), b, (-1, 2), (1, 2))
    R = torch.full((p.nnzR,), float("nan"), dtype=torch.float64, device="cuda")
    p.execute(R, a.data, b.data, prec=PREC)
    torch.cuda.synchronize()
    data = R.cpu().numpy()
    for (i, j), o in zip(p.blocksR, p.offsR):
        m, n = md[i - 1], nd[j - 1]
        want = np.zeros((m, n))
        for k in range(1, len(kd) + 1):  # sequential pair order: T1's blocks outer
            want = want + product(A[i, k], B[k, j])
        assert np.array_equal(bits(data[o:o + m * n].reshape((m, n), order="F")), bits(want))
