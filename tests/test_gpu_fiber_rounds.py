"""Fibers per workgroup of the matrix-form and chain kernels: 1, 2, 4 (and 8)
rounds of 256, at the counts where the number changes and where the last
round or workgroup is partial.

Whole-number values make every sum exact, so results must be equal; the
chain must equal its two separate steps bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    import itg
    from itg import ndtensors as ND
    torch.cuda.init()
    return torch, itg, ND


# 256 r * 1023 + 1 fibers make 1024 workgroups of r rounds
@pytest.mark.parametrize("nfib", [256, 257, 1000, 523776, 523777, 1047552, 1047553, 2095104,
                                  2095105, 2097409])
@pytest.mark.parametrize("cplx", [False, True], ids=["f64", "c128"])
def test_matrix_form_rounds(env, nfib, cplx):
    torch, itg, ND = env
    K, N = (3, 2) if not cplx else (5, 2)
    rng = np.random.default_rng(nfib)
    def ints(shape):
        x = rng.integers(-8, 9, shape).astype(np.float64)
        return x + 1j * rng.integers(-8, 9, shape) if cplx else x
    X, W = np.asfortranarray(ints((nfib, K))), np.asfortranarray(ints((K, N)))
    a, b = ND.DenseTensor.from_numpy(X), ND.DenseTensor.from_numpy(W)
    with ND.timer() as t:
        T = ND.contract(a, (1, -1), b, (-1, 2), (1, 2))
        torch.cuda.synchronize()
    assert list(t.results) == ["fiber_mv_kernel"]
    assert np.array_equal(T.to_numpy(), X @ W)


@pytest.mark.parametrize("chi,cplx", [(2048, False), (3000, False), (2200, True)])
def test_chain_rounds(env, chi, cplx):
    torch, itg, ND = env
    from itg.configs import heff_network
    from itg.network import ContractionSequence
    net = heff_network(chi, qns=True, seed=chi, dtype=np.complex128 if cplx else np.float64)[:5]
    plain = ContractionSequence(net, fuse=False)
    _k, p1, X, B1, Y, _l = plain.steps[1]
    _k, p2, _Y, B2, Z, _l = plain.steps[2]
    X.data.copy_(torch.randn(X.data.numel() * (2 if cplx else 1), dtype=torch.float64,
                             device=X.data.device).view(X.data.dtype))
    p1.execute(Y.data, X.data, B1.data)
    p2.execute(Z.data, Y.data, B2.data)
    zsep = Z.data.clone()
    Z.data.fill_(float("nan"))
    ND.BSChain(p1, p2).execute(Z.data, X.data, B1.data, B2.data)
    torch.cuda.synchronize()
    assert torch.equal(Z.data, zsep)
