"""itg_bs_autotune times both tile shapes of the FP64 GEMM on the plan's own
operands, and whichever it keeps, the bits are those of the untuned plan."""
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


def _blocks(torch, ND, rng, rows, cols, dtype):
    """Rank-2 tensor of the diagonal blocks (b, b)."""
    offs, o = {}, 0
    for b, (r, c) in enumerate(zip(rows, cols), 1):
        offs[(b, b)] = o
        o += r * c
    x = rng.standard_normal(o)
    if dtype is complex:
        x = x + 1j * rng.standard_normal(o)
    return ND.BlockSparseTensor(torch.from_numpy(x).cuda(), offs, (rows, cols))


# sizes that the planner runs whole, in quarters, and with ragged edges
@pytest.mark.parametrize("m,k,n", [((512,), (300,), (1024,)), ((160, 40), (150, 30), (140, 50)),
                                   ((2000,), (400,), (2000,)), ((65, 1, 130), (47, 31, 900), (33, 129, 7))])
@pytest.mark.parametrize("dtype", [float, complex])
def test_shapes_timed_and_bits_kept(env, m, k, n, dtype):
    torch, itg, ND = env
    rng = np.random.default_rng(sum(m) + sum(n))
    A, B = _blocks(torch, ND, rng, m, k, dtype), _blocks(torch, ND, rng, k, n, dtype)
    p = ND.bs_plan(A, (1, -1), B, (-1, 2), (1, 2))
    R = torch.full((p.nnzR,), float("nan"), dtype=A.data.dtype, device="cuda")
    p.execute(R, A.data, B.data)
    want = R.clone()
    R.fill_(float("nan"))
    with ND.timer() as t:
        p.autotune(R, A.data, B.data, prec="fp64")
    if "gemm_join_kernel" not in t.results:  # else computed in parts: kept
        assert t.results["gemm_f64_kernel"][0] >= 1 + 2 * 2  # a run, then both shapes more than once
    else:
        assert dtype is complex and m in ((512,), (65, 1, 130))
    assert torch.equal(R, want)
    R.fill_(float("nan"))
    p.execute(R, A.data, B.data)
    torch.cuda.synchronize()
    assert torch.equal(R, want)


def test_part_form_kept(env):
    torch, itg, ND = env
    rng = np.random.default_rng(1)
    A, B = (_blocks(torch, ND, rng, (1500,), (1500,), float) for _ in range(2))
    p = ND.bs_plan(A, (1, -1), B, (-1, 2), (1, 2))
    R = torch.empty(p.nnzR, dtype=torch.float64, device="cuda")
    p.execute(R, A.data, B.data)
    want = R.clone()
    p.autotune(R, A.data, B.data, prec="fp64")
    with ND.timer() as t:
        p.execute(R, A.data, B.data)
        torch.cuda.synchronize()
    assert "gemm_join_kernel" in t.results and torch.equal(R, want)
