"""A permutation is queued on the current stream, behind whatever that stream still
has to do, when its call returns: a source (or a destination) that the caller drops
then, and whose memory belongs to another stream, stays untouched until it has run.
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


def dense(ND, rng):
    return ND.DenseTensor.from_numpy(rand(rng, (300, 200, 10)))


def blocks(ND, rng):
    import torch
    sizes, offs, o = ((40, 70), (50, 30), (90, 60)), {}, 0
    for b in np.ndindex(2, 2, 2):
        offs[tuple(c + 1 for c in b)] = o
        o += int(np.prod([s[c] for s, c in zip(sizes, b)]))
    return ND.BlockSparseTensor(torch.from_numpy(rand(rng, (o,))).cuda(), offs, sizes)


def reuse(torch, n):
    """New tensors of this size on the current stream, overwritten."""
    return [torch.full((n,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(4)]


@pytest.mark.parametrize("make", [dense, blocks])
@pytest.mark.parametrize("side", [True, False], ids=["run_on_side_stream", "made_on_side_stream"])
def test_dropped_source(env, make, side):
    torch, itg, ND = env
    rng = np.random.default_rng(0)
    s, main = torch.cuda.Stream(), torch.cuda.current_stream()
    owner, runner = (main, s) if side else (s, main)
    with torch.cuda.stream(owner):
        T = make(ND, rng)
    torch.cuda.synchronize()
    want = ND.permutedims(T, (3, 1, 2)).data.clone()
    torch.cuda.synchronize()
    n = T.data.numel()
    with torch.cuda.stream(runner):
        torch.cuda._sleep(20_000_000)  # some 10 ms ahead of the permutation
        R = ND.permutedims(T, (3, 1, 2))
    del T
    with torch.cuda.stream(owner):
        X = reuse(torch, n)
    torch.cuda.synchronize()
    assert torch.equal(R.data, want)
    del X


def test_dropped_destination(env):
    torch, itg, ND = env
    rng = np.random.default_rng(1)
    T = dense(ND, rng)
    R = ND.DenseTensor(torch.empty_like(T.data), (10, 300, 200))
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        torch.cuda._sleep(20_000_000)
        ND.permutedims_(R, T, (3, 1, 2))
    n = T.data.numel()
    del R
    X = reuse(torch, n)
    torch.cuda.synchronize()
    assert all(bool(torch.isnan(x).all()) for x in X)
