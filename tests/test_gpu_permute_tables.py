"""permutedims calls whose tables go through the handle's staging ring: many
calls in flight on two streams with different structures, tables too large
for the ring, orders 1 to 5 with empty sectors, and the refusal under stream
capture; and the forms a block can take (streamed, or tiles whose sides
follow the block's dims). Values are moved, or scaled by powers of two and
added once: compared exactly with numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(ND, rng, sectors, density=1.0, dtype=np.float64):
    import itertools
    import torch
    offs, n = {}, 0
    for b in itertools.product(*(range(1, len(s) + 1) for s in sectors)):
        if rng.random() <= density:
            offs[b] = n
            n += int(np.prod([s[c - 1] for s, c in zip(sectors, b)]))
    x = rng.standard_normal(n)
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.standard_normal(n)
    return ND.BlockSparseTensor(torch.from_numpy(x.astype(dtype)).cuda(), offs, sectors)


def _check(T, R, perm):
    assert list(R.blockoffsets) == [tuple(b[p - 1] for p in perm) for b in T.blockoffsets]
    th, rh = T.data.cpu().numpy(), R.data.cpu().numpy()
    for b, bp in zip(T.blockoffsets, R.blockoffsets):
        assert np.array_equal(R.block_numpy(bp, rh),
                              T.block_numpy(b, th).transpose([p - 1 for p in perm]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
def test_many_calls_on_two_streams(dtype):
    import torch
    from itg import ndtensors as ND
    rng = np.random.default_rng(1)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    work = []
    for k in range(14):
        n = 1 + k % 5
        sectors = tuple(tuple(int(x) for x in rng.integers(0, 9, size=rng.integers(1, 5)))
                        for _ in range(n))
        work.append((_tensor(ND, rng, sectors, 0.7, dtype), tuple(rng.permutation(n) + 1)))
    torch.cuda.synchronize()
    out = []
    for k, (T, perm) in enumerate(work):
        with torch.cuda.stream(streams[k % 2]):
            if T.blockoffsets and T.data.numel() == 0:  # no data pointer: refused
                with pytest.raises(ND.ItgError):
                    ND.permutedims(T, perm)
                out.append(None)
            else:
                out.append(ND.permutedims(T, perm))
    torch.cuda.synchronize()
    assert sum(R is not None for R in out) >= 10
    for (T, perm), R in zip(work, out):
        if R is not None:
            _check(T, R, perm)


def test_tables_larger_than_the_ring():
    import torch
    from itg import ndtensors as ND
    rng = np.random.default_rng(2)
    T = _tensor(ND, rng, ((1, 2) * 85, (2, 1, 1) * 57))  # 29070 blocks
    R = ND.permutedims(T, (2, 1))
    S = ND.permutedims(R, (2, 1))
    torch.cuda.synchronize()
    assert torch.equal(S.data, T.data)
    x = T.data.cpu().numpy()
    assert np.array_equal(R.to_numpy_dense(), T.to_numpy_dense().T)
    assert x.size == R.data.numel()


def test_refused_under_capture():
    import torch
    from itg import ndtensors as ND
    rng = np.random.default_rng(3)
    T = _tensor(ND, rng, ((3, 4), (5, 2), (2,)))
    want = ND.permutedims(T, (3, 1, 2))
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        with pytest.raises(ND.ItgError):
            ND.permutedims(T, (3, 1, 2))
    got = ND.permutedims(T, (3, 1, 2))
    assert torch.equal(got.data, want.data)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("dims,perm", [
    ((1,), (1,)), ((5, 7), (2, 1)), ((2, 600), (2, 1)), ((600, 3), (2, 1)), ((31, 33), (2, 1)),
    ((32, 32), (2, 1)), ((33, 8), (2, 1)), ((8, 32), (2, 1)), ((16, 16), (2, 1)), ((15, 17), (2, 1)),
    ((1, 65, 1, 70), (4, 3, 2, 1)), ((3, 5, 130), (3, 1, 2)), ((40, 1, 2, 50), (3, 4, 2, 1)),
    ((2, 9, 3, 40), (4, 2, 1, 3)), ((70, 2, 3, 5), (3, 1, 4, 2)), ((1030, 2, 1), (2, 3, 1)),
    ((2, 3, 2, 3, 2, 3, 2, 3), (8, 6, 4, 2, 7, 5, 3, 1)), ((4, 600, 2), (3, 2, 1))])
def test_block_forms(dims, perm, dtype):
    import torch
    from itg import ndtensors as ND
    rng = np.random.default_rng(sum(dims))

    def draw(shape):
        x = rng.standard_normal(shape)
        return (x + 1j * rng.standard_normal(shape) if np.dtype(dtype).kind == "c" else x).astype(
            dtype)

    p0 = [p - 1 for p in perm]
    x, y = draw(dims), draw([dims[p] for p in p0])
    T = ND.DenseTensor.from_numpy(x)
    assert np.array_equal(ND.permutedims(T, perm).to_numpy(), x.transpose(p0))
    R = ND.permutedims_(ND.DenseTensor.from_numpy(y), T, perm, alpha=2.0, beta=0.5)
    wide = np.complex128 if np.dtype(dtype).kind == "c" else np.float64
    want = (2.0 * x.transpose(p0).astype(wide) + 0.5 * y.astype(wide)).astype(dtype)
    assert np.array_equal(R.to_numpy(), want)
