"""One handle on several streams: calls whose workspace is the handle's (products
computed in parts along K, contractions of few values from permuted copies,
Float32 operands, split precision) alternate between two streams, and graph
replays run beside eager calls; every result has the bits of the same call made
alone.
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


class Product:
    """R = A B with buffers of its own; dims by label."""

    def __init__(self, ND, rng, dims, la, lb, lR, cplx=False, f32=False, prec="fp64"):
        def tensor(labels):
            x = rand(rng, tuple(dims[i] for i in labels), cplx)
            return ND.DenseTensor.from_numpy(x.astype(np.float32) if f32 else x)
        self.ND, self.labels, self.prec = ND, (la, lb, lR), prec
        self.a, self.b, self.r = tensor(la), tensor(lb), tensor(lR)

    def __call__(self):
        la, lb, lR = self.labels
        self.ND.contract_(self.r, lR, self.a, la, self.b, lb, prec=self.prec)
        return self.r.data


def maker(ND, rng, name):
    def plain(m, k, n, **kw):
        return Product(ND, rng, {1: m, -1: k, 2: n}, (1, -1), (-1, 2), (1, 2), **kw)
    return {
        "parts": lambda: plain(1500, 1500, 1500),
        "parts_c128": lambda: plain(1500, 700, 1500, cplx=True),
        "few_values": lambda: Product(ND, rng, {1: 300, 2: 40, -1: 5, -2: 4, 3: 700},
                                      (1, -1, 2, -2), (3, -2, -1), (1, 2, 3)),
        "float32": lambda: plain(700, 300, 500, f32=True),
        "split": lambda: plain(700, 600, 500, prec="split_int8"),
    }[name]


# kernels that a call of each kind must have run (else it needs no workspace)
RUN = {"parts": "gemm_join_kernel", "parts_c128": "gemm_join_kernel",
       "few_values": "permute_kernel", "split": "split_gemm_kernel"}
NAMES = ["parts", "parts_c128", "few_values", "float32", "split"]


def alone(torch, ND, name, p):
    """The bits of a call made alone."""
    with ND.timer() as t:
        want = p().clone()
        torch.cuda.synchronize()
    assert name not in RUN or (RUN[name] in t.results and len(t.results) > 1)
    return want


@pytest.mark.parametrize("name", NAMES)
def test_two_streams(env, name):
    torch, itg, ND = env
    rng = np.random.default_rng(NAMES.index(name))
    kinds = [name, name, "parts"]
    ps = [maker(ND, rng, k)() for k in kinds]
    want = [alone(torch, ND, k, p) for k, p in zip(kinds, ps)]
    s = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[] for _ in ps]
    for i in range(20):
        for j, p in enumerate(ps):
            with torch.cuda.stream(s[(i + j) % 2]):
                got[j].append(p().clone())
        # the products' own buffers change streams: the caller orders those
        s[0].wait_stream(s[1])
        s[1].wait_stream(s[0])
    torch.cuda.synchronize()
    for w, g in zip(want, got):
        assert all(torch.equal(x, w) for x in g)


@pytest.mark.parametrize("name", ["parts", "parts_c128", "few_values"])
def test_replay_beside_eager_calls(env, name):
    """A caller's own capture of a product that is computed in parts, or of few
    values, replayed on one stream while eager calls of the same kind use the
    handle's workspace on another."""
    torch, itg, ND = env
    rng = np.random.default_rng(10 + NAMES.index(name))
    p, q = maker(ND, rng, name)(), maker(ND, rng, name)()
    wp, wq = alone(torch, ND, name, p), alone(torch, ND, name, q)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        p()
    s = torch.cuda.Stream()
    got_p, got_q = [], []
    for _ in range(20):
        with torch.cuda.stream(s):
            g.replay()
            got_p.append(p.r.data.clone())
        got_q.append(q().clone())
    torch.cuda.synchronize()
    assert all(torch.equal(x, wp) for x in got_p)
    assert all(torch.equal(x, wq) for x in got_q)


@pytest.mark.parametrize("name", NAMES)
def test_graph_launch_beside_eager_calls(env, name):
    """A graph launched by the library is ordered with the handle's eager calls,
    whatever workspace it uses."""
    torch, itg, ND = env
    rng = np.random.default_rng(20 + NAMES.index(name))
    p, q = maker(ND, rng, name)(), maker(ND, rng, name)()
    wp, wq = alone(torch, ND, name, p), alone(torch, ND, name, q)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        g = ND.Graph.capture(p)
    got_p, got_q = [], []
    for _ in range(20):
        with torch.cuda.stream(s):
            g.launch()
            got_p.append(p.r.data.clone())
        with torch.cuda.stream(t):
            got_q.append(q().clone())
    torch.cuda.synchronize()
    assert all(torch.equal(x, wp) for x in got_p)
    assert all(torch.equal(x, wq) for x in got_q)
