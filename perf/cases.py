"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values; `kind` says which program it stands for:

  heff     one application of a two-site effective Hamiltonian,
           ((((L*psi)*W1)*W2)*R), through a kept ContractionSequence: the
           inner loop of an eigensolver (forward direction). Dense or with
           U(1) blocks, Float64 or ComplexF64, FP64 or split precision.
  grad     the energy E = <psi|H|psi>/<psi|psi> and its gradient with
           respect to psi by reverse mode (forward and backward, eager).
  batch    many small independent dense networks contracted together.
  small    the update of a left environment, (L*A)*W, eager: the smallest
           calls, where launches and latency count.
  pair     one eager dense contraction A*B of any shape and index order:
           matrix products, tensor contractions that have to permute,
           matrix-vector products, short contracted extents.
  permute  permutedims of a U(1) block-sparse intermediate.
  state    two operations on block-sparse states: the bond's singular values
           multiplied into x (a diagonal contraction), and <x|y>.

Sizes of the network cases come from the workloads of the package
(itg.configs, bench.py); the others are generic, odd sizes among them.
Inputs are N(0, 1) on the device, as everywhere in this repository. The U(1)
block structures are enumerated here in plain Python, so that the reference
values need nothing but torch.
"""
import itertools
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "itensors.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DTYPES = {"f32": torch.float32, "f64": torch.float64, "c128": torch.complex128}
_BYTES = {"f32": 4, "f64": 8, "c128": 16}


def listed():
    return [
        # an environment update at a bond dimension where MPS codes start out
        {"name": "small_f64", "kind": "small", "chi": 128, "d": 2, "w": 5, "dtype": "f64"},
        # the eigensolver's inner loop at the package's headline bond dimension
        {"name": "heff_u1_f64", "kind": "heff", "qns": True, "chi": 4096, "dtype": "f64",
         "prec": "fp64"},
        # the same in split precision
        {"name": "heff_u1_split", "kind": "heff", "qns": True, "chi": 4096, "dtype": "f64",
         "prec": "split_int8"},
        # time evolution with quantum numbers: complex data, uneven smaller blocks
        {"name": "heff_u1_c128", "kind": "heff", "qns": True, "chi": 1500, "dtype": "c128",
         "prec": "fp64"},
        # the same network without quantum numbers
        {"name": "heff_dense_f64", "kind": "heff", "qns": False, "chi": 1024, "dtype": "f64",
         "prec": "fp64"},
        # the largest: dense complex time evolution in split precision
        {"name": "heff_dense_c128_split", "kind": "heff", "qns": False, "chi": 1536,
         "dtype": "c128", "prec": "split_int8"},
        # many small networks at once (parallel sweeps, disorder averages)
        {"name": "batch_f64", "kind": "batch", "n": 256, "lo": 16, "hi": 96, "dtype": "f64"},
        # gradient-based optimisation of a state with quantum numbers
        {"name": "grad_u1_f64", "kind": "grad", "qns": True, "chi": 1024, "prec": "fp64"},
        # a plain matrix product with odd sizes
        {"name": "pair_matmul_f64", "kind": "pair", "a": "i:3001,k:2049", "b": "k:2049,j:1777",
         "dtype": "f64", "prec": "fp64"},
        # a tensor contraction whose operands have to be permuted, in Float32
        {"name": "pair_tensor_f32", "kind": "pair", "a": "i:96,k:70,j:50,l:30",
         "b": "l:30,m:45,k:70,n:11", "dtype": "f32", "prec": "fp64"},
        # reordering the largest intermediate of the network
        {"name": "permute_u1_f64", "kind": "permute", "chi": 4096, "perm": "1,3,4,5,2",
         "dtype": "f64"},
        # regauging a state and its overlap with another
        {"name": "state_u1_f64", "kind": "state", "chi": 4096, "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_pair(rng):
    while True:
        m, n, k = (_log(rng, 1, 6000) for _ in range(3))
        dtype = rng.choice(["f64", "f64", "f32", "c128"])
        if max(m * k, k * n, m * n) > 1 << 25 or m * n * k > 6e10 or m * n * k < 1000:
            continue
        split = {}
        for name, x in (("m", m), ("n", n), ("k", k)):
            if x >= 16 and rng.random() < 0.5:
                p = _log(rng, 2, x // 4)
                split[name] = [p, max(1, x // p)]
            else:
                split[name] = [x]
        a = [f"{c}:{d}" for c, d in zip("ij", split["m"])] + [f"{c}:{d}" for c, d in zip("kl", split["k"])]
        b = [f"{c}:{d}" for c, d in zip("no", split["n"])] + [f"{c}:{d}" for c, d in zip("kl", split["k"])]
        rng.shuffle(a)
        rng.shuffle(b)
        prec = "fp64"
        if dtype != "f32" and min(m, n, k) >= 64 and rng.random() < 0.25:
            prec = "split_int8"
        return {"kind": "pair", "a": ",".join(a), "b": ",".join(b), "dtype": dtype, "prec": prec}


def draw(rng):
    kind = rng.choice(["small", "heff", "heff", "heff", "batch", "grad", "pair", "pair", "pair",
                       "permute", "state"])
    dtype = rng.choice(["f64", "f64", "c128"])
    prec = rng.choice(["fp64", "fp64", "split_int8"])
    if kind == "small":
        return {"kind": kind, "chi": _log(rng, 8, 256), "d": rng.randint(2, 4),
                "w": rng.randint(3, 9), "dtype": rng.choice(["f64", "f64", "c128", "f32"])}
    if kind == "heff":
        qns = rng.random() < 0.6
        hi = 4096 if qns else (1536 if dtype == "f64" else 1000)
        return {"kind": kind, "qns": qns, "chi": _log(rng, 48, hi), "dtype": dtype, "prec": prec}
    if kind == "batch":
        lo = rng.randint(4, 24)
        return {"kind": kind, "n": _log(rng, 16, 256), "lo": lo, "hi": lo + rng.randint(8, 80),
                "dtype": dtype}
    if kind == "grad":
        qns = rng.random() < 0.6
        return {"kind": kind, "qns": qns, "chi": _log(rng, 32, 1500 if qns else 512), "prec": prec}
    if kind == "pair":
        return _draw_pair(rng)
    if kind == "permute":
        perm = [1, 2, 3, 4, 5]
        while perm == sorted(perm):
            rng.shuffle(perm)
        return {"kind": kind, "chi": _log(rng, 64, 4096), "perm": ",".join(map(str, perm)),
                "dtype": rng.choice(["f64", "f64", "c128", "f32"])}
    return {"kind": "state", "chi": _log(rng, 64, 4096), "dtype": dtype}


# ------------------------------------------------------------ block structure
# A tensor's structure: (index names, {block: dims}) with 0-based blocks in
# storage order; a block sparse tensor's values lie block after block, each
# column-major. Charges and arrows are those of the two-site network (MPO link
# 0, +2, -2, 0; physical +1, -1; bond q = -12 .. 12, sizes ~ exp(-q^2 / 32)).
_ARROWS = {
    "L": (("ap", 1), ("w", -1), ("a", -1)),
    "psi": (("a", 1), ("s1", 1), ("s2", 1), ("b", -1)),
    "W1": (("w", 1), ("s1", -1), ("s1p", 1), ("wp", -1)),
    "W2": (("wp", 1), ("s2", -1), ("s2p", 1), ("wpp", -1)),
    "R": (("bp", -1), ("wpp", 1), ("b", 1)),
}
_NET = ("L", "psi", "W1", "W2", "R")


def _bond(chi):
    qs = range(-12, 13)
    e = [math.exp(-q * q / 32.0) for q in qs]
    n = [round(chi * x / sum(e)) for x in e]
    n[12] = chi - (sum(n) - n[12])
    return [(q, d) for q, d in zip(qs, n) if d > 0]


def _space(name, chi):
    if name in ("a", "ap", "b", "bp"):
        return _bond(chi)
    if name in ("w", "wp", "wpp"):
        return [(0, 1), (2, 1), (-2, 1), (0, 2)]
    return [(1, 1), (-1, 1)]


def _structure(tensor, chi, qns):
    legs = _ARROWS[tensor]
    names = tuple(n for n, _ in legs)
    if not qns:
        size = {"a": chi, "ap": chi, "b": chi, "bp": chi, "w": 5, "wp": 5, "wpp": 5}
        return names, {(0,) * len(names): tuple(size.get(n, 2) for n in names)}
    spaces = [_space(n, chi) for n in names]
    blocks = {}
    for rev in itertools.product(*(range(len(s)) for s in reversed(spaces))):
        b = tuple(reversed(rev))
        if sum(d * s[c][0] for (_, d), s, c in zip(legs, spaces, b)) == 0:
            blocks[b] = tuple(s[c][1] for s, c in zip(spaces, b))
    return names, blocks


def _pairs(A, B):
    """The block pairs of A*B, A's blocks outer; the output's index names."""
    (na, ba), (nb, bb) = A, B
    shared = [n for n in na if n in nb]
    ia, ib = [na.index(n) for n in shared], [nb.index(n) for n in shared]
    fa = [i for i, n in enumerate(na) if n not in shared]
    fb = [i for i, n in enumerate(nb) if n not in shared]
    by = {}
    for y in bb:
        by.setdefault(tuple(y[i] for i in ib), []).append(y)
    out = []
    for x in ba:
        for y in by.get(tuple(x[i] for i in ia), ()):
            out.append((x, y, tuple(x[i] for i in fa) + tuple(y[i] for i in fb)))
    return out, tuple(na[i] for i in fa) + tuple(nb[i] for i in fb), ia, ib, fa, fb


def _structure_of(A, B):
    """Structure of A*B and the multiply-adds it takes."""
    pairs, names, ia, _ib, fa, fb = _pairs(A, B)
    blocks, macs = {}, 0
    for x, y, r in pairs:
        dx, dy = A[1][x], B[1][y]
        d = tuple(dx[i] for i in fa) + tuple(dy[i] for i in fb)
        blocks[r] = d
        macs += math.prod(d) * math.prod(dx[i] for i in ia)
    return (names, blocks), macs


def _nnz(S):
    return sum(math.prod(d) for d in S[1].values())


def _views(data, S):
    """The blocks of flat column-major data as torch tensors."""
    out, o = {}, 0
    for b, d in S[1].items():
        n = math.prod(d)
        out[b] = data[o:o + n].view(tuple(reversed(d))).permute(*reversed(range(len(d))))
        o += n
    return S[0], out


def _times(A, B):
    """A*B of two (names, {block: torch tensor})."""
    pairs, names, ia, ib, _fa, _fb = _pairs(A, B)
    out = {}
    for x, y, r in pairs:
        t = torch.tensordot(A[1][x], B[1][y], dims=(ia, ib))
        out[r] = out[r] + t if r in out else t
    return names, out


def _flat(T):
    """Flat column-major storage of (names, {block: torch tensor})."""
    return torch.cat([t.permute(*reversed(range(t.dim()))).reshape(-1) if t.dim() else t.reshape(-1)
                      for t in T[1].values()])


def _network(chi, qns):
    return [_structure(t, chi, qns) for t in _NET]


def _fold(structures):
    """Structures after each step of the left-to-right fold, and its MACs."""
    cur, macs, steps = structures[0], 0, []
    for S in structures[1:]:
        cur, m = _structure_of(cur, S)
        macs += m
        steps.append(cur)
    return steps, macs


# ------------------------------------------------------------------- inputs
def _randn(sizes, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + 17)
    real = torch.float64 if dtype == "c128" else _DTYPES[dtype]
    out = []
    for n in sizes:
        if dtype == "c128":
            out.append(torch.view_as_complex(torch.randn(n, 2, generator=g, dtype=real, device="cuda")))
        else:
            out.append(torch.randn(n, generator=g, dtype=real, device="cuda"))
    return out


def _parse(text):
    return [(t.split(":")[0], int(t.split(":")[1])) for t in text.split(",")]


def _batch_chis(case, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(case["lo"], case["hi"] + 1, (case["n"],), generator=g).tolist()


def _inputs(case, seed):
    """Flat input vectors of a case and their structures."""
    kind, dtype = case["kind"], case.get("dtype", "f64")
    if kind in ("heff", "grad"):
        S = _network(case["chi"], case["qns"])
    elif kind == "small":
        chi, d, w = case["chi"], case["d"], case["w"]
        S = [(("ap", "w", "a"), {(0, 0, 0): (chi, w, chi)}), (("a", "s", "b"), {(0, 0, 0): (chi, d, chi)}),
             (("w", "s", "sp", "wp"), {(0, 0, 0, 0): (w, d, d, w)})]
    elif kind == "pair":
        S = [(tuple(n for n, _ in p), {(0,) * len(p): tuple(d for _, d in p)})
             for p in (_parse(case["a"]), _parse(case["b"]))]
    elif kind == "permute":
        S = [_fold(_network(case["chi"], True)[:4])[0][-1]]
    elif kind == "state":
        # x, y and the values on the bond's diagonal
        S = [_structure("psi", case["chi"], True)] * 2 + [(("d",), {(0,): (case["chi"],)})]
    else:
        # the bond dimensions are part of the batch's plan: the same for every seed
        S = [s for chi in _batch_chis(case, 11) for s in _network(chi, False)]
    return _randn([_nnz(s) for s in S], dtype, seed), S


def _tensor(data, S, inds):
    """An ITensor over `inds` from flat data and its structure."""
    import itg
    from itg import ndtensors as ND

    if not all(i.hasqns for i in inds):
        return itg.ITensor(ND.DenseTensor(data, tuple(i.dim for i in inds)), inds)
    offs, o = {}, 0
    for b, d in S[1].items():
        offs[tuple(c + 1 for c in b)] = o
        o += math.prod(d)
    return itg.ITensor(ND.BlockSparseTensor(data, offs, tuple(i.blockdims() for i in inds)), inds)


def _net_tensors(ix, data, S):
    inds = (ix.L(), ix.psi(), ix.W1(), ix.W2(), ix.R())
    return [_tensor(x, s, i) for x, s, i in zip(data, S, inds)]


def prepare(case, seed):
    import itg
    from itg.configs import HeffIndices
    from itg.network import BatchedSequence, ContractionSequence

    kind = case["kind"]
    data, S = _inputs(case, seed)
    st = {"kind": kind, "prec": case.get("prec", "fp64")}
    if kind in ("heff", "grad"):
        ix = HeffIndices(case["chi"], case["qns"])
        net = _net_tensors(ix, data, S)
        if kind == "heff":
            # an eigensolver keeps the sequence (its plans and intermediates)
            st["seq"] = ContractionSequence(net, prec=st["prec"])
        else:
            st["net"], st["out"] = net, ix.out()
    elif kind == "small":
        bond = [itg.Index(case["chi"], t) for t in ("a'", "a", "b")]
        s, sp = itg.Index(case["d"], "s"), itg.Index(case["d"], "s'")
        w, wp = itg.Index(case["w"], "w"), itg.Index(case["w"], "w'")
        st["ts"] = [_tensor(x, None, i) for x, i in
                    zip(data, ((bond[0], w, bond[1]), (bond[1], s, bond[2]), (w, s, sp, wp)))]
    elif kind == "pair":
        named = {}
        for n, d in _parse(case["a"]) + _parse(case["b"]):
            named.setdefault(n, itg.Index(d, n))
        st["ts"] = [_tensor(x, None, tuple(named[n] for n in s[0])) for x, s in zip(data, S)]
    elif kind == "permute":
        ix = HeffIndices(case["chi"], True)
        st["ts"] = [_tensor(data[0], S[0], (ix.ap, ix.b, ix.s1p, ix.s2p, ix.wpp))]
        st["perm"] = tuple(int(p) for p in case["perm"].split(","))
    elif kind == "state":
        ix = HeffIndices(case["chi"], True)
        st["ts"] = [_tensor(x, s, ix.psi()) for x, s in zip(data[:2], S)]
        new = itg.Index(ix.b.space, "b'", dir=ix.b.dir)
        st["sv"] = itg.diag_itensor(0.0, ix.b.dag(), new, device="cuda",
                                    dtype="complex128" if case["dtype"] == "c128" else "float64")
        st["sv"].tensor.data.copy_(data[2])
    else:
        nets = []
        for k, chi in enumerate(_batch_chis(case, 11)):
            ix = HeffIndices(chi, False)
            nets.append(_net_tensors(ix, data[5 * k:5 * k + 5], S[5 * k:5 * k + 5]))
        st["batch"] = BatchedSequence(nets, prec=st["prec"])
    return st


def run(state):
    import itg
    from itg import chainrules, ndtensors

    kind = state["kind"]
    if kind == "heff":
        return state["seq"].run().tensor.data
    if kind == "grad":
        E, grad = chainrules.heff_energy_and_grad(*state["net"], state["out"], prec=state["prec"])
        return E, grad.tensor.data
    if kind == "batch":
        # every result, one after the other
        state["batch"].run()
        return state["batch"].arenas[-1]
    if kind == "small":
        L, A, W = state["ts"]
        return ((L * A) * W).tensor.data
    if kind == "pair":
        A, B = state["ts"]
        return itg.contract(A, B, prec=state["prec"]).tensor.data
    if kind == "permute":
        return ndtensors.permutedims(state["ts"][0].tensor, state["perm"]).data
    x, y = state["ts"]
    return (x * state["sv"]).tensor.data, (itg.dag(x) * y).tensor.data


def work(case):
    """Bytes (inputs read once, outputs written once) and flops of one pass."""
    kind, dtype = case["kind"], case.get("dtype", "f64")
    es = _BYTES[dtype]
    mul = 8 if dtype == "c128" else 2
    if kind in ("heff", "grad"):
        S = _network(case["chi"], case["qns"])
        steps, macs = _fold(S)
        nin = sum(_nnz(s) for s in S)
        if kind == "heff":
            return {"bytes": (nin + _nnz(steps[-1])) * es, "flops": macs * mul}
        # H psi and H^T psi
        return {"bytes": (nin + _nnz(S[1])) * es, "flops": 2 * macs * mul}
    if kind == "batch":
        nbytes = flops = 0
        for chi in _batch_chis(case, 11):
            S = _network(chi, False)
            steps, macs = _fold(S)
            nbytes += (sum(_nnz(s) for s in S) + _nnz(steps[-1])) * es
            flops += macs * mul
        return {"bytes": nbytes, "flops": flops}
    if kind == "permute":
        n = _nnz(_fold(_network(case["chi"], True)[:4])[0][-1])
        return {"bytes": 2 * n * es, "flops": 0}
    if kind == "state":
        n = _nnz(_structure("psi", case["chi"], True))
        return {"bytes": (3 * n + case["chi"]) * es, "flops": 2 * n * mul}
    if kind == "small":
        chi, d, w = case["chi"], case["d"], case["w"]
        macs = chi * w * chi * d * chi + chi * chi * w * d * d * w
        n = chi * w * chi + chi * d * chi + w * d * d * w + chi * chi * d * w
        return {"bytes": n * es, "flops": macs * mul}
    S = [(tuple(n for n, _ in p), {(0,) * len(p): tuple(d for _, d in p)})
         for p in (_parse(case["a"]), _parse(case["b"]))]
    R, macs = _structure_of(*S)
    return {"bytes": (_nnz(S[0]) + _nnz(S[1]) + _nnz(R)) * es, "flops": macs * mul}


def exact(case, seed):
    """What run() returns, from plain torch in 64 bits."""
    kind = case["kind"]
    data, S = _inputs(case, seed)
    data = [x.double() if x.dtype == torch.float32 else x for x in data]
    T = [_views(x, s) for x, s in zip(data, S)]
    if kind in ("heff", "small", "pair"):
        cur = T[0]
        for t in T[1:]:
            cur = _times(cur, t)
        return _flat(cur)
    if kind == "batch":
        out = []
        for k in range(0, len(T), 5):
            cur = T[k]
            for t in T[k + 1:k + 5]:
                cur = _times(cur, t)
            out.append(_flat(cur))
        return torch.cat(out)
    if kind == "permute":
        perm = [int(p) - 1 for p in case["perm"].split(",")]
        return _flat((None, {b: t.permute(*perm) for b, t in T[0][1].items()}))
    if kind == "state":
        bond = [d for _, d in _bond(case["chi"])]
        sv = torch.split(data[2], bond)
        scaled = {b: t * sv[b[3]] for b, t in T[0][1].items()}
        return _flat((None, scaled)), (data[0].conj() * data[1]).sum().reshape(1)
    # gradient of <psi|H|psi>/<psi|psi> for real data
    L, psi, W1, W2, R = T
    up = {"a": "ap", "s1": "s1p", "s2": "s2p", "b": "bp"}
    primed = (tuple(up[n] for n in psi[0]), psi[1])
    Hx, Ht = L, L
    for t in (psi, W1, W2, R):
        Hx = _times(Hx, t)
    for t in (primed, W1, W2, R):
        Ht = _times(Ht, t)
    order = lambda T, names: {tuple(b[T[0].index(n)] for n in names):
                              t.permute(*(T[0].index(n) for n in names)) for b, t in T[1].items()}
    hx, ht = order(Hx, primed[0]), order(Ht, psi[0])
    den = float((data[1] * data[1]).sum())
    E = sum(float((t * hx[b]).sum()) for b, t in psi[1].items() if b in hx) / den
    grad = {}
    for b, t in psi[1].items():
        g = -2.0 * E * t
        for other in (hx, ht):
            if b in other:
                g = g + other[b]
        grad[b] = g / den
    return E, _flat((None, grad))
