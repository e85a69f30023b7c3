"""The work that programs have this framework do, as cases that can be timed.

A case is a dict of plain values.  `listed()` gives the named ones, `draw(rng)`
one more of the same ranges, `prepare` what a program holds before the call
(keys, masked inputs, a model), `run` one pass through the public entry points
(the C ABI of include/mpcx.h through its ctypes binding) and its outputs,
`work` the bytes and operations one pass cannot do without, and `exact` the
plain fixed-point result where the outputs are not masked by the dealer.

All outputs are ring elements, bits or key bytes, so every case is exact: two
correct implementations agree on every bit.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "idash26-track3_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mpcx  # noqa: E402
import synth  # noqa: E402

S = 12  # fixed-point scale
N_NODES = 140  # atoms a molecule is padded to
FEAT, GCN, DFC, PROT, FUS = 78, (78, 156, 312), (1024, 128), 128, (1024, 512, 1)
LUT_NMAX = 138  # largest degree + 1 in the D^-1/2 table
FEAT_GROUPS = (44, 11, 11, 11, 1)  # one-hot groups of an atom's features

KINDS = {"TR": mpcx.TR, "TRRELU": mpcx.TRRELU, "RELU": mpcx.RELU, "TRSLACK": mpcx.TRSLACK, "TRMOD": mpcx.TRMOD,
         "EXT": mpcx.EXT, "EXTRELU": mpcx.EXTRELU, "RELUPOOL": mpcx.RELUPOOL}


def listed():
    return [
        # a batch of molecules through the whole two-party affinity forward, keys resident: the headline
        {"name": "forward 64", "op": "forward", "bw": 32, "B": 64, "lanes": 3},
        # one molecule: the latency of a single request
        {"name": "forward 1", "op": "forward", "bw": 32, "B": 1, "lanes": 1},
        # the 64-bit ring, a batch of middle size
        {"name": "forward 16 ring64", "op": "forward", "bw": 64, "B": 16, "lanes": 3},
        # keys are used once: the dealer's run for a batch, then the forward that spends them
        {"name": "deal+forward 16", "op": "deal", "bw": 32, "B": 16, "lanes": 3},
        # secure ReLU as one gate call over a large activation
        {"name": "relu 2^22", "op": "gate", "dir": "eval", "kind": "RELU", "bw": 32, "n": 1 << 22},
        # the dealer's keys of the GCN-2 layer's activation gate, 64 molecules
        {"name": "extrelu keygen 1.4M", "op": "gate", "dir": "keygen", "kind": "EXTRELU", "bw": 32,
         "n": 64 * N_NODES * 156},
        # the exact truncation after one molecule's fully connected layer: the smallest gate call
        {"name": "truncate 1024", "op": "gate", "dir": "eval", "kind": "TR", "bw": 32, "n": 1024},
        # adjacency normalisation of many graphs
        {"name": "adjnorm 1024", "op": "adjnorm", "dir": "eval", "bw": 32, "B": 1024, "N": N_NODES, "lanes": 3},
        # masked max-pool of a batch's last GCN activation
        {"name": "maxpool 64", "op": "maxpool", "dir": "eval", "bw": 32, "B": 64, "N": N_NODES, "C": 312},
        # Beaver products, element by element (a batch's adjacency-sized operand)
        {"name": "mul 64x140x140", "op": "mul", "dir": "eval", "bw": 32, "n": 64 * N_NODES * N_NODES},
        # secret x secret products of a GCN aggregation, one per molecule
        {"name": "sxs 64x140x140x312", "op": "sxs", "dir": "eval", "bw": 32, "B": 64, "M": N_NODES, "K": N_NODES,
         "N": 312},
        # masked activations x public weights of the GCN-3 layer, in the 64-bit ring
        {"name": "gemm 8960x156x312 ring64", "op": "gemm", "bw": 64, "M": 64 * N_NODES, "K": 156, "N": 312},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, its logarithm uniform."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["forward", "deal", "gate", "gate", "gate", "adjnorm", "maxpool", "mul", "sxs", "gemm"])
    bw = rng.choice([32, 32, 64])
    c = {"op": op, "bw": bw}
    if op in ("forward", "deal"):
        c["B"] = _log(rng, 1, (64 if bw == 32 else 20) if op == "forward" else (16 if bw == 32 else 6))
        c["lanes"] = rng.choice([1, 2, 3]) if c["B"] > 1 else 1
        return c
    if op != "gemm":
        c["dir"] = rng.choice(["eval", "keygen"])
    if op == "gate":
        c["kind"] = rng.choice(sorted(KINDS))
        c["n"] = _log(rng, 256, 1 << (20 if c["dir"] == "keygen" or bw == 64 else 22))
    elif op == "adjnorm":
        c["B"], c["N"] = _log(rng, 1, 512 if bw == 32 else 256), rng.randint(20, N_NODES)
        c["lanes"] = rng.choice([1, 3])
    elif op == "maxpool":
        c["B"], c["N"], c["C"] = _log(rng, 1, 64 if bw == 32 else 24), rng.randint(20, N_NODES), _log(rng, 64, 312)
    elif op == "mul":
        c["n"] = _log(rng, 512, 1 << 22)
    elif op == "sxs":
        c["B"] = _log(rng, 1, 64)
        c["M"] = c["K"] = rng.randint(20, N_NODES)
        c["N"] = rng.choice([78, 156, 312, rng.randint(33, 312)])
    else:
        c["M"] = _log(rng, 1, 8960)
        c["K"], c["N"] = rng.choice([(78, 78), (78, 156), (156, 312), (312, 1024), (1024, 128), (256, 1024), (1024, 512),
                                     (rng.randint(33, 1024), rng.randint(1, 1024))])
    return c


# ---------------- inputs ----------------
def _molecules(B, seed):
    """Features (B, N, 78) at scale S, adjacency (B, N, N) with self loops, atom
    mask (B, N): random trees of 10..60 atoms and degree at most 4."""
    rng = np.random.default_rng(seed)
    X = np.zeros((B, N_NODES, FEAT), np.int64)
    A = np.zeros((B, N_NODES, N_NODES), np.int64)
    mask = np.zeros((B, N_NODES), np.int64)
    for b in range(B):
        n = int(rng.integers(10, 61))
        deg = np.zeros(n, np.int64)
        for v in range(1, n):
            u = int(rng.choice(np.flatnonzero(deg[:v] < 4)))
            A[b, u, v] = A[b, v, u] = 1
            deg[u] += 1
            deg[v] += 1
        A[b, range(n), range(n)] = 1
        mask[b, :n] = 1
        off = 0
        for g in FEAT_GROUPS:
            hot = rng.integers(0, g, n) if g > 1 else np.zeros(n, np.int64)
            X[b, np.arange(n), off + hot] = 1 << S
            off += g
    return X, A, mask


def _fixed(x):
    x = x * float(1 << S)
    return np.where(x >= 0, np.floor(x + 0.5), np.ceil(x - 0.5)).astype(np.int64)


def _layers():
    io, fin = [], FEAT
    for g in GCN:
        io.append((fin, g))
        fin = g
    io += [(GCN[2], DFC[0]), (DFC[0], DFC[1])]
    fin = DFC[1] + PROT
    for f in FUS:
        io.append((fin, f))
        fin = f
    return io


def _weights(seed):
    """[(W (in, out), b (out))] of every layer, quantised at scale S."""
    rng = np.random.default_rng(seed)
    return [(_fixed(rng.standard_normal((i, o)) * math.sqrt(2.0 / i)), _fixed(rng.uniform(-1, 1, o) / math.sqrt(i)))
            for i, o in _layers()]


def _model_inputs(case, seed):
    X, A, mask = _molecules(case["B"], seed)
    prot = _fixed(np.random.default_rng(seed + 1).standard_normal((case["B"], PROT)))
    return X, A, mask, prot, _weights(seed + 2)


def _shares(v, bw, seed):
    rng = np.random.default_rng(seed)
    m = np.uint64((1 << bw) - 1)
    v0 = rng.integers(0, 1 << 64, size=v.shape, dtype=np.uint64, endpoint=False) & m
    return v0, (v.astype(np.uint64) - v0) & m


def _rand(shape, bw, gen, span=None):
    """Ring elements on the GPU: uniform, or (span) signed values in [-span, span)."""
    t = torch.int32 if bw == 32 else torch.int64
    if span is not None:
        return torch.randint(-span, span, shape, dtype=torch.int64, device="cuda", generator=gen).to(t)
    lo = torch.randint(0, 1 << 32, shape, dtype=torch.int64, device="cuda", generator=gen)
    if bw == 64:
        lo |= torch.randint(0, 1 << 32, shape, dtype=torch.int64, device="cuda", generator=gen) << 32
    return lo.to(t) if bw == 64 else (lo - ((lo >> 31) << 32)).to(t)


def _zeros(nbytes):
    return torch.zeros(max(int(nbytes), 1), dtype=torch.uint8, device="cuda")


# ---------------- the state and one pass ----------------
def prepare(case, seed):
    op, bw = case["op"], case["bw"]
    ctx = mpcx.Ctx(bw=bw, scale=S)
    lib, h, p = ctx.lib, ctx.h, mpcx.dptr
    st = {"case": case, "ctx": ctx, "seed": seed + 1}
    if op in ("forward", "deal"):
        B = case["B"]
        X, A, mask, prot, W = _model_inputs(case, seed)
        blob = np.concatenate([np.concatenate([w.reshape(-1), b]) for w, b in W])
        m = mpcx.Model(ctx, synth.Dims(bw=bw, s=S, n_nodes=N_NODES, feat=FEAT, gcn=GCN, dfc=DFC, prot=PROT, fus=FUS,
                                       lut_nmax=LUT_NMAX), blob, lanes=case["lanes"])
        m.keygen(B, st["seed"])
        sh = [v for k, t in enumerate((X, A, mask)) for v in _shares(t, bw, seed + 3 + k)]
        m.set_inputs(B, *sh, prot)
        st["model"] = m
        return st
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if op == "gate":
        n, kind = case["n"], KINDS[case["kind"]]
        st["r"] = _rand((n,), bw, g)
        kb = lib.mpcx_tr_key_bytes(h, kind, n)
        st["k"], st["ro"], st["y"] = [_zeros(kb), _zeros(kb)], torch.zeros_like(st["r"]), torch.zeros_like(st["r"])
        st["x"] = st["r"] + _rand((n,), bw, g, span=8 << S)
    elif op == "maxpool":
        B, N, Cc = case["B"], case["N"], case["C"]
        st["r"] = _rand((B, N, Cc), bw, g)
        kb = lib.mpcx_maxpool_key_bytes(h, B, N, Cc)
        st["k"], st["ro"] = [_zeros(kb), _zeros(kb)], torch.zeros((B, Cc), dtype=st["r"].dtype, device="cuda")
        st["y"] = torch.zeros_like(st["ro"])
        st["x"] = st["r"] + _rand((B, N, Cc), bw, g, span=8 << S).clamp_(min=0)
    elif op == "mul":
        n = case["n"]
        st["ia"] = torch.arange(n, dtype=torch.int32, device="cuda")
        st["r"], st["r2"] = _rand((n,), bw, g), _rand((n,), bw, g)
        kb = lib.mpcx_mul_key_bytes(h, n, n, n)
        st["k"], st["ro"], st["y"] = [_zeros(kb), _zeros(kb)], torch.zeros_like(st["r"]), torch.zeros_like(st["r"])
        st["x"], st["x2"] = st["r"] + _rand((n,), bw, g, span=8 << S), st["r2"] + _rand((n,), bw, g, span=8 << S)
    elif op == "sxs":
        B, M, K, N = case["B"], case["M"], case["K"], case["N"]
        st["r"], st["r2"] = _rand((B, M, K), bw, g), _rand((B, K, N), bw, g)
        kb = lib.mpcx_sxs_key_bytes(h, B, M, K, N)
        st["k"], st["ro"] = [_zeros(kb), _zeros(kb)], torch.zeros((B, M, N), dtype=st["r"].dtype, device="cuda")
        st["y"] = torch.zeros_like(st["ro"])
        st["x"], st["x2"] = (st["r"] + _rand((B, M, K), bw, g, span=1 << S),
                             st["r2"] + _rand((B, K, N), bw, g, span=8 << S))
    elif op == "gemm":
        # on the CPU from the seed, so that exact() makes the same operands
        a, w = _gemm_operands(case, seed)
        t = np.int32 if bw == 32 else np.int64
        u = np.uint32 if bw == 32 else np.uint64
        st["x"], st["x2"] = (torch.from_numpy(v.astype(u).view(t)).cuda() for v in (a, w))
        st["y"] = torch.zeros((case["M"], case["N"]), dtype=st["x"].dtype, device="cuda")
    else:  # adjnorm
        B, N = case["B"], case["N"]
        ctx.set_adjnorm_lanes(case["lanes"])
        kb = lib.mpcx_adjnorm_key_bytes(h, B, N)
        st["k"] = [_zeros(kb), _zeros(kb)]
        st["ro"] = torch.zeros((B, N, N), dtype=torch.int32 if bw == 32 else torch.int64, device="cuda")
        st["y"] = torch.zeros_like(st["ro"])
        a = (torch.rand((B, N, N), device="cuda", generator=g) < 1.0 / N).to(st["ro"].dtype)  # sparse, symmetric, self loops
        a = torch.clamp(a + a.transpose(1, 2) + torch.eye(N, dtype=a.dtype, device="cuda"), max=1)
        st["x"] = _rand((B, N, N), bw, g)
        st["x2"] = a - st["x"]
    torch.cuda.synchronize()
    if case.get("dir") == "eval":  # the keys that this call spends
        _keygen(st)
        ctx.sync()
    return st


def _keygen(st):
    case, ctx, p = st["case"], st["ctx"], mpcx.dptr
    lib, h, op, (k0, k1) = ctx.lib, ctx.h, case["op"], [mpcx.dptr(k) for k in st["k"]]
    if op == "gate":
        e = lib.mpcx_tr_keygen(h, KINDS[case["kind"]], case["n"], p(st["r"]), p(st["ro"]), st["seed"], 1, k0, k1)
    elif op == "maxpool":
        e = lib.mpcx_maxpool_keygen(h, case["B"], case["N"], case["C"], p(st["r"]), p(st["ro"]), st["seed"], 1, k0, k1)
    elif op == "mul":
        n = case["n"]
        e = lib.mpcx_mul_keygen(h, n, n, n, p(st["ia"]), p(st["ia"]), p(st["r"]), p(st["r2"]), p(st["ro"]), st["seed"], 1,
                                k0, k1)
    elif op == "sxs":
        e = lib.mpcx_sxs_keygen(h, case["B"], case["M"], case["K"], case["N"], p(st["r"]), p(st["r2"]), p(st["ro"]),
                                st["seed"], 1, k0, k1)
    else:
        e = lib.mpcx_adjnorm_keygen(h, case["B"], case["N"], st["seed"], p(st["ro"]), k0, k1)
    ctx.check(e, op + " keygen")
    return [st["ro"], *st["k"]]


def run(st):
    case, ctx, p = st["case"], st["ctx"], mpcx.dptr
    lib, h, op = ctx.lib, ctx.h, case["op"]
    if op == "forward":
        st["model"].forward(case["B"])
        return st["model"].output(case["B"])
    if op == "deal":
        st["model"].keygen(case["B"], st["seed"])
        st["model"].forward(case["B"])
        return st["model"].output(case["B"])
    if op == "gemm":
        ctx.check(lib.mpcx_ring_gemm(h, case["M"], case["K"], case["N"], p(st["x"]), p(st["x2"]), p(st["y"])), "ring_gemm")
        return st["y"]
    if case["dir"] == "keygen":
        return _keygen(st)
    k0, k1 = (p(k) for k in st["k"])
    if op == "gate":
        e = lib.mpcx_tr_eval(h, KINDS[case["kind"]], case["n"], k0, k1, p(st["x"]), None, 0, p(st["y"]))
    elif op == "maxpool":
        e = lib.mpcx_maxpool_eval(h, case["B"], case["N"], case["C"], k0, k1, p(st["x"]), p(st["y"]))
    elif op == "mul":
        n = case["n"]
        e = lib.mpcx_mul_eval(h, n, n, n, p(st["ia"]), p(st["ia"]), k0, k1, p(st["x"]), p(st["x2"]), p(st["y"]))
    elif op == "sxs":
        e = lib.mpcx_sxs_eval(h, case["B"], case["M"], case["K"], case["N"], k0, k1, p(st["x"]), p(st["x2"]), p(st["y"]))
    else:
        e = lib.mpcx_adjnorm_eval(h, case["B"], case["N"], LUT_NMAX, k0, k1, p(st["x"]), p(st["x2"]), p(st["y"]))
    ctx.check(e, op + " eval")
    return st["y"]


# ---------------- the same results in plain numpy ----------------
def _gemm_operands(case, seed):
    """Masked activations (uniform in the ring) and quantised weights, as uint64."""
    rng = np.random.default_rng(seed)
    m = np.uint64((1 << case["bw"]) - 1)
    a = rng.integers(0, 1 << 64, (case["M"], case["K"]), dtype=np.uint64, endpoint=False) & m
    w = _fixed(rng.standard_normal((case["K"], case["N"])) * math.sqrt(2.0 / case["K"])).astype(np.uint64) & m
    return a, w


def _dot(a, b):
    """a @ b of small whole numbers: every partial sum below 2^53."""
    return np.rint(a.astype(np.float64) @ b.astype(np.float64)).astype(np.int64)


def _ring_dot(a, w):
    """a @ w mod 2^64 of uint64: 16-bit digits of a times small signed w."""
    w = w.astype(np.int64)
    return sum(_dot((a >> np.uint64(k)) & np.uint64(0xffff), w).astype(np.uint64) << np.uint64(k) for k in (0, 16, 32, 48))


def exact(case, seed):
    if case["op"] == "gemm":
        a, w = _gemm_operands(case, seed)
        if case["bw"] == 32:
            w = w.astype(np.uint32).view(np.int32).astype(np.int64)
            return _ring_dot(a, w.astype(np.uint64)).astype(np.uint32).view(np.int32)
        return _ring_dot(a, w).view(np.int64)
    if case["op"] not in ("forward", "deal"):
        return None  # masked by the dealer's randomness, or its keys
    X, A, mask, prot, W = _model_inputs(case, seed)
    d = A.sum(2)
    T = np.zeros(256, np.int64)
    T[1:LUT_NMAX + 1] = [int(math.floor((1 << S) / math.sqrt(k) + 0.5)) for k in range(1, LUT_NMAX + 1)]
    t = T[d]
    An = A * ((t[:, :, None] * t[:, None, :]) >> S)
    H = X
    for w, b in W[:3]:
        H = np.maximum((_dot(An, _dot(H, w) >> S) >> S) + b, 0)
    v = np.where(mask[:, :, None] == 1, H, -1).max(1)
    v = np.maximum((_dot(v, W[3][0]) >> S) + W[3][1], 0)
    v = (_dot(v, W[4][0]) >> S) + W[4][1]
    v = np.concatenate([v, prot], 1)
    for w, b in W[5:-1]:
        v = np.maximum((_dot(v, w) >> S) + b, 0)
    return ((_dot(v, W[-1][0]) >> S) + W[-1][1]).reshape(-1)


def tolerance(case):
    return "exact"


# ---------------- work ----------------
AES_OPS = 10 * 16 * 2  # one AES-128 call: 16 byte substitutions and 16 word or byte XORs in each of 10 rounds


def _dcf_bits(kind, bw):
    """Widths of a gate kind's comparisons."""
    return {"TR": (bw - 1, S), "TRRELU": (bw - 1, S), "RELU": (bw - 1,), "TRSLACK": (S,), "TRMOD": (S,),
            "EXT": (bw - S - 1,), "EXTRELU": (bw - S - 1,), "RELUPOOL": (bw - S,)}[kind]


def _gate(kind, n, bw, direction):
    """Bytes and operations of a gate over n elements, both parties: an
    evaluation reads each comparison's correction words and leaf once (they are
    the same in both keys), both roots and one table word and (ReLU) one share
    per party; a dealer writes both keys whole."""
    T = bw // 8
    aes = [max(m - 7, 0) + 1 for m in _dcf_bits(kind, bw)]
    relu = "RELU" in kind
    if direction == "eval":
        b = sum(16 * a + 2 * 16.125 for a in aes) + 2 * T * (1 + relu) + 2 * T
        return n * b, n * 2 * sum(aes) * AES_OPS
    cases = {"TR": 8, "TRRELU": 8, "EXT": 4, "EXTRELU": 4, "TRSLACK": 8}.get(kind, 2)
    b = 2 * (sum(16 * a + 16.125 for a in aes) + T * (cases + relu)) + 2 * T
    # both walks, and per element the drawn roots and mask bits, table words, share and output mask
    return n * b, n * (2 * sum(aes) + 4 * len(aes) + cases + relu + 1) * AES_OPS


def _ring_macs(bw):
    """8-bit products of one ring multiply-add: the digit pairs that reach the result."""
    return 10 if bw == 32 else 36


def _adjnorm(B, N, bw, direction):
    T, P = bw // 8, N * (N + 1) // 2
    b, f = _gate("TRSLACK", B * P, bw, direction)
    # A's reveal and product, the degrees' table, the outer product over the triangle
    b += 2 * T * (4 * B * N * N + 3 * B * P + 6 * B * N) + 2 * 48 * B * N
    f += B * N * (6 if direction == "eval" else 13) * AES_OPS
    f += (8 * B * (N * N + P) if direction == "eval" else (4 * B * N * N + 3 * B * P) * AES_OPS)
    return b, f


def _pairs(N):
    out = []
    while N > 1:
        out.append(N // 2)
        N = N // 2 + N % 2
    return out


def _maxpool(kind, B, N, C, bw, direction):
    r = [_gate(kind, B * p * C, bw, direction) for p in _pairs(N)]
    return sum(x[0] for x in r) + B * (N + 1) * C * bw // 8, sum(x[1] for x in r)


def _sxs(B, M, K, N, bw, direction):
    T = bw // 8
    a, b, c = B * M * K, B * K * N, B * M * N
    if direction == "eval":
        return T * (3 * (a + b + c)), 2 * 3 * B * M * K * N * _ring_macs(bw)
    return T * (3 * (a + b + c)), 2 * 2 * B * M * K * N * _ring_macs(bw) + (a + b + 2 * c) * AES_OPS


def _forward(B, bw, direction):
    T, R = bw // 8, B * N_NODES
    parts = [_adjnorm(B, N_NODES, bw, direction)]
    io = _layers()
    for i, o in io[:3]:
        parts += [_gemm(R, i, o, bw), _gate("TRMOD", R * o, bw, direction), _gate("EXT", R * o, bw, direction),
                  _sxs(B, N_NODES, N_NODES, o, bw, direction), _gate("TRMOD", R * o, bw, direction),
                  _gate("EXTRELU", R * o, bw, direction)]
    parts.append(_maxpool("RELUPOOL", B, N_NODES, GCN[2], bw, direction))
    for i, o in io[3:]:
        parts.append(_gemm(B, i, o, bw))
        if o > 1:
            parts += [_gate("TRMOD", B * o, bw, direction), _gate("EXTRELU", B * o, bw, direction)]
    return sum(x[0] for x in parts) + T * R * (2 * FEAT + 2), sum(x[1] for x in parts)


def _gemm(M, K, N, bw):
    return bw // 8 * (M * K + K * N + M * N), 2 * M * K * N * _ring_macs(bw)


def work(case):
    op, bw, d = case["op"], case["bw"], case.get("dir")
    if op == "forward":
        b, f = _forward(case["B"], bw, "eval")
    elif op == "deal":
        b, f = (sum(v) for v in zip(_forward(case["B"], bw, "keygen"), _forward(case["B"], bw, "eval")))
    elif op == "gate":
        b, f = _gate(case["kind"], case["n"], bw, d)
    elif op == "adjnorm":
        b, f = _adjnorm(case["B"], case["N"], bw, d)
    elif op == "maxpool":
        b, f = _maxpool("RELU", case["B"], case["N"], case["C"], bw, d)
    elif op == "mul":
        n, T = case["n"], bw // 8
        b, f = (n * (9 * T + 8), 8 * n) if d == "eval" else (n * (9 * T + 8), 4 * n * AES_OPS)
    elif op == "sxs":
        b, f = _sxs(case["B"], case["M"], case["K"], case["N"], bw, d)
    else:
        b, f = _gemm(case["M"], case["K"], case["N"], bw)
    return {"bytes": float(b), "flops": float(f)}
