"""Performance cases: what users of this library run, through its plans.

A case is one pass of one operator (or of a stack of calls: the layers of a
model, the heads of an attention layer):

  spmm       C = A * B          forward of a block-sparse layer
  sddmm      mask (.) (X * Y)   sampled scores, and the gradient of a sparse
                                layer's block values (X = dC, Y = B^T as stored)
  attention  the fused pair bf16(mask (.) (Q * K^T)) * V, one call per head
  spgemm     C = A * B, all BSR

Plans are made once in prepare(), as a program keeps them.  Where a program
would replay its launches (`graph`), the stack's calls are captured in a HIP
graph; otherwise run() makes the calls one by one.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()
capi, W = pkg.capi, pkg.workloads


def listed():
    return [
        # One small layer called on its own: launch and host latency.
        dict(name="spmm_small", op="spmm", H=1024, W=1024, R=32, C=32, pattern="random", density=0.10, N=256,
             out="f32", calls=1, graph=False),
        # Decode: a batch of 32 tokens through eight pruned projections of
        # ragged size, replayed as a graph.
        dict(name="spmm_decode", op="spmm", H=4128, W=3104, R=32, C=32, pattern="random", density=0.08, N=32,
             out="bf16", calls=8, graph=True),
        # Prefill: four 25% dense layers on 512 tokens (the density sweep's
        # shape), replayed as a graph.
        dict(name="spmm_layers", op="spmm", H=4096, W=4096, R=32, C=32, pattern="random", density=0.25, N=512,
             out="f32", calls=4, graph=True),
        # A large matrix with a skewed row distribution (the benchmark's headline).
        dict(name="spmm_skewed", op="spmm", H=16384, W=16384, R=32, C=32, pattern="zipf", density=0.02, N=1024,
             out="f32", calls=1, graph=False),
        # Middle-sized blocks, non-square matrix, a long batch.
        dict(name="spmm_blocks64", op="spmm", H=8192, W=6144, R=64, C=64, pattern="random", density=0.10, N=2048,
             out="bf16", calls=1, graph=False),
        # The reference's own configuration: 8192^3, 256 x 256 blocks, 25%.
        dict(name="spmm_blocks256", op="spmm", H=8192, W=8192, R=256, C=256, pattern="random", density=0.25, N=8192,
             out="bf16", calls=1, graph=False),
        # Sampled scores: the benchmark's SDDMM, four layers as a graph.
        dict(name="sddmm_scores", op="sddmm", H=4096, W=4096, R=32, C=32, pattern="random", density=0.10, K=256,
             y="row", out="f32", calls=4, graph=True),
        # Backward of one of spmm_layers' layers: dA = (dC * B^T) at A's blocks.
        dict(name="sddmm_weight_grad", op="sddmm", H=4096, W=4096, R=32, C=32, pattern="random", density=0.25, K=512,
             y="col", out="f32", calls=1, graph=False),
        # The reference's SDDMM configuration: 8192^3, 256 x 256 blocks, 25%.
        dict(name="sddmm_blocks256", op="sddmm", H=8192, W=8192, R=256, C=256, pattern="random", density=0.25, K=8192,
             y="row", out="bf16", calls=1, graph=False),
        # Long-sequence attention, eight heads: 8 causal block diagonals plus
        # 1% global blocks, the heads side by side in token-major Q, K and V.
        dict(name="attention_heads", op="attention", seq=8192, R=32, bands=8, glob=0.01, d=128, out="bf16", calls=8,
             graph=True),
        # Sparse times sparse with small blocks (the benchmark's) ...
        dict(name="spgemm_blocks32", op="spgemm", H=8192, W=8192, V=8192, R=32, C=32, BC=32, density=0.05, out="f32",
             calls=1, graph=False),
        # ... and with large ones.
        dict(name="spgemm_blocks128", op="spgemm", H=4096, W=4096, V=4096, R=128, C=128, BC=128, density=0.25,
             out="bf16", calls=1, graph=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """A case of the same ranges, at most about 1/3 of the largest listed one's
    work (its kernels may be the less tuned ones)."""
    while True:
        op = rng.choice(["spmm", "spmm", "spmm", "sddmm", "sddmm", "attention", "attention", "spgemm"])
        out = rng.choice(["f32", "bf16"])
        calls = rng.choice([1, 1, 2, 4, 8])
        graph = calls > 1 and rng.random() < 0.7
        R, C = rng.choice([(32, 32), (32, 32), (64, 64), (128, 128), (256, 256), (64, 32), (32, 64), (128, 64)])
        H, Wd = (max(1, round(_log(rng, 1024, 16384) / b)) * b for b in (R, C))
        density = round(_log(rng, 0.01, 0.5), 4)
        c = dict(op=op, H=H, W=Wd, R=R, C=C, density=density, out=out, calls=calls, graph=graph)
        if op == "spmm":
            c["pattern"] = "zipf" if R == 32 and C == 32 and density <= 0.05 and rng.random() < 0.3 else "random"
            c["N"] = 32 * round(_log(rng, 1, 256))
        elif op == "sddmm":
            c["pattern"], c["y"] = "random", rng.choice(["row", "col"])
            c["K"] = 32 * round(_log(rng, 1, 256))
        elif op == "spgemm":
            c["BC"] = rng.choice([R, C, 32])
            c["V"] = max(1, round(_log(rng, 1024, 8192) / c["BC"])) * c["BC"]
            if H * c["V"] > 8192 * 8192 or H * Wd > 8192 * 8192:
                continue
        else:
            b = rng.choice([32, 32, 64, 128])
            c = dict(op=op, seq=b * round(_log(rng, 1024, 16384) / b), R=b, bands=rng.choice([2, 4, 8, 16]),
                     glob=round(_log(rng, 0.002, 0.05), 4), d=rng.choice([32, 64, 128]), out=out, calls=calls,
                     graph=graph)
            if c["bands"] * b >= c["seq"]:
                continue
        w = work(c)
        if max(w["bytes"], w["flops"] / 50) <= 2e9 and 1e6 <= w["bytes"] <= 1e9:
            return c


# ---------------------------------------------------------------------------
# Structures (numpy, seeded) and values (torch on the GPU, seeded).
def _random(H, Wd, R, C, density, rng):
    return W.random_positions(H, Wd, R, C, max(1, round(density * (H // R) * (Wd // C))), rng)


def _zipf(H, Wd, R, C, density, rng):
    """Zipf(1.2) blocks per block row, capped at 512."""
    nbr, nbc = H // R, Wd // C
    counts = W.zipf_row_counts(nbr, nbc, density, 1.2, min(512, nbc), rng)
    indptr = np.zeros(nbr + 1, np.int32)
    np.cumsum(counts, out=indptr[1:])
    cols = [np.sort(rng.choice(nbc, size=int(n), replace=False)) for n in counts]
    return W.BsrArrays(H, Wd, R, C, indptr, np.concatenate(cols).astype(np.int32))


def _structures(case, seed):
    """Per call: (A or mask,), or (A, B) for spgemm.  The heads of an
    attention layer share one mask.  spgemm's do not depend on the seed: its
    output's size comes from them."""
    op = case["op"]
    rng = np.random.default_rng([0 if op == "spgemm" else int(seed), 17])
    if op == "attention":
        m = W.band_global_mask(case["seq"], case["R"], case["bands"], case["glob"], rng)
        return [(m,)] * case["calls"]
    got = []
    for _ in range(case["calls"]):
        if op == "spgemm":
            got.append((_random(case["H"], case["W"], case["R"], case["C"], case["density"], rng),
                        _random(case["W"], case["V"], case["C"], case["BC"], case["density"], rng)))
        else:
            make = _zipf if case["pattern"] == "zipf" else _random
            got.append((make(case["H"], case["W"], case["R"], case["C"], case["density"], rng),))
    return got


def _inputs(case, structures, seed):
    """Operand tensors per call (bf16): weights and activations U[-1, 1],
    scores' operands normal, attention Q, K, V normal with std d^-1/2; masks 1."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    op = case["op"]

    def uniform(*shape):
        return torch.empty(shape, device="cuda").uniform_(-1, 1, generator=g).bfloat16()

    def normal(*shape, std=1.0):
        return torch.empty(shape, device="cuda").normal_(0, std, generator=g).bfloat16()

    def blocks(s):
        return s.nblocks * s.R * s.C

    if op == "attention":
        (m,), heads, d = structures[0], case["calls"], case["d"]
        q, k, v = (normal(case["seq"], heads * d, std=d ** -0.5) for _ in range(3))
        ones = torch.ones(blocks(m), device="cuda", dtype=torch.bfloat16)
        return [(ones, *(t[:, h * d:(h + 1) * d] for t in (q, k, v))) for h in range(heads)]
    got = []
    for s in structures:
        if op == "spmm":
            got.append((uniform(blocks(s[0])), uniform(case["W"], case["N"])))
        elif op == "sddmm":
            y = (case["K"], case["W"]) if case["y"] == "row" else (case["W"], case["K"])
            got.append((torch.ones(blocks(s[0]), device="cuda", dtype=torch.bfloat16), normal(case["H"], case["K"]),
                        normal(*y)))
        else:
            got.append((uniform(blocks(s[0])), uniform(blocks(s[1]))))
    return got


def _bsr(s):
    return capi.Bsr(s.H, s.W, s.R, s.C, s.indptr, s.indices)


class State:
    """Plans, operands and outputs of a case's calls, and their graph."""

    def __init__(self, case, seed):
        structures = _structures(case, seed)
        self.inputs = _inputs(case, structures, seed)
        self.graph = None
        op, out = case["op"], case["out"]
        dtype = torch.float32 if out == "f32" else torch.bfloat16
        if op == "attention":
            self.plans = [capi.AttentionPlan(_bsr(structures[0][0]), case["d"], out)] * case["calls"]
            self.result = torch.empty(case["seq"], case["calls"] * case["d"], device="cuda", dtype=dtype)
            self.outputs = [self.result[:, h * case["d"]:(h + 1) * case["d"]] for h in range(case["calls"])]
        else:
            if op == "spmm":
                self.plans = [capi.SpmmPlan(_bsr(a), case["N"], out) for a, in structures]
                shapes = [(case["H"], case["N"])] * case["calls"]
            elif op == "sddmm":
                layout = capi.ROW_MAJOR if case["y"] == "row" else capi.COL_MAJOR
                self.plans = [capi.SddmmPlan(_bsr(m), case["K"], layout, out) for m, in structures]
                shapes = [(m.nblocks * m.R * m.C,) for m, in structures]
            else:
                self.plans = [capi.SpgemmPlan(_bsr(a), _bsr(b), out) for a, b in structures]
                shapes = [(p.out_values,) for p in self.plans]
            self.result = self.outputs = [torch.empty(s, device="cuda", dtype=dtype) for s in shapes]
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                self.launch()
            torch.cuda.current_stream().wait_stream(side)
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph, stream=side):
                self.launch()

    def launch(self):
        stream = torch.cuda.current_stream().cuda_stream
        for plan, operands, out in zip(self.plans, self.inputs, self.outputs):
            plan.run(*operands, out, stream=stream)


def prepare(case, seed):
    return State(case, seed)


def run(state):
    if state.graph is not None:
        state.graph.replay()
    else:
        state.launch()
    return state.result


# ---------------------------------------------------------------------------
def work(case):
    """Bytes: each operand's values and index arrays read once, the output
    written once.  Flops: the products of stored blocks (spgemm: the expected
    number of pairs and of output blocks of uniform positions)."""
    op, R, so = case["op"], case["R"], 4 if case["out"] == "f32" else 2
    if op == "attention":
        nb, d = case["seq"] // R, case["d"]
        band = sum(nb - o for o in range(min(case["bands"], nb)))
        n = band + round(case["glob"] * nb * nb)
        head = 3 * 2 * case["seq"] * d + so * case["seq"] * d
        mask = 2 * n * R * R + 4 * (n + nb + 1)
        return {"bytes": case["calls"] * head + mask, "flops": case["calls"] * 4.0 * n * R * R * d}
    C, H, Wd = case["C"], case["H"], case["W"]
    n = max(1, round(case["density"] * (H // R) * (Wd // C)))
    a = 2 * n * R * C + 4 * (n + H // R + 1)
    if op == "spmm":
        b, f = 2 * Wd * case["N"] + so * H * case["N"], 2.0 * n * R * C * case["N"]
    elif op == "sddmm":
        b, f = 2 * (H + Wd) * case["K"] + so * n * R * C, 2.0 * n * R * C * case["K"]
    else:
        BC, V = case["BC"], case["V"]
        m = max(1, round(case["density"] * (Wd // C) * (V // BC)))
        pairs = n * m / (Wd // C)
        cells = (H // R) * (V // BC)
        stored = cells * (1 - math.exp(-pairs / cells))
        b, f = 2 * m * C * BC + 4 * m + so * stored * R * BC, 2.0 * pairs * R * C * BC
    return {"bytes": case["calls"] * (a + b), "flops": case["calls"] * f}


def tolerance(case):
    """About four times the error measured against exact(): bf16 outputs 1.7e-3
    (their rounding); f32 outputs 0.5e-7 to 2.2e-7 up to K = 16384 sums, more
    for the longest; attention in f32 1.7e-5 (scores that round the other way,
    each up to 2^-8 of itself, which a row of few keys shows in one value)."""
    if case["out"] == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1e-4, "max": 2e-2} if case["op"] == "attention" else {"rel": 2e-6}


# ---------------------------------------------------------------------------
def _dense(s, values):
    """The dense matrix of a BSR one, in 64 bits."""
    nbr, nbc = s.H // s.R, s.W // s.C
    at = torch.from_numpy(s.block_rows().astype(np.int64) * nbc + s.indices).cuda()
    d = torch.zeros(nbr * nbc, s.R, s.C, device="cuda", dtype=torch.float64)
    d.index_add_(0, at, values.double().view(-1, s.R, s.C))
    return d.view(nbr, nbc, s.R, s.C).transpose(1, 2).reshape(s.H, s.W)


def _blocks(d, rows, cols, R, C):
    """The R x C blocks of a dense matrix at the given block positions, flat."""
    t = d.view(d.shape[0] // R, R, d.shape[1] // C, C).transpose(1, 2)
    rows, cols = (torch.as_tensor(np.asarray(v, np.int64)).cuda() for v in (rows, cols))
    return t[rows, cols].reshape(-1)


def exact(case, seed):
    structures = _structures(case, seed)
    inputs = _inputs(case, structures, seed)
    got = []
    for s, x in zip(structures, inputs):
        if case["op"] == "spmm":
            got.append(_dense(s[0], x[0]) @ x[1].double())
        elif case["op"] == "sddmm":
            m, y = s[0], x[2].double()
            d = x[1].double() @ (y if case["y"] == "row" else y.T.contiguous())
            got.append(_blocks(d, m.block_rows(), m.indices, m.R, m.C) * x[0].double())
        elif case["op"] == "attention":
            # The scores are bf16 by the operator's definition.
            sc = (x[1].double() @ x[2].double().T.contiguous() * _dense(s[0], x[0])).bfloat16().double()
            got.append(sc @ x[3].double())
        else:
            a, b = s
            pa, pb = (torch.zeros(t.H // t.R, t.W // t.C, device="cuda") for t in s)
            for p, t in ((pa, a), (pb, b)):
                p[torch.from_numpy(t.block_rows().astype(np.int64)), torch.from_numpy(t.indices.astype(np.int64))] = 1
            at = (pa @ pb > 0.5).nonzero().cpu().numpy()
            got.append(_blocks(_dense(a, x[0]) @ _dense(b, x[1]), at[:, 0], at[:, 1], a.R, b.C))
    return torch.cat(got, dim=1) if case["op"] == "attention" else got
