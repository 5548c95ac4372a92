"""Performance cases: the optimizer steps and Newton-Schulz calls that a training program makes, over their range.

Three kinds of program are covered, each through the package's public entry points:

  * "muon" / "dion": `Muon.step()` / `Dion.step()` over the matrices of a stack of transformer layers.  A layer has
    the query and output projections (d x d), the key and value projections (kv x d), one or two up projections
    (ff x d) and one down projection (d x ff).  With `vocab` > 0 the optimizer also holds the other parameters of the
    model, in the groups of an ordinary training script: embedding and lm_head (Lion), gains and biases (AdamW).
  * "scalar": the element-wise groups alone: embedding and gains (Lion), lm_head (AdamW).
  * "ns": one call of `zeropower_via_newtonschulz5` on a matrix or a batch of matrices.

The optimizers are in the middle of a run: momentum, variance and Q hold what earlier steps leave, gradients are there.
"""
import math

import torch

from dion_amd import Dion, DionMixedPrecisionConfig, Muon, zeropower_via_newtonschulz5

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
LR, MU, WD = 0.02, 0.95, 0.01


def listed():
    return [
        # One orthogonalisation of a small matrix by hand (a custom update rule, a test, a notebook): pure latency.
        dict(name="ns_one_small", path="ns", batch=1, rows=256, cols=768, dtype="fp32"),
        # The same call on the largest matrix of a Llama-3-8B layer.
        dict(name="ns_one_4096x14336", path="ns", batch=1, rows=4096, cols=14336, dtype="bf16"),
        # A small model trained in fp32 with all its parameters in one optimizer: many small calls, host time counts.
        dict(name="muon_small_model", path="muon", layers=4, d=256, kv=256, ff=1024, up=1, attention=True, vocab=4096,
             dtype="fp32"),
        # All matrices of GPT-small, bf16: the headline workload of the benchmark.
        dict(name="muon_gpt_small", path="muon", layers=12, d=768, kv=768, ff=3072, up=1, attention=True, vocab=0,
             dtype="bf16"),
        # Widths off every alignment grid (pruned models, odd heads and hidden sizes), fp32 weights.
        dict(name="muon_odd_widths", path="muon", layers=2, d=1021, kv=341, ff=2731, up=2, attention=True, vocab=0,
             dtype="fp32"),
        # One Llama-3-8B layer, bf16: large matrices, bound by the matrix products.
        dict(name="muon_llama8b_layer", path="muon", layers=1, d=4096, kv=1024, ff=14336, up=2, attention=True,
             vocab=0, dtype="bf16"),
        # The small model again under Dion, fp32 states, rank fraction 1/2.
        dict(name="dion_small_model", path="dion", layers=4, d=256, kv=256, ff=1024, up=1, attention=True, vocab=4096,
             dtype="fp32", rank_fraction=0.5),
        # GPT-small under low-rank Dion (bf16 weights and momentum, fp32 Q).
        dict(name="dion_gpt_small_r025", path="dion", layers=12, d=768, kv=768, ff=3072, up=1, attention=True, vocab=0,
             dtype="bf16", rank_fraction=0.25),
        # The same at full rank, the optimizer's default rank fraction.
        dict(name="dion_gpt_small_r1", path="dion", layers=12, d=768, kv=768, ff=3072, up=1, attention=True, vocab=0,
             dtype="bf16", rank_fraction=1.0),
        # Odd widths under Dion: the rank is odd as well.
        dict(name="dion_odd_widths", path="dion", layers=2, d=1021, kv=341, ff=2731, up=2, attention=True, vocab=0,
             dtype="bf16", rank_fraction=0.25),
        # The MLP matrices of one Llama-3-70B layer at rank 512: the largest single matrices.
        dict(name="dion_llama70b_layer", path="dion", layers=1, d=8192, kv=0, ff=28672, up=2, attention=False, vocab=0,
             dtype="bf16", rank_fraction=1.0 / 16),
        # The element-wise groups of GPT-small: bound by memory.
        dict(name="scalar_gpt_small", path="scalar", vocab=50304, d=768, gains=25, dtype="bf16"),
    ]


def _size(rng, lo, hi):
    """A dimension, log-uniform over [lo, hi]: most often on a grid that models use, sometimes odd."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice((128, 64, 64, 8, 1, 1))
    if step > 1:
        return max(lo, v // step * step)
    return min(hi, v | 1)


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 200)


def draw(rng):
    path = rng.choice(("ns", "muon", "muon", "muon", "dion", "dion", "dion", "scalar"))
    most = max(_cost(c) for c in listed() if c["path"] == path)
    while True:
        dtype = rng.choice(("bf16", "bf16", "fp32"))
        if path == "ns":
            case = dict(path=path, batch=rng.choice((1, 1, 2, 4, 16)), rows=_size(rng, 64, 8192),
                        cols=_size(rng, 64, 14336), dtype=dtype)
        elif path == "scalar":
            case = dict(path=path, vocab=_size(rng, 1000, 130000), d=_size(rng, 128, 4096),
                        gains=rng.randint(1, 60), dtype=dtype)
        else:
            d = _size(rng, 128, 4096)
            kv = rng.choice((d, d, max(8, d // 4), max(8, d // 3)))
            ff = min(_size(rng, 2 * d, 4 * d), 4 * d)
            layers = max(1, int(round(math.exp(rng.uniform(0, math.log(12))))))
            vocab = rng.choice((0, 0, _size(rng, 1000, 50000)))
            case = dict(path=path, layers=layers, d=d, kv=kv, ff=ff, up=rng.choice((1, 2)),
                        attention=rng.random() < 0.8, vocab=vocab, dtype=dtype)
            if path == "dion":
                # Full rank belongs to small models: its cost grows with the cube of the width.
                case["rank_fraction"] = rng.choice((1.0 / 16, 0.125, 0.25, 0.5, 1.0) if d <= 1024
                                                   else (1.0 / 16, 0.125, 0.25))
                if dtype == "fp32" and d > 2048:
                    continue
        if _cost(case) <= most:
            return case


def _shapes(case):
    """(shape, count) of the matrices of the stack."""
    d, kv, ff, layers = case["d"], case["kv"], case["ff"], case["layers"]
    count = {}
    if case["attention"]:
        for s in ((d, d), (d, d), (kv, d), (kv, d)):
            count[s] = count.get(s, 0) + layers
    for s in ((ff, d),) * case["up"] + ((d, ff),):
        count[s] = count.get(s, 0) + layers
    return list(count.items())


def _others(case):
    """(name, algorithm, shape, count) of the parameters that are no matrices of the stack."""
    d, ff = case["d"], case.get("ff")
    if case["path"] == "scalar":
        return [("embedding", "lion", (case["vocab"], d), 1), ("gains", "lion", (d,), case["gains"]),
                ("lm_head", "adamw", (case["vocab"], d), 1)]
    if not case["vocab"]:
        return []
    return [("embedding", "lion", (case["vocab"], d), 1), ("lm_head", "lion", (case["vocab"], d), 1),
            ("gains", "adamw", (d,), 2 * case["layers"] + 1), ("biases", "adamw", (ff,), case["layers"])]


def _rank(case, m, n):
    return min(math.ceil(case["rank_fraction"] * min(m, n)), m, n)


def _buffer(shape, count):
    """Storage of `count` tensors of one shape, each at an aligned address like an allocation of its own."""
    n = math.prod(shape)
    return (count, -(-n // 256) * 256), n


class _Maker:
    """Draws the tensors of one state from its seed, on the GPU; keeps the updated ones, by name, for the result."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.out = {}

    def draw(self, shape, count, dtype, std, keep=None, square=False):
        full, n = _buffer(shape, count)
        buf = torch.randn(full, generator=self.gen, device="cuda", dtype=dtype).mul_(std)
        if square:
            buf.square_()
        if keep:
            self.out[keep] = buf[:, :n]
        return [row[:n].view(shape) for row in buf]


def prepare(case, seed):
    mk = _Maker(seed)
    dtype = DTYPES[case["dtype"]]
    if case["path"] == "ns":
        batch, m, n = case["batch"], case["rows"], case["cols"]
        shape = (m, n) if batch == 1 else (batch, m, n)
        return dict(ns=torch.randn(shape, generator=mk.gen, device="cuda", dtype=dtype))

    groups, state, grads = [], {}, []

    def parameters(name, shape, count, **states):
        xs = mk.draw(shape, count, dtype, 0.02, keep=name + ".x")
        gs = mk.draw(shape, count, dtype, 1e-3)
        params = [torch.nn.Parameter(x) for x in xs]
        for p, g in zip(params, gs):
            p.grad = g
        for p, *values in zip(params, *states.values()):
            state[p] = dict(zip(states, values))
        return params

    matrices = []
    for shape, count in _shapes(case) if case["path"] != "scalar" else ():
        name = "%dx%d" % shape
        # gradients of N(0, 1e-6) under momentum 0.95: N(0, 1e-6 / (1 - 0.95^2)) after many steps
        states = dict(momentum=mk.draw(shape, count, dtype, 3.2e-3, keep=name + ".momentum"))
        if case["path"] == "dion":
            m, n = shape
            r = _rank(case, m, n)
            qdtype = torch.float32
            qs = mk.draw((m if m < n else n, r), count, qdtype, 1.0, keep=name + ".q")
            for q in qs:
                q.div_(q.norm(dim=0, keepdim=True))
            states["Q"] = qs
        matrices += parameters(name, shape, count, **states)
    if matrices:
        groups.append(dict(params=matrices))
    for name, algorithm, shape, count in _others(case):
        states = dict(momentum=mk.draw(shape, count, dtype, 3e-4, keep=name + ".momentum"))
        if algorithm == "adamw":
            states["variance"] = mk.draw(shape, count, dtype, 1e-3, keep=name + ".variance", square=True)
        groups.append(dict(params=parameters(name, shape, count, **states), algorithm=algorithm, lr=1e-3))

    if case["path"] == "dion":
        config = DionMixedPrecisionConfig(momentum_dtype=dtype, Q_dtype=torch.float32)
        opt = Dion(groups, lr=0.01, mu=MU, weight_decay=WD, rank_fraction=case["rank_fraction"],
                   mixed_precision_config=config)
    else:
        opt = Muon(groups, lr=LR, mu=MU, weight_decay=WD, nesterov=True, adjust_lr="spectral_norm")
    for p, st in state.items():
        opt.state[p] = st
    for g in opt.param_groups:
        g["step"] = 500
    return dict(opt=opt, out=mk.out)


def run(state):
    if "ns" in state:
        return zeropower_via_newtonschulz5(state["ns"])
    state["opt"].step()
    return state["out"]


def work(case):
    """Every tensor read once and written once where it changes; products counted once, symmetric ones by half."""
    size = DTYPES[case["dtype"]].itemsize
    nbytes = flops = 0

    def newton_schulz(m, n):
        m, n = min(m, n), max(m, n)
        return 5 * (3 * m * m * n + m**3)

    if case["path"] == "ns":
        elements = case["batch"] * case["rows"] * case["cols"]
        return dict(bytes=elements * (size + 2), flops=case["batch"] * newton_schulz(case["rows"], case["cols"]))
    for (m, n), count in _shapes(case) if case["path"] != "scalar" else ():
        nbytes += count * 5 * m * n * size   # weights and momentum read and written, gradients read
        if case["path"] == "muon":
            flops += count * newton_schulz(m, n)
        else:
            r, long, short = _rank(case, m, n), max(m, n), min(m, n)
            nbytes += count * 2 * short * r * 4
            # four products over the matrix, the Gram matrix and the triangular solve, the factorisation
            flops += count * (8 * m * n * r + 2 * long * r * r + r**3 // 3)
    for _, algorithm, shape, count in _others(case):
        elements = count * math.prod(shape)
        nbytes += elements * size * (7 if algorithm == "adamw" else 5)
        flops += elements * (16 if algorithm == "adamw" else 8)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """Newton-Schulz computes in bf16 whatever its input: its result is good to 1e-2 of its norm.  A Muon step adds it,
    scaled by the learning rate, to the weights: bf16 weights show their own rounding, fp32 ones 1e-2 of an update that
    is a few per cent of the weights.  Dion in fp32 is fp32 throughout; in bf16 its factors are rounded to bf16.  At full
    rank the condition of a square factor multiplies the rounding."""
    if case["path"] == "ns":
        return {"rel": 1e-2}
    if case["path"] == "muon":
        return {"rel": 4e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
    if case["path"] == "dion":
        full = case["rank_fraction"] == 1.0
        if case["dtype"] == "bf16":
            return {"rel": 2e-2 if full else 1e-2}
        return {"rel": 5e-3 if full else 3e-4}
    return {"rel": 4e-3} if case["dtype"] == "bf16" else {"rel": 1e-5}
