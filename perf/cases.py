"""The work that a user of cubework_amd has it do, as cases that can be timed and compared.

A training program built on the tensor-parallel layers spends its time in decoder blocks (forward and backward), in
single layers of a larger grid whose peers' operands have arrived, in the vocabulary-parallel embedding, head and loss,
and in clipping the gradients; an evaluation loop runs the block forward alone. The listed cases take each of these at
a size it really has, from one short sequence to the OPT-1.3B-shaped block at 8192 tokens, in the types that are used
(bf16 and fp16 parameters, fp32 parameters under autocast, plain fp32) and with the ragged sizes that data brings along:
sequence lengths that are no multiple of anything, head sizes of 48 and 80, vocabularies of 50257 and 50272 / 4.

Kinds, each through the public layers or operators:
  step       OPTBlock, forward + backward: every parameter's gradient and the input's
  eval       OPTBlock under no_grad
  linear     Linear2D / Linear1D_Col, forward + backward; grid = 2 is rank (0, 1) of a 2 x 2 grid with its peers'
             operands staged as a broadcast would deliver them
  norm       LayerNorm2D, forward + backward; grid as for linear
  loss       VocabParallelCrossEntropyLoss1D as rank 1 of `ranks` slices (rank 0 of 1), forward + backward
  head       VocabParallelClassifier1D and its loss, forward + backward
  embed      vocabulary slice lookup and its gradient, rank 1 of `ranks`
  clip       clip_grad_norm over the gradients of `layers` blocks
"""
import math

import torch

from cubework_amd import ops
from cubework_amd.clip_grad import clip_grad_norm
from cubework_amd.distributed import ParallelManager as pm
from cubework_amd.distributed import initialize
from cubework_amd.module.loss import VocabParallelCrossEntropyLoss1D
from cubework_amd.module.parallel_1d import Linear1D_Col, VocabParallelClassifier1D
from cubework_amd.module.parallel_2d import LayerNorm2D, Linear2D
from cubework_amd.opt_block import OPTBlock

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
#: (hidden, heads) of the models the layers are used for (feed-forward 4 x hidden); head sizes 48, 64, 80 and 128
WIDTHS = ((768, 16), (1024, 16), (2048, 32), (2560, 32), (4096, 32))
#: vocabularies: OPT's table, its slices, GPT-2's (odd), a small one
VOCABS = (50272, 50257, 12568, 32000, 1000)


def listed():
    return [
        # one short sequence through the smallest model's block (head size 48): a step made of launches, not of arithmetic
        {"name": "step_768_1x128_bf16", "kind": "step", "hidden": 768, "heads": 16, "batch": 1, "seq": 128, "dtype": "bf16",
         "act": "relu"},
        # the way the training scripts run: fp32 parameters and residual stream, fp16 products under autocast
        {"name": "step_1024_8x512_autocast", "kind": "step", "hidden": 1024, "heads": 16, "batch": 8, "seq": 512,
         "dtype": "autocast", "act": "gelu_tanh"},
        # head size 80 and a batch whose longest sequence is odd
        {"name": "step_2560_2x777_bf16", "kind": "step", "hidden": 2560, "heads": 32, "batch": 2, "seq": 777, "dtype": "bf16",
         "act": "relu"},
        # the OPT-1.3B-shaped block at its training batch: the largest step
        {"name": "step_2048_4x2048_bf16", "kind": "step", "hidden": 2048, "heads": 32, "batch": 4, "seq": 2048, "dtype": "bf16",
         "act": "relu"},
        # evaluation of one prompt with the widest block (head size 128): forward only
        {"name": "eval_4096_1x300_bf16", "kind": "eval", "hidden": 4096, "heads": 32, "batch": 1, "seq": 300, "dtype": "bf16",
         "act": "relu"},
        # one rank of a 2 x 2 SUMMA grid: two k-steps of [8192, 2048] x [2048, 2048] forward, the gradients' products backward
        {"name": "linear2d_grid_8192_bf16", "kind": "linear", "grid": 2, "rows": 8192, "in": 4096, "out": 4096, "dtype": "bf16",
         "act": "gelu_tanh"},
        # a column-parallel layer in fp32, where parity with the CPU path is held to 1e-5
        {"name": "linear1d_4096_fp32", "kind": "linear", "grid": 0, "rows": 4096, "in": 1024, "out": 4096, "dtype": "fp32",
         "act": "none"},
        # LayerNorm over half of the hidden size, statistics exchanged with the row's peer
        {"name": "norm_grid_16384_bf16", "kind": "norm", "grid": 2, "rows": 16384, "hidden": 2048, "dtype": "bf16"},
        # the loss over a quarter of the vocabulary, statistics of the other three staged
        {"name": "loss_8192x12568_bf16", "kind": "loss", "rows": 8192, "vocab": 12568, "ranks": 4, "dtype": "bf16"},
        # head and loss over a whole odd vocabulary, for an odd number of tokens
        {"name": "head_1023x50257_bf16", "kind": "head", "rows": 1023, "hidden": 768, "vocab": 50257, "dtype": "bf16"},
        # the lookup that begins a step and the scatter that ends it
        {"name": "embed_8192x2048_bf16", "kind": "embed", "rows": 8192, "hidden": 2048, "vocab": 12568, "ranks": 4,
         "dtype": "bf16"},
        # clipping: 48 tensors, half of them of a few KB
        {"name": "clip_4x1024_fp32", "kind": "clip", "layers": 4, "hidden": 1024, "dtype": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """A layer width: mostly multiples of 64, as models have them, some of 8, a few only of 4."""
    n, unit = _log(rng, lo, hi), rng.choice((64, 64, 64, 8, 8, 4))
    return max(unit, n // unit * unit)


def draw(rng):
    kind = rng.choice(("step", "step", "step", "eval", "linear", "linear", "norm", "loss", "head", "embed", "clip"))
    half = rng.choice(("bf16", "bf16", "fp16"))
    if kind in ("step", "eval"):
        hidden, heads = rng.choice(WIDTHS)
        # as many tokens as the largest listed step's arithmetic allows
        most = min(16384, int(8192 * (2048 / hidden) ** 2 * (0.75 if kind == "step" else 1.0)))
        tokens = _log(rng, 64, most)
        batch = rng.choice((1, 1, 2, 3, 4, 8))
        seq = min(2048, max(32, tokens // batch))
        dtype = rng.choice((half, half, "autocast"))
        return {"kind": kind, "hidden": hidden, "heads": heads, "batch": batch, "seq": seq, "dtype": dtype,
                "act": rng.choice(("relu", "gelu_tanh"))}
    if kind == "linear":
        grid, dtype = rng.choice(((2, half), (1, half), (0, half), (0, "fp32"), (1, "fp32")))
        q = max(grid, 1)
        n_in, n_out = _features(rng, 256, 6144), _features(rng, 256, 8192)
        budget = (3e10 if dtype == "fp32" else 2.5e11) / (n_in * n_out)
        return {"kind": kind, "grid": grid, "rows": _log(rng, 32, max(64, min(16384, budget))), "in": n_in // q * q,
                "out": n_out // (q * q) * q * q, "dtype": dtype, "act": rng.choice(("none", "none", "gelu_tanh", "relu"))}
    if kind == "norm":
        grid = rng.choice((1, 2))
        return {"kind": kind, "grid": grid, "rows": _log(rng, 64, 16384), "hidden": rng.choice(WIDTHS)[0],
                "dtype": rng.choice((half, half, "fp32"))}
    if kind == "loss":
        vocab, ranks = rng.choice(VOCABS), rng.choice((1, 2, 4))
        vocab = vocab if ranks == 1 else max(250, vocab // ranks)
        return {"kind": kind, "rows": _log(rng, 64, min(16384, int(1.2e8 / vocab))), "vocab": vocab, "ranks": ranks,
                "dtype": rng.choice((half, half, "fp32"))}
    if kind == "head":
        vocab, hidden = rng.choice(VOCABS), rng.choice(WIDTHS)[0]
        return {"kind": kind, "rows": _log(rng, 64, max(128, min(8192, int(3.5e10 / (vocab * hidden))))), "hidden": hidden,
                "vocab": vocab, "dtype": half}
    if kind == "embed":
        ranks = rng.choice((1, 2, 4))
        return {"kind": kind, "rows": _log(rng, 64, 16384), "hidden": rng.choice(WIDTHS)[0],
                "vocab": max(250, rng.choice(VOCABS) // ranks), "ranks": ranks, "dtype": rng.choice((half, half, "fp32"))}
    return {"kind": kind, "layers": rng.choice((1, 2, 3, 4)), "hidden": rng.choice(WIDTHS[:4])[0],
            "dtype": rng.choice((half, "fp32", "fp32"))}


# ----------------------------------------------------------------------------------------------------------- inputs
class _Random:
    """Seeded tensors made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, shape, dtype, std=1.0):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=self.gen)

    def uniform(self, shape, dtype, lo, hi):
        return torch.empty(shape, dtype=dtype, device=DEV).uniform_(lo, hi, generator=self.gen)

    def ids(self, n, most):
        return torch.randint(0, most, (n,), device=DEV, generator=self.gen)

    def fill(self, module):
        """Weights ~ N(0, 0.02), biases ~ N(0, 0.02), LayerNorm scales ~ U(0.9, 1.1)."""
        with torch.no_grad():
            for name, p in module.named_parameters():
                if "norm" in name and name.endswith("weight"):
                    p.uniform_(0.9, 1.1, generator=self.gen)
                else:
                    p.normal_(0.0, 0.02, generator=self.gen)
        return module


def _dtype(case):
    return torch.float32 if case["dtype"] == "autocast" else DTYPES[case["dtype"]]


def prepare(case, seed):
    r = _Random(seed)
    st = {"case": case}
    with torch.device(DEV):
        _PREPARE[case["kind"]](case, r, st)
    return st


def _prepare_block(case, r, st):
    initialize("2d", 1)
    dt = _dtype(case)
    blk = OPTBlock(hidden=case["hidden"], heads=case["heads"], ffn=4 * case["hidden"], dtype=dt, activation=case["act"])
    st["block"] = r.fill(blk)
    st["params"] = list(blk.parameters())
    shape = (case["batch"], case["seq"], case["hidden"])
    st["x"] = r.normal(shape, dt).requires_grad_(case["kind"] == "step")
    st["dy"] = r.normal(shape, dt)


def _prepare_linear(case, r, st):
    dt, act = _dtype(case), None if case["act"] == "none" else case["act"]
    q = max(case["grid"], 1)
    if case["grid"] == 0:
        initialize("1d", 1)
        layer = Linear1D_Col(case["in"], case["out"], activation=act)
    else:
        initialize("2d", q * q, row=0, col=q - 1)
        layer = Linear2D(case["in"], case["out"], activation=act)
    st["layer"] = r.fill(layer.to(dt))
    rows, k, n = case["rows"], case["in"] // q, case["out"] // q
    st["x"] = r.normal((rows, k), dt).requires_grad_(True)
    st["dy"] = r.normal((rows, n), dt)
    if case["grid"] == 2:
        st["peer"] = {"x": r.normal((rows, k), dt), "w": r.normal((k, n), dt, 0.02), "bias": r.normal((n // 2,), dt, 0.02),
                      "dbias": r.normal((n,), torch.float32, math.sqrt(rows)), "dx": r.normal((rows, k), dt),
                      "dw": r.normal((k, n), dt, math.sqrt(rows))}


def _prepare_norm(case, r, st):
    dt, q = _dtype(case), case["grid"]
    initialize("2d", q * q, row=0, col=q - 1)
    layer = LayerNorm2D(case["hidden"]).to(dt)
    with torch.no_grad():
        layer.weight.uniform_(0.9, 1.1, generator=r.gen)
        layer.bias.normal_(0.0, 0.02, generator=r.gen)
    st["layer"] = layer
    rows, c = case["rows"], case["hidden"] // q
    st["x"] = r.normal((rows, c), dt).requires_grad_(True)
    st["dy"] = r.normal((rows, c), dt)
    if q == 2:
        other = r.normal((rows, c), torch.float32)
        st["peer"] = {"stats": torch.stack((other.sum(1), (other * other).sum(1)), 1),
                      "gamma": r.uniform((c // 2,), dt, 0.9, 1.1), "beta": r.normal((c // 2,), dt, 0.02),
                      "sums": r.normal((rows, 2), torch.float32, math.sqrt(c)),
                      "dgamma": r.normal((c,), torch.float32, math.sqrt(rows)),
                      "dbeta": r.normal((c,), torch.float32, math.sqrt(rows))}


def _loss_gradient(case):
    """1, or the power of two by which training in fp16 scales its loss so that the logits' gradients are representable."""
    return torch.tensor(4096.0 if case["dtype"] == "fp16" else 1.0)


def _prepare_loss(case, r, st):
    ranks = case["ranks"]
    initialize("1d", ranks, rank=min(1, ranks - 1))
    st["loss"] = VocabParallelCrossEntropyLoss1D()
    st["x"] = r.normal((case["rows"], case["vocab"]), _dtype(case), 2.0).requires_grad_(True)
    st["targets"] = r.ids(case["rows"], ranks * case["vocab"])
    st["dloss"] = _loss_gradient(case)
    if ranks > 1:
        # the other slices' maximum, sum of exponentials, target logit and mask: logits ~ N(0, 2) as here
        shape = (ranks - 1, case["rows"])
        start = torch.tensor([k * case["vocab"] for k in range(ranks) if k != 1]).unsqueeze(1)
        mask = (st["targets"] < start) | (st["targets"] >= start + case["vocab"])
        st["peer"] = [r.uniform(shape, torch.float32, 6.0, 9.0), r.uniform(shape, torch.float32, 5.0, 50.0),
                      r.normal(shape, torch.float32, 2.0).masked_fill(mask, 0.0), mask.to(torch.uint8)]


def _prepare_head(case, r, st):
    initialize("1d", 1)
    dt = _dtype(case)
    st["layer"] = r.fill(VocabParallelClassifier1D(case["hidden"], case["vocab"], bias=False).to(dt))
    st["loss"] = VocabParallelCrossEntropyLoss1D()
    st["x"] = r.normal((case["rows"], case["hidden"]), dt).requires_grad_(True)
    st["targets"] = r.ids(case["rows"], case["vocab"])
    st["dloss"] = _loss_gradient(case)


def _prepare_embed(case, r, st):
    initialize("1d", 1)
    dt = _dtype(case)
    st["weight"] = r.normal((case["vocab"], case["hidden"]), dt, 0.02).requires_grad_(True)
    st["ids"] = r.ids(case["rows"], case["ranks"] * case["vocab"])
    st["dy"] = r.normal((case["rows"], case["hidden"]), dt)
    st["start"] = 0 if case["ranks"] == 1 else case["vocab"]


def _clip_shapes(case):
    h, f = case["hidden"], 4 * case["hidden"]
    block = [(h,), (h,), (h, 3 * h), (3 * h,), (h, h), (h,), (h,), (h,), (h, f), (f,), (f, h), (h,)]
    return block * case["layers"]


def _prepare_clip(case, r, st):
    initialize("2d", 1)
    dt = _dtype(case)
    params = []
    for shape in _clip_shapes(case):
        p = torch.nn.Parameter(torch.empty(shape, dtype=dt))
        p.grad = r.normal(shape, dt, 0.01)
        params.append(p)
    st["params"] = params


_PREPARE = {"step": _prepare_block, "eval": _prepare_block, "linear": _prepare_linear, "norm": _prepare_norm,
            "loss": _prepare_loss, "head": _prepare_head, "embed": _prepare_embed, "clip": _prepare_clip}


# ------------------------------------------------------------------------------------------------------------- passes
def run(st):
    return _RUN[st["case"]["kind"]](st)


def _forward_block(st):
    if st["case"]["dtype"] == "autocast":
        with torch.autocast("cuda"):
            return st["block"](st["x"])
    return st["block"](st["x"])


def _run_step(st):
    x, params = st["x"], st["params"]
    x.grad = None
    for p in params:
        p.grad = None
    y = _forward_block(st)
    y.backward(st["dy"])
    return [y.detach(), x.grad] + [p.grad for p in params]


def _run_eval(st):
    with torch.no_grad():
        return _forward_block(st)


def _run_linear(st):
    layer, x, peer = st["layer"], st["x"], st.get("peer")
    x.grad = layer.weight.grad = layer.bias.grad = None
    row, col = pm.PARALLEL_2D_ROW, pm.PARALLEL_2D_COL
    if peer:
        row.stage("broadcast", peer["x"])
        col.stage("broadcast", peer["w"])
        col.stage("all_gather", [None, peer["bias"]])
    y = layer(x)
    if peer:
        col.stage("reduce_scatter", [peer["dbias"]])
        col.stage("broadcast", peer["w"])
        row.stage("reduce", [peer["dx"]])
        row.stage("broadcast", peer["x"])
        col.stage("reduce", [peer["dw"]])
    y.backward(st["dy"])
    out = [y.detach(), x.grad, layer.weight.grad, layer.bias.grad]
    if peer:
        # what this rank sends: its products for the row's and the column's peer
        for mode in (row, col):
            out += [t for _, t in mode.outbox["reduce"]]
            mode.outbox.clear()
    return out


def _run_norm(st):
    layer, x, peer = st["layer"], st["x"], st.get("peer")
    x.grad = layer.weight.grad = layer.bias.grad = None
    row, col = pm.PARALLEL_2D_ROW, pm.PARALLEL_2D_COL
    if peer:
        col.stage("all_gather", [None, peer["gamma"]])
        col.stage("all_gather", [None, peer["beta"]])
        row.stage("all_reduce", [peer["stats"]])
    y = layer(x)
    if peer:
        row.stage("all_reduce", [peer["sums"]])
        col.stage("reduce_scatter", [peer["dgamma"]])
        col.stage("reduce_scatter", [peer["dbeta"]])
    y.backward(st["dy"])
    return [y.detach(), x.grad, layer.weight.grad, layer.bias.grad]


def _run_loss(st):
    x = st["x"]
    x.grad = None
    if "peer" in st:
        pm.PARALLEL_1D.stage("vpce_stats", st["peer"])
    loss = st["loss"](x, st["targets"])
    loss.backward(st["dloss"])
    return [loss.detach(), x.grad]


def _run_head(st):
    layer, x = st["layer"], st["x"]
    x.grad = layer.weight.grad = None
    logits = layer(x)
    loss = st["loss"](logits, st["targets"])
    loss.backward(st["dloss"])
    return [logits.detach(), loss.detach(), x.grad, layer.weight.grad]


def _run_embed(st):
    weight = st["weight"]
    weight.grad = None
    y = ops.vocab_embedding(st["ids"], weight, st["start"])
    y.backward(st["dy"])
    return [y.detach(), weight.grad]


def _run_clip(st):
    norm = clip_grad_norm(st["params"], 1.0)
    return [norm] + [p.grad for p in st["params"]]


_RUN = {"step": _run_step, "eval": _run_eval, "linear": _run_linear, "norm": _run_norm, "loss": _run_loss,
        "head": _run_head, "embed": _run_embed, "clip": _run_clip}


# --------------------------------------------------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    size = 4 if case["dtype"] in ("fp32", "autocast") else 2
    if kind in ("step", "eval"):
        h, b, s = case["hidden"], case["batch"], case["seq"]
        tokens, weights = b * s, 12 * h * h + 13 * h
        linears = 2.0 * tokens * 12 * h * h
        attention = 4.0 * b * s * s * h / 2  # the causal half of both products
        if kind == "eval":
            return {"bytes": size * (2.0 * tokens * h + weights), "flops": linears + attention}
        return {"bytes": size * (4.0 * tokens * h + 2.0 * weights), "flops": 3 * linears + 3.5 * attention}
    if kind == "linear":
        q, rows = max(case["grid"], 1), case["rows"]
        k, n = case["in"] // q, case["out"] // q
        x, w, y = rows * k, k * n, rows * n
        # per rank: q products forward and q for each gradient; operands of every step, results, what goes to the peers
        elements = q * (x + w) + 2 * y + q * (x + w) + ((q - 1) * (x + w) if q > 1 else 0)
        return {"bytes": size * float(elements), "flops": 3.0 * q * 2 * rows * k * n}
    if kind == "norm":
        return {"bytes": size * 4.0 * case["rows"] * case["hidden"] / case["grid"],
                "flops": 20.0 * case["rows"] * case["hidden"] / case["grid"]}
    if kind == "loss":
        n = float(case["rows"] * case["vocab"])
        return {"bytes": size * 2 * n, "flops": 8 * n}
    if kind == "head":
        rows, h, v = case["rows"], case["hidden"], case["vocab"]
        # the logits are an output; their gradient is not
        return {"bytes": size * (2.0 * rows * h + 2.0 * v * h + 1.0 * rows * v), "flops": 3 * 2.0 * rows * h * v}
    if kind == "embed":
        rows, h, v = case["rows"], case["hidden"], case["vocab"]
        live = rows / case["ranks"]
        return {"bytes": size * h * (live + rows + live + v) + 16.0 * rows, "flops": live * h}
    n = float(sum(math.prod(s) for s in _clip_shapes(case)))
    return {"bytes": size * 2 * n, "flops": 3 * n}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    # 16-bit storage between the operators: bf16 rounds to 2^-9, fp16 (also under autocast) to 2^-12, a few times in a row
    rel = 1e-2 if case["dtype"] == "bf16" else 3e-3
    # inside a block ReLU's derivative jumps where the layers before it round a value near zero to the other side: a
    # share f of such elements is a relative error of sqrt(2 f) in the gradients
    return {"rel": 2 * rel if case["kind"] == "step" and case["act"] == "relu" else rel}
