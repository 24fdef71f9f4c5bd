"""Performance cases of the fused non-GEMM ops, through their public entry points.

The work that a transformer gives this package: the norms, the attention softmax,
bias-GeLU, the residual block and the optimizer step, one op at a time where an op
has its own workload and as the chain of one layer where latency and launches
count.  Sizes come from the five workloads of the repository's benchmark (causal
softmax [48, 512, 512], norm [16384, 4096], padding mask [16, 16, 1024, 1024],
bias-GeLU [16384, 16384], and the layer of hidden size 6144 with 64 heads) and
from their neighbours: one token at a time, prompts of any length.

A case is a dict of plain values:
  op     "norm" | "softmax" | "gelu" | "residual" | "layer" | "adam"
  train  forward and backward (True), or forward only without autograd
  dtype  "bf16" | "fp16" | "fp32"
  norm, gelu, residual:  rows, hidden;  norm: rms;  residual: p (dropout)
  softmax:  batch, heads, sq, sk, mask ("causal" | "padding" | "additive" |
            "causal_padding"), p
  layer:    batch, seq, keys (cached keys + seq), hidden, heads, mask, p
  adam:     layers, hidden (the parameters of `layers` blocks of that width)
"""
import math

import torch

import oslo_amd.torch.nn as onn
from oslo_amd.torch.optim import FusedAdam

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # one decoding step of a batch of four: the norm in front of a block
        {"name": "norm_decode", "op": "norm", "train": False, "dtype": "bf16", "rms": False,
         "rows": 4, "hidden": 6144},
        # attention of one new token over a left-padded cache, mask as models pass it
        {"name": "softmax_decode", "op": "softmax", "train": False, "dtype": "bf16", "batch": 4,
         "heads": 64, "sq": 1, "sk": 1777, "mask": "additive", "p": 0.0},
        # one layer over a padded batch of prompts whose longest has 1003 tokens
        {"name": "layer_prefill", "op": "layer", "train": False, "dtype": "fp16", "batch": 2,
         "seq": 1003, "keys": 1003, "hidden": 4096, "heads": 32, "mask": "causal_padding", "p": 0.0},
        # one layer of a small causal model in training, float32, batch 4 x 512 tokens, 12 heads
        {"name": "layer_train_small", "op": "layer", "train": True, "dtype": "fp32", "batch": 4,
         "seq": 512, "keys": 512, "hidden": 768, "heads": 12, "mask": "causal", "p": 0.1},
        # one layer of an encoder in training on sentences padded to the longest of the batch
        {"name": "layer_train_ragged", "op": "layer", "train": True, "dtype": "fp16", "batch": 8,
         "seq": 381, "keys": 381, "hidden": 1024, "heads": 16, "mask": "additive", "p": 0.1},
        # LayerNorm of a large batch, forward and backward
        {"name": "norm_train", "op": "norm", "train": True, "dtype": "bf16", "rms": False,
         "rows": 16384, "hidden": 4096},
        # causal attention of a 2048-token context with 64 heads: the largest tensors
        {"name": "softmax_train_causal", "op": "softmax", "train": True, "dtype": "bf16",
         "batch": 4, "heads": 64, "sq": 2048, "sk": 2048, "mask": "causal", "p": 0.0},
        # padding-masked attention of an encoder
        {"name": "softmax_train_padding", "op": "softmax", "train": True, "dtype": "fp16",
         "batch": 16, "heads": 16, "sq": 1024, "sk": 1024, "mask": "padding", "p": 0.0},
        # causal attention with attention dropout at a length that is no round number
        {"name": "softmax_train_ragged", "op": "softmax", "train": True, "dtype": "bf16",
         "batch": 4, "heads": 32, "sq": 1531, "sk": 1531, "mask": "causal", "p": 0.1},
        # first half of a wide MLP
        {"name": "gelu_train", "op": "gelu", "train": True, "dtype": "bf16", "rows": 16384,
         "hidden": 16384},
        # residual block (bias, dropout, residual add, LayerNorm) of the wide layer
        {"name": "residual_train", "op": "residual", "train": True, "dtype": "bf16",
         "rows": 8192, "hidden": 6144, "p": 0.1},
        # optimizer step of twelve blocks of width 768 (85 M parameters, 144 tensors)
        {"name": "adam_step", "op": "adam", "train": True, "dtype": "fp32", "layers": 12,
         "hidden": 768},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A model width: a whole number of 64-wide heads."""
    return 64 * max(low // 64, _log_int(rng, low, high) // 64)


def draw(rng):
    op = rng.choice(["norm", "softmax", "softmax", "gelu", "residual", "layer", "layer", "adam"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    train = rng.random() < 0.7
    case = {"op": op, "train": train, "dtype": dtype}
    if op in ("norm", "gelu", "residual"):
        case["hidden"] = _width(rng, 256, 16384 if op == "gelu" else 8192)
        most = 2 ** 26 // case["hidden"] * (4 if op == "gelu" and dtype != "fp32" else 1)
        case["rows"] = min(_log_int(rng, 1, 32768), most)
        if op == "norm":
            case["rms"] = rng.random() < 0.5
        if op == "residual":
            case["p"] = rng.choice([0.0, 0.1])
    elif op == "softmax":
        sk = _log_int(rng, 16, 4096)
        decode = not train and rng.random() < 0.5
        sq = 1 if decode else sk
        rows = min(_log_int(rng, 16, 512), max(16, 2 ** 30 // (sq * sk * _ESIZE[dtype])))
        heads = rng.choice([8, 12, 16])
        batch = max(1, rows // heads)
        mask = rng.choice(["causal", "padding", "additive", "causal_padding"])
        case.update(batch=batch, heads=heads, sq=sq, sk=sk, mask=mask,
                    p=rng.choice([0.0, 0.1]) if train else 0.0)
    elif op == "layer":
        heads = rng.choice([8, 12, 16, 32])
        batch = rng.randint(1, 8)
        if not train and rng.random() < 0.5:
            keys, seq = _log_int(rng, 16, 4096), 1
        else:
            keys = seq = _log_int(rng, 32, 1536)
        batch = min(batch, max(1, 2 ** 29 // (heads * seq * keys * _ESIZE[dtype])))
        case.update(batch=batch, seq=seq, keys=keys, hidden=heads * rng.choice([64, 128]),
                    heads=heads, mask=rng.choice(["causal", "additive", "causal_padding"]),
                    p=rng.choice([0.0, 0.1]) if train else 0.0)
    else:
        case.update(train=True, layers=_log_int(rng, 1, 16), hidden=_width(rng, 128, 1024),
                    dtype=rng.choice(["fp32", "fp32", "bf16"]))
    return case


# ---------------------------------------------------------------- inputs
class _Maker:
    """Random tensors on the GPU from one seed."""

    def __init__(self, case, seed):
        torch.manual_seed(seed)  # (the dropout of the pass draws from torch's generator)
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.dtype = _DTYPES[case["dtype"]]
        self.gen = torch.Generator(device=self.device).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.gen, device=self.device, dtype=self.dtype)
        if std != 1.0:
            t.mul_(std)
        return t.add_(mean) if mean else t

    def lengths(self, batch, keys):
        """Valid keys per sentence of a padded batch: half to all of them, one full."""
        n = torch.randint(max(1, keys // 2), keys + 1, (batch,), generator=self.gen, device=self.device)
        n[0] = keys
        return n

    def module(self, m, train):
        """The module on the GPU with weights as training leaves them."""
        m = m.to(self.device, self.dtype).train(train)
        with torch.no_grad():
            for name, w in m.named_parameters():
                w.copy_(self.normal(*w.shape, std=0.02, mean=1.0 if name == "weight" else 0.0))
                w.requires_grad_(train)
        return m


def _attention(mk, case, batch, heads, sq, sk, train):
    """The softmax module and the mask of a padded batch in the form the model passes it."""
    causal = case["mask"].startswith("causal")
    module = onn.FusedScaleMaskSoftmax(
        input_in_fp16=case["dtype"] == "fp16", input_in_bf16=case["dtype"] == "bf16",
        attn_mask_type=onn.AttnMaskType.causal if causal else onn.AttnMaskType.padding,
        scale=0.125, attn_dropout=case["p"]).train(train)
    mask = None
    if case["mask"] != "causal":
        valid = mk.lengths(batch, sk)
        hidden = torch.arange(sk, device=mk.device) >= valid[:, None]
        hidden = hidden.view(batch, 1, 1, sk)
        if case["mask"] == "additive":
            mask = torch.zeros(hidden.shape, dtype=mk.dtype, device=mk.device).masked_fill_(hidden, -10000.0)
        else:
            mask = hidden
    return module, mask


def _leaf(t, train):
    return t.requires_grad_(train)


def prepare(case, seed):
    mk = _Maker(case, seed)
    op, train = case["op"], case["train"]
    s = {"op": op, "train": train, "case": case}
    if op == "norm":
        rows, hidden = case["rows"], case["hidden"]
        cls = onn.FusedRMSNorm if case["rms"] else onn.FusedLayerNorm
        s["module"] = mk.module(cls(hidden), train)
        s["x"] = _leaf(mk.normal(rows, hidden, mean=0.1), train)
        s["leaves"] = [s["x"]] + list(s["module"].parameters())
        s["grads"] = [mk.normal(rows, hidden)] if train else None
    elif op == "softmax":
        b, h, sq, sk = case["batch"], case["heads"], case["sq"], case["sk"]
        s["module"], s["mask"] = _attention(mk, case, b, h, sq, sk, train)
        s["x"] = _leaf(mk.normal(b, h, sq, sk, std=8.0), train)
        s["leaves"] = [s["x"]]
        s["grads"] = [mk.normal(b, h, sq, sk)] if train else None
    elif op == "gelu":
        rows, hidden = case["rows"], case["hidden"]
        s["x"] = _leaf(mk.normal(rows, hidden), train)
        s["bias"] = _leaf(mk.normal(hidden, std=0.02), train)
        s["leaves"] = [s["x"], s["bias"]]
        s["grads"] = [mk.normal(rows, hidden)] if train else None
    elif op == "residual":
        rows, hidden = case["rows"], case["hidden"]
        s["module"] = mk.module(onn.FusedBiasDropoutAddLayerNorm(hidden, p=case["p"], return_sum=True), train)
        s["x"] = _leaf(mk.normal(rows, hidden), train)
        s["bias"] = _leaf(mk.normal(hidden, std=0.02), train)
        s["residual"] = _leaf(mk.normal(rows, hidden), train)
        s["leaves"] = [s["x"], s["bias"], s["residual"]] + list(s["module"].parameters())
        s["grads"] = [mk.normal(rows, hidden), mk.normal(rows, hidden)] if train else None
    elif op == "layer":
        # What the matrix products of a pre-LN block hand to the ops between
        # them: its input, the attention scores, the attention output, the two
        # MLP products, and the biases that those products leave to be added.
        b, seq, keys, hidden, h = (case[k] for k in ("batch", "seq", "keys", "hidden", "heads"))
        s["ln"] = mk.module(onn.FusedLayerNorm(hidden), train)
        s["attn"], s["mask"] = _attention(mk, case, b, h, seq, keys, train)
        s["ln2"] = mk.module(onn.FusedBiasDropoutAddLayerNorm(hidden, p=case["p"], return_sum=True), train)
        s["drop"] = onn.FusedBiasDropout(p=case["p"]).train(train)
        s["x"] = _leaf(mk.normal(b, seq, hidden), train)
        s["scores"] = _leaf(mk.normal(b, h, seq, keys, std=8.0), train)
        s["context"] = _leaf(mk.normal(b, seq, hidden), train)
        s["fc1"] = _leaf(mk.normal(b, seq, 4 * hidden), train)
        s["fc2"] = _leaf(mk.normal(b, seq, hidden), train)
        s["biases"] = [_leaf(mk.normal(n, std=0.02), train) for n in (hidden, 4 * hidden, hidden)]
        s["leaves"] = ([s["x"], s["scores"], s["context"], s["fc1"], s["fc2"]] + s["biases"]
                       + list(s["ln"].parameters()) + list(s["ln2"].parameters()))
        s["grads"] = None
        if train:
            s["grads"] = [mk.normal(b, seq, hidden), mk.normal(b, h, seq, keys), mk.normal(b, seq, hidden),
                          mk.normal(b, seq, 4 * hidden), mk.normal(b, seq, hidden)]
    else:
        # the parameters of a model, flat in memory with each tensor on a
        # 256-byte boundary, as gradient buckets and sharded checkpoints keep them
        shapes = _adam_shapes(case)
        spans, at = [], 0
        for shape in shapes:
            spans.append(at)
            at += -(-math.prod(shape) // 128) * 128
        flat = {"param": mk.normal(at, std=0.02), "grad": mk.normal(at, std=1e-3),
                "exp_avg": mk.normal(at, std=1e-3), "exp_avg_sq": mk.normal(at, std=1e-3).square_()}

        def view(key, k):
            return flat[key][spans[k]:spans[k] + math.prod(shapes[k])].view(shapes[k])

        params = [torch.nn.Parameter(view("param", k)) for k in range(len(shapes))]
        opt = FusedAdam(params, lr=1e-4, weight_decay=0.01)
        for k, prm in enumerate(params):
            prm.grad = view("grad", k)
            opt.state[prm] = {"exp_avg": view("exp_avg", k), "exp_avg_sq": view("exp_avg_sq", k)}
        opt.param_groups[0]["step"] = 1000  # (in the middle of a training run)
        s["opt"], s["updated"] = opt, [flat["param"], flat["exp_avg"], flat["exp_avg_sq"]]
    return s


def _adam_shapes(case):
    h = case["hidden"]
    block = [(h,), (h,), (3 * h, h), (3 * h,), (h, h), (h,), (h,), (h,), (4 * h, h), (4 * h,), (h, 4 * h), (h,)]
    return block * case["layers"]


# ---------------------------------------------------------------- one pass
def _forward(s):
    op = s["op"]
    if op == "norm":
        return [s["module"](s["x"])]
    if op == "softmax":
        return [s["module"](s["x"], s["mask"])]
    if op == "gelu":
        return [onn.fused_bias_gelu(s["x"], s["bias"])]
    if op == "residual":
        return list(s["module"](s["x"], s["bias"], s["residual"]))
    normed = s["ln"](s["x"])
    probs = s["attn"](s["scores"], s["mask"])
    normed2, stream = s["ln2"](s["context"], s["biases"][0], s["x"])
    act = onn.fused_bias_gelu(s["fc1"], s["biases"][1])
    out = s["drop"](s["fc2"], s["biases"][2], stream)
    return [normed, probs, normed2, act, out]


def run(s):
    if s["op"] == "adam":
        s["opt"].step()
        return s["updated"]
    if not s["train"]:
        with torch.no_grad():
            return _forward(s)
    for t in s["leaves"]:
        t.grad = None
    outs = _forward(s)
    torch.autograd.backward(outs, s["grads"])
    return [o.detach() for o in outs] + [t.grad for t in s["leaves"]]


# ---------------------------------------------------------------- what a pass cannot do without
def _visible(case, sq, sk):
    """Share of the scores that a row may look at (padding hides a quarter of the keys on average)."""
    share = 1.0
    if case["mask"].startswith("causal") and sq > 1:
        share = (sk + 1) / (2 * sk)
    if case["mask"] in ("padding", "causal_padding"):
        share *= 0.75 + 0.25 / case.get("batch", 1)
    return share


def _softmax_work(case, batch, heads, sq, sk):
    n, e, f = batch * heads * sq * sk, _ESIZE[case["dtype"]], _visible(case, sq, sk)
    return (n * e * (1 + f) + (n * e * (1 + 2 * f) if case["train"] else 0), n * (12 if case["train"] else 6))


def work(case):
    op, train, e = case["op"], case["train"], _ESIZE[case["dtype"]]
    if op == "adam":
        n = sum(math.prod(shape) for shape in _adam_shapes(case))
        return {"bytes": 7 * n * e, "flops": 16 * n}
    if op == "softmax":
        b, f = _softmax_work(case, case["batch"], case["heads"], case["sq"], case["sk"])
        return {"bytes": b, "flops": f}
    if op == "layer":
        n = case["batch"] * case["seq"] * case["hidden"]
        b, f = _softmax_work(case, case["batch"], case["heads"], case["seq"], case["keys"])
        # norm 2 (+ 3), residual norm 4 (+ 4), bias-GeLU 2 (+ 3) of four times
        # the width, bias-dropout-add 3 (+ 2); the input is read by two of them
        b += n * e * ((17 + 21) if train else 17)
        return {"bytes": b, "flops": f + n * (150 if train else 60)}
    n = case["rows"] * case["hidden"]
    fwd, bwd, ops = {"norm": (2, 3, 16), "gelu": (2, 3, 24), "residual": (4, 4, 24)}[op]
    return {"bytes": n * e * (fwd + (bwd if train else 0)), "flops": n * ops}


def tolerance(case):
    # Four times the distance between the path and the same pass evaluated
    # wider, at the listed sizes.  float32 against float64 formulas: rel 1.4e-7,
    # max 1.2e-5 (a parameter after its optimizer step).  16-bit against the
    # float32 kernels on the same values: rel 2.8e-3 (bf16) and 3.6e-4 (fp16),
    # where a tensor between two kernels is stored rounded, and one unit in the
    # last place of a 16-bit result (max 7.8e-3 and 1.8e-3).
    if case["dtype"] == "fp32":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.03} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 7.5e-3}
