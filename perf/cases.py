"""The work that programs have these operators do, as cases that can be timed.

A case is a dict of plain values: its "kind" names a path through the package's public entry points, the other
values its sizes, data type and options.  `listed()` gives the cases that are always measured, `draw(rng)` one more of
the same kinds and ranges.  `prepare(case, seed)` makes what a program holds before it calls (inputs, outputs and the
workspace it keeps), `run(state)` is one pass of that program, `work(case)` the bytes and operations that the calls of
a pass cannot do without: per call, every input read once and every output written once.  A forward and a backward
call each count their own operands, because in a program other layers run between the two.
"""
import importlib
import math

import torch

hk = importlib.import_module("hotspa-ae_amd")
ops = importlib.import_module("hotspa-ae_amd.hetu_ops")

TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
IGNORED = -100


def listed():
    return [
        # one decoding step of a served language model: a residual block's RMSNorm on one token of each of 16 requests
        {"name": "decode_norm", "kind": "decode_norm", "rows": 16, "cols": 4096, "dtype": "bf16"},
        # a training step's RMSNorm on 32768 packed tokens: the benchmark's shape, forward and backward
        {"name": "rms_norm_train", "kind": "rms_norm_train", "rows": 32768, "cols": 4096, "dtype": "bf16"},
        # LayerNorm with scale and bias on feature rows of a width that is no multiple of anything, both directions
        {"name": "layer_norm_odd", "kind": "layer_norm", "rows": 8191, "cols": 1021, "dtype": "bf16"},
        # attention probabilities of 2048-token sequences, forward and backward: the benchmark's shape
        {"name": "attention", "kind": "attention", "heads": 128, "queries": 2048, "keys": 2048, "dtype": "bf16"},
        # the same of an image encoder's 577 tokens (24 x 24 patches and one more): ragged rows
        {"name": "attention_odd", "kind": "attention", "heads": 192, "queries": 577, "keys": 577, "dtype": "bf16"},
        # class probabilities of every pixel (a softmax over the channel dimension), forward and backward
        {"name": "pixel_classes", "kind": "pixel_classes", "batch": 8, "classes": 21, "pixels": 513 * 513, "dtype": "fp32"},
        # a language model's loss per token and its gradient, 5 % of the tokens ignored: the benchmark's shape
        {"name": "cross_entropy", "kind": "cross_entropy", "rows": 16384, "cols": 32000, "dtype": "bf16"},
        # the same over an odd vocabulary that is longer than a workgroup's registers hold
        {"name": "cross_entropy_odd", "kind": "cross_entropy", "rows": 4096, "cols": 50257, "dtype": "bf16"},
        # mean loss of a small classifier's batch and its gradient through the operator layer: latency and launches
        {"name": "classifier_loss", "kind": "mean_loss", "rows": 256, "cols": 1000, "dtype": "fp32"},
        # gradient of a convolution's bias: sum over samples and pixels, one value per channel
        {"name": "channel_sum", "kind": "reduce", "batch": 64, "channels": 256, "inner": 56 * 56, "over": "ends",
         "op": "sum", "dtype": "bf16"},
        # a pre-norm block in training: dropout, residual sum and RMSNorm in one pass, and its gradients
        {"name": "dropout_norm", "kind": "dropout_norm", "rows": 8192, "cols": 4096, "dtype": "bf16"},
        # batch normalisation of a late convolution stage in training, forward and backward
        {"name": "batch_norm", "kind": "batch_norm", "batch": 64, "channels": 256, "pixels": 14 * 14, "dtype": "bf16"},
    ]


# ---------------------------------------------------------------------------
# one more case of the same ranges
# ---------------------------------------------------------------------------
def _between(rng, low, high):
    """A whole number of [low, high], spread over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _width(rng, low, high, odd):
    """A row width: with probability `odd` any number at all, else a multiple of 64 (of 8 below 256)."""
    n = _between(rng, low, high)
    if rng.random() < odd:
        return n
    step = 64 if n >= 256 else 8
    return max(step, n // step * step)


def _dtype(rng):
    return rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])


def _rows(rng, low, high, cols, most, dtype):
    """A row count whose array of `cols` columns holds at most `most` 16-bit elements' bytes."""
    high = max(low, min(high, most * 2 // (cols * SIZE[dtype])))
    return _between(rng, low, high)


def draw(rng):
    kind = rng.choice(["decode_norm", "rms_norm_train", "layer_norm", "attention", "pixel_classes", "cross_entropy",
                       "mean_loss", "reduce", "dropout_norm", "batch_norm"])
    dt = _dtype(rng)
    if kind == "decode_norm":
        return {"kind": kind, "rows": _between(rng, 1, 256), "cols": _width(rng, 512, 8192, 0.2), "dtype": dt}
    if kind == "rms_norm_train":
        cols = _width(rng, 512, 8192, 0.2)
        return {"kind": kind, "rows": _rows(rng, 256, 32768, cols, 32768 * 4096, dt), "cols": cols, "dtype": dt}
    if kind == "layer_norm":
        cols = _width(rng, 64, 8192, 0.5)
        return {"kind": kind, "rows": _rows(rng, 64, 32768, cols, 16384 * 5120, dt), "cols": cols, "dtype": dt}
    if kind == "attention":
        keys = _width(rng, 32, 4096, 0.5)
        queries = keys if rng.random() < 0.7 else _between(rng, 1, 2048)
        heads = _rows(rng, 4, 512, keys * queries, 192 * 1024 * 1024, dt)
        return {"kind": kind, "heads": heads, "queries": queries, "keys": keys, "dtype": dt}
    if kind == "pixel_classes":
        classes = _between(rng, 2, 256)
        batch = _between(rng, 1, 32)
        pixels = _rows(rng, 49, 1024 * 1024, classes * batch, 88 * 1024 * 1024, dt)
        return {"kind": kind, "batch": batch, "classes": classes, "pixels": pixels, "dtype": dt}
    if kind == "cross_entropy":
        cols = _width(rng, 1000, 131072, 0.4)
        return {"kind": kind, "rows": _rows(rng, 64, 16384, cols, 4096 * 50257, dt), "cols": cols, "dtype": dt}
    if kind == "mean_loss":
        cols = _width(rng, 100, 131072, 0.4)
        return {"kind": kind, "rows": _rows(rng, 16, 4096, cols, 1024 * 50257, dt), "cols": cols, "dtype": dt}
    if kind == "reduce":
        over = rng.choice(["ends", "first", "last"])
        channels = _between(rng, 16, 1024)
        inner = _between(rng, 1, 16384) if rng.random() < 0.5 else 8 * _between(rng, 1, 1024)
        batch = _rows(rng, 2, min(512, max(2, 200000 // inner)), channels * inner, 64 * 256 * 3136, dt)
        return {"kind": kind, "batch": batch, "channels": channels, "inner": inner, "over": over,
                "op": rng.choice(["sum", "mean", "max"]), "dtype": dt}
    if kind == "dropout_norm":
        # the dropout interface takes hidden sizes that are multiples of 8
        cols = _width(rng, 512, 8192, 0.2) // 8 * 8
        return {"kind": kind, "rows": _rows(rng, 64, 16384, cols, 16384 * 4096, dt), "cols": cols, "dtype": dt}
    channels = _between(rng, 3, 1024)
    side = _between(rng, 4, 112)
    batch = _rows(rng, 2, 256, channels * side * side, 64 * 256 * 3136, dt)
    return {"kind": "batch_norm", "batch": batch, "channels": channels, "pixels": side * side, "dtype": dt}


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
class _Maker:
    """Seeded inputs on the GPU; large ones in pieces, so that no full-size fp32 copy exists beside them."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        out = torch.empty(shape, dtype=dtype, device="cuda")
        flat, step = out.view(-1), 1 << 26
        for o in range(0, flat.numel(), step):
            part = flat[o:o + step]
            part.copy_(torch.randn(part.numel(), generator=self.gen, device="cuda") * std + mean)
        return out

    def uniform(self, shape, dtype, low, high):
        return (torch.rand(shape, generator=self.gen, device="cuda") * (high - low) + low).to(dtype)

    def labels(self, rows, cols, ignored_share):
        lab = torch.randint(0, cols, (rows,), generator=self.gen, device="cuda", dtype=torch.int64)
        lab[torch.rand(rows, generator=self.gen, device="cuda") < ignored_share] = IGNORED
        return lab


def _floats(nbytes):
    """The workspace a program keeps for a call that asks for `nbytes` of it."""
    return torch.empty(max(1, (nbytes + 3) // 4), dtype=torch.float32, device="cuda")


def _like(t):
    return torch.empty_like(t)


def _reduced(case):
    """(shape, axes) of a reduction of a [batch, channels, inner] array."""
    b, c, n = case["batch"], case["channels"], case["inner"]
    return [b, c, n], {"ends": [0, 2], "first": [0], "last": [2]}[case["over"]]


def prepare(case, seed):
    m, kind, dt = _Maker(seed), case["kind"], TYPES[case["dtype"]]
    s = {"kind": kind}
    if kind in ("decode_norm", "rms_norm_train", "layer_norm", "dropout_norm"):
        rows, cols = case["rows"], case["cols"]
        s["x"] = m.normal((rows, cols), dt)
        s["gamma"] = m.uniform((cols,), dt, 0.8, 1.2)
        s["y"] = _like(s["x"])
        s["mean"] = torch.empty(rows, device="cuda")
        s["rstd"] = torch.empty(rows, device="cuda")
    if kind == "decode_norm":
        s["residual"] = m.normal((rows, cols), dt)
        s["sum"] = _like(s["x"])
    elif kind in ("rms_norm_train", "layer_norm"):
        s["dy"] = m.normal((rows, cols), dt)
        s["dx"] = _like(s["x"])
        s["dgamma"] = _like(s["gamma"])
        if kind == "layer_norm":
            s["beta"] = m.normal((cols,), dt, 0.1)
            s["dbeta"] = _like(s["beta"])
        s["workspace"] = _floats(hk.norm_bwd_workspace_bytes(hk.dtype_code(s["x"]), rows, cols))
    elif kind == "dropout_norm":
        s["residual"] = m.normal((rows, cols), dt)
        s["dy"] = m.normal((rows, cols), dt)
        s["dsum"] = m.normal((rows, cols), dt)
        s["sum"], s["dx"], s["dresidual"] = _like(s["x"]), _like(s["x"]), _like(s["x"])
        s["keep"] = torch.empty((rows, cols), dtype=torch.uint8, device="cuda")
        s["dgamma"] = _like(s["gamma"])
        s["seed"] = 1 + int(seed)
        _dropout_forward(s)
        s["workspace"] = None
        s["workspace"] = _dropout_backward(s)
    elif kind == "attention":
        shape = (case["heads"], case["queries"], case["keys"])
        s["x"] = m.normal(shape, dt, 3.0)
        s["dy"] = m.normal(shape, dt)
        s["y"], s["dx"], s["dim"] = _like(s["x"]), _like(s["x"]), -1
    elif kind == "pixel_classes":
        shape = (case["batch"], case["classes"], case["pixels"])
        s["x"] = m.normal(shape, dt, 2.0)
        s["dy"] = m.normal(shape, dt)
        s["y"], s["dx"], s["dim"] = _like(s["x"]), _like(s["x"]), 1
    elif kind in ("cross_entropy", "mean_loss"):
        rows, cols = case["rows"], case["cols"]
        s["x"] = m.normal((rows, cols), dt, 2.0)
        s["labels"] = m.labels(rows, cols, 0.05)
        s["dx"] = _like(s["x"])
        if kind == "cross_entropy":
            s["loss"] = torch.empty(rows, dtype=dt, device="cuda")
            s["dloss"] = m.uniform((rows,), dt, 0.5 / rows, 1.5 / rows)
        else:
            s["loss"] = torch.empty(1, dtype=dt, device="cuda")
            s["dloss"] = torch.ones(1, dtype=dt, device="cuda")
    elif kind == "reduce":
        shape, axes = _reduced(case)
        s["x"] = m.normal(shape, dt, 1.0, 0.5)
        s["axes"], s["op"] = axes, case["op"]
        kept = [n for i, n in enumerate(shape) if i not in axes]
        s["out"] = torch.empty(kept, dtype=dt, device="cuda")
        s["workspace"] = _floats(hk.reduce_workspace_bytes(hk.dtype_code(s["x"]), shape, list(s["x"].stride()), axes))
    elif kind == "batch_norm":
        shape = (case["batch"], case["channels"], case["pixels"])
        c = case["channels"]
        s["x"] = m.normal(shape, dt, 1.5, 0.3)
        s["dy"] = m.normal(shape, dt)
        s["y"], s["dx"] = _like(s["x"]), _like(s["x"])
        s["scale"] = m.uniform((c,), torch.float32, 0.5, 1.5)
        s["bias"] = m.normal((c,), torch.float32, 0.1)
        s["running_mean"] = torch.zeros(c, device="cuda")
        s["running_var"] = torch.ones(c, device="cuda")
        s["mean"], s["invstd"] = torch.empty(c, device="cuda"), torch.empty(c, device="cuda")
        s["dscale"], s["dbias"] = torch.empty(c, device="cuda"), torch.empty(c, device="cuda")
        s["workspace"] = _floats(hk.batch_norm_workspace_bytes(s["x"]))
    if kind == "mean_loss":
        # the operator layer works on streams of its own: a program that fills its inputs on another one waits first
        torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _dropout_forward(s):
    hk.dropout_add_ln_fwd_ex(s["x"], s["gamma"], s["y"], s["mean"], s["rstd"], residual=s["residual"], x=s["sum"],
                             dmask=s["keep"], dropout_p=0.1, eps=1e-6, is_rms=True, seed=s["seed"])


def _dropout_backward(s):
    return hk.dropout_add_ln_bwd_ex(s["dy"], s["sum"], s["mean"], s["rstd"], s["gamma"], s["dx"], dx=s["dsum"],
                                    dmask=s["keep"], dresidual=s["dresidual"], dgamma=s["dgamma"], dropout_p=0.1,
                                    is_rms=True, workspace=s["workspace"])


def run(s):
    kind = s["kind"]
    if kind == "decode_norm":
        hk.dropout_add_ln_fwd(s["x"], s["residual"], s["gamma"], None, s["y"], s["sum"], s["mean"], s["rstd"], 1e-6, True)
        return s["y"], s["sum"], s["rstd"]
    if kind == "rms_norm_train":
        hk.dropout_add_ln_fwd(s["x"], None, s["gamma"], None, s["y"], None, s["mean"], s["rstd"], 1e-6, True)
        hk.dropout_add_ln_bwd(s["dy"], None, s["x"], s["mean"], s["rstd"], s["gamma"], s["dx"], None, s["dgamma"], None,
                              True, workspace=s["workspace"])
        return s["y"], s["rstd"], s["dx"], s["dgamma"]
    if kind == "layer_norm":
        hk.layer_norm_fwd(s["x"], s["gamma"], s["beta"], s["y"], s["mean"], s["rstd"], 1e-5)
        hk.layer_norm_bwd(s["dy"], s["x"], s["gamma"], s["beta"], s["mean"], s["rstd"], s["dx"], s["dgamma"], s["dbeta"],
                          1e-5, workspace=s["workspace"])
        return s["y"], s["rstd"], s["dx"], s["dgamma"], s["dbeta"]
    if kind == "dropout_norm":
        _dropout_forward(s)
        _dropout_backward(s)
        return s["y"], s["sum"], s["keep"], s["rstd"], s["dx"], s["dresidual"], s["dgamma"]
    if kind in ("attention", "pixel_classes"):
        hk.softmax_fwd(s["x"], s["y"], s["dim"])
        hk.softmax_bwd(s["y"], s["dy"], s["dx"], s["dim"])
        return s["y"], s["dx"]
    if kind == "cross_entropy":
        hk.sce_sparse_fwd(s["x"], s["labels"], s["loss"], IGNORED)
        hk.sce_sparse_bwd(s["x"], s["labels"], s["dloss"], s["dx"], IGNORED)
        return s["loss"], s["dx"]
    if kind == "mean_loss":
        ops.ndarray_sceloss(s["x"], s["labels"], s["loss"], "mean", ignored_index=IGNORED)
        ops.sceloss_gradient(s["x"], s["labels"], s["dloss"], s["dx"], "mean", ignored_index=IGNORED)
        return s["loss"], s["dx"]
    if kind == "reduce":
        hk.reduce(s["x"], s["out"], s["axes"], s["op"], workspace=s["workspace"])
        return s["out"]
    hk.batch_norm_fwd(s["x"], s["scale"], s["bias"], s["y"], 0.1, 1e-5, s["running_mean"], s["running_var"], s["mean"],
                      s["invstd"], workspace=s["workspace"])
    hk.batch_norm_bwd(s["dy"], s["x"], s["scale"], s["dx"], s["dscale"], s["dbias"], s["mean"], s["invstd"],
                      workspace=s["workspace"])
    return (s["y"], s["mean"], s["invstd"], s["running_mean"], s["running_var"], s["dx"], s["dscale"], s["dbias"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how near another correct implementation comes
# ---------------------------------------------------------------------------
def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    if kind in ("attention", "pixel_classes"):
        n = case["heads"] * case["queries"] * case["keys"] if kind == "attention" else \
            case["batch"] * case["classes"] * case["pixels"]
        return {"bytes": 5 * n * es, "flops": 10 * n}
    if kind == "batch_norm":
        n, c = case["batch"] * case["channels"] * case["pixels"], case["channels"]
        return {"bytes": 5 * n * es + 15 * 4 * c, "flops": 12 * n}
    if kind == "reduce":
        shape, axes = _reduced(case)
        n = shape[0] * shape[1] * shape[2]
        kept = n
        for a in axes:
            kept //= shape[a]
        return {"bytes": (n + kept) * es, "flops": n}
    rows, cols = case["rows"], case["cols"]
    n = rows * cols
    if kind == "decode_norm":
        return {"bytes": 4 * n * es + cols * es + 8 * rows, "flops": 5 * n}
    if kind == "rms_norm_train":
        return {"bytes": 5 * n * es + 3 * cols * es + 12 * rows, "flops": 14 * n}
    if kind == "layer_norm":
        return {"bytes": 5 * n * es + 5 * cols * es + 16 * rows, "flops": 20 * n}
    if kind == "dropout_norm":
        return {"bytes": 4 * n * es + 5 * n * es + 2 * n + 3 * cols * es + 12 * rows, "flops": 20 * n}
    if kind == "cross_entropy":
        # ignored rows are not read
        return {"bytes": int(2.9 * n * es) + rows * (16 + 2 * es), "flops": 10 * n}
    return {"bytes": int(2.9 * n * es) + rows * 16, "flops": 10 * n}


def tolerance(case):
    """About four times what the outputs were seen to differ by from the same formulas in 64 bits over all kinds (2-norm
    and single values): bf16 2e-3 and 6e-3, the rounding of what is stored; fp16 2.3e-4 and 4.9e-4, but 2.7e-3 and 7e-3
    for the gradients of the losses, most of which are smaller than fp16's smallest normal number; fp32 2.6e-7 and 1e-5
    (sums over up to a thousand rows, and brackets that nearly cancel), with room for sums over more of them."""
    if case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 4e-5}
    if case["dtype"] == "bf16" or case["kind"] in ("cross_entropy", "mean_loss"):
        return {"rel": 1e-2, "max": 2.5e-2}
    return {"rel": 1e-3, "max": 2e-3}
