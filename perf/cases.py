"""The work that stands for this framework in measurements: `@dvm_amd.kernel` functions called on torch tensors that
live on the GPU, and an eager torch program under `dvm_amd.lazy_fusion()`.

`listed()` holds twelve calls of ten operators, `draw(rng)` one more call of the same operators anywhere in their
ranges: one element to 2^25, one row to 8192, 16- and 32-bit floats, dense and strided operands, forward and backward,
prefill and decode. A program decorates a function once and keeps it; what is measured is the call. Every kernel here is
dynamic: the shapes are those of the call's tensors, as in a serving or training loop.
"""
import math

import torch

import dvm_amd as dvm

_TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_DVM = {"float32": dvm.float32, "float16": dvm.float16, "bfloat16": dvm.bfloat16}
_SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}


def listed():
    return [
        # the smallest fused call: two fp32 tiles added (a launch and the host work in front of it)
        {"name": "add_small", "op": "add", "rows": 32, "cols": 32, "dtype": "float32"},
        # batch-norm of a convolutional network in training, the whole batch's statistics in the same call
        {"name": "batchnorm_train", "op": "batchnorm", "n": 32, "c": 256, "h": 56, "w": 56},
        # residual add + RMSNorm between the blocks of a transformer: a prompt of 8192 tokens
        {"name": "rmsnorm_prefill", "op": "rmsnorm", "rows": 8192, "hidden": 4096, "dtype": "bfloat16"},
        # the same function while tokens are generated: as many rows as there are sequences in flight
        {"name": "rmsnorm_decode", "op": "rmsnorm", "rows": 37, "hidden": 4096, "dtype": "bfloat16"},
        # softmax over a vocabulary of 32001 (odd rows, not aligned), fp32 logits of 2048 tokens
        {"name": "softmax_vocab", "op": "softmax", "rows": 2048, "cols": 32001, "dtype": "float32"},
        # optimizer step on a 4096 x 4096 weight: new parameters and moments
        {"name": "adam_step", "op": "adam", "numel": 16777216},
        # linear layer with bias and SiLU of a prompt, weights [in, out]
        {"name": "linear_prefill", "op": "linear", "m": 8192, "n": 4096, "k": 4096, "dtype": "bfloat16", "weight_out_in": False},
        # the same layer for the tokens of eight sequences, weights [out, in]: a read of the weights
        {"name": "linear_decode", "op": "linear", "m": 8, "n": 8192, "k": 8192, "dtype": "bfloat16", "weight_out_in": True},
        # backward of a linear layer: gradients of its input, weight and bias
        {"name": "linear_backward", "op": "linear_backward", "m": 4096, "n": 4096, "k": 2048, "dtype": "bfloat16"},
        # attention of a prompt, heads outermost
        {"name": "attention_prefill", "op": "attention", "batch": 8, "heads": 32, "queries": 2048, "keys": 2048, "d": 128,
         "dtype": "float16", "seq_first": False},
        # attention of one new token per sequence over a cache of 1999, tokens outermost ([batch, tokens, heads, d])
        {"name": "attention_decode", "op": "attention", "batch": 16, "heads": 32, "queries": 1, "keys": 1999, "d": 128,
         "dtype": "bfloat16", "seq_first": True},
        # an eager program without a decorator: RMSNorm, gate and residual of a feed-forward block, torch operators
        {"name": "eager_gate", "op": "eager_gate", "rows": 512, "hidden": 4096, "dtype": "bfloat16"},
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _log8(rng, low, high):
    return _log(rng, low // 8, high // 8) * 8


def draw(rng):
    op = rng.choice(["add", "batchnorm", "rmsnorm", "softmax", "adam", "linear", "linear_decode", "linear_backward", "attention",
                     "attention_decode", "eager_gate"])
    half = rng.choice(["float16", "bfloat16"])
    floats = rng.choice(["float32", "float16", "bfloat16"])
    if op == "add":
        return {"op": op, "rows": _log(rng, 1, 2048), "cols": _log(rng, 1, 4096), "dtype": floats}
    if op == "batchnorm":
        n, c, h = _log(rng, 1, 32), _log(rng, 16, 512), _log(rng, 7, 112)
        while n * c * h * h > 25690112:
            n, c, h = (n + 1) // 2, (c + 1) // 2, h
        return {"op": op, "n": n, "c": c, "h": h, "w": h}
    if op == "rmsnorm":
        return {"op": op, "rows": _log(rng, 1, 8191), "hidden": rng.choice([_log8(rng, 512, 8192), _log(rng, 500, 4096), 4096]), "dtype": half}
    if op == "softmax":
        cols = _log(rng, 64, 65537)
        return {"op": op, "rows": _log(rng, 1, max(1, min(8192, 65536000 // cols))), "cols": cols, "dtype": floats}
    if op == "adam":
        return {"op": op, "numel": _log(rng, 1000, 16777215)}
    if op == "linear":
        return {"op": op, "m": _log(rng, 128, 8191), "n": _log8(rng, 512, 4096), "k": _log8(rng, 512, 4096), "dtype": half,
                "weight_out_in": rng.random() < 0.5}
    if op == "linear_decode":
        return {"op": "linear", "m": _log(rng, 1, 64), "n": _log8(rng, 1024, 8192), "k": _log8(rng, 1024, 8192), "dtype": half,
                "weight_out_in": rng.random() < 0.5}
    if op == "linear_backward":
        return {"op": op, "m": _log(rng, 256, 4096), "n": _log8(rng, 512, 4096), "k": _log8(rng, 512, 2048), "dtype": half}
    if op == "attention":
        batch, heads, s = _log(rng, 1, 8), _log(rng, 4, 32), _log(rng, 64, 2047)
        return {"op": op, "batch": batch, "heads": heads, "queries": s, "keys": rng.choice([s, _log(rng, 64, 2048)]), "d": rng.choice([64, 128]),
                "dtype": half, "seq_first": rng.random() < 0.5}
    if op == "attention_decode":
        return {"op": "attention", "batch": _log(rng, 1, 16), "heads": _log(rng, 4, 32), "queries": _log(rng, 1, 8), "keys": _log(rng, 64, 4096),
                "d": rng.choice([64, 128]), "dtype": half, "seq_first": rng.random() < 0.5}
    return {"op": op, "rows": _log(rng, 1, 4096), "hidden": _log8(rng, 512, 4096), "dtype": floats}


# ---- the kernels of a user's program ----

def _add_kernel(case):
    dt = _DVM[case["dtype"]]

    @dvm.kernel(ktype="split", dynamic=True)
    def add(k, x, y):
        return k.store(k.add(k.load(x, dt), k.load(y, dt)))
    return add


def _batchnorm_kernel(case):
    """Mean and biased variance over N, H, W, then x * scale + shift with one scale and shift per channel."""
    inv = 1.0 / (case["n"] * case["h"] * case["w"])

    @dvm.kernel(ktype="split", dynamic=True)
    def batchnorm(k, x, gamma, beta):
        x, gamma, beta = k.load(x, dvm.float32), k.load(gamma, dvm.float32), k.load(beta, dvm.float32)
        mean = k.mul(k.sum(x, (0, 2, 3), True), inv)
        var = k.sub(k.mul(k.sum(k.mul(x, x), (0, 2, 3), True), inv), k.mul(mean, mean))
        scale = k.div(gamma, k.sqrt(k.add(var, 1e-5)))
        return k.store(k.add(k.mul(x, scale), k.sub(beta, k.mul(mean, scale))))
    return batchnorm


def _rmsnorm_kernel(case):
    dt, inv = _DVM[case["dtype"]], 1.0 / case["hidden"]

    @dvm.kernel(ktype="split", dynamic=True)
    def add_rmsnorm(k, x, residual, weight):
        h = k.cast(k.add(k.load(x, dt), k.load(residual, dt)), dvm.float32)
        rstd = k.div(1.0, k.sqrt(k.add(k.mul(k.sum(k.mul(h, h), (1,), True), inv), 1e-6)))
        return k.store(k.cast(k.mul(k.mul(h, rstd), k.load(weight, dvm.float32)), dt))
    return add_rmsnorm


def _softmax_kernel(case):
    dt = _DVM[case["dtype"]]

    @dvm.kernel(ktype="split", dynamic=True)
    def softmax(k, x):
        x = k.load(x, dt)
        if case["dtype"] != "float32":
            x = k.cast(x, dvm.float32)
        e = k.exp(k.sub(x, k.max(x, (1,), True)))
        p = k.div(e, k.sum(e, (1,), True))
        return k.store(p if case["dtype"] == "float32" else k.cast(p, dt))
    return softmax


def _adam_kernel(case):
    @dvm.kernel(ktype="split", dynamic=True)
    def adam(k, p, g, m, v, lr, eps):
        p, g, m, v = (k.load(t, dvm.float32) for t in (p, g, m, v))
        m = k.add(k.mul(m, 0.9), k.mul(g, 0.1))
        v = k.add(k.mul(v, 0.999), k.mul(k.mul(g, g), 0.001))
        p = k.sub(p, k.mul(k.div(m, k.add(k.sqrt(v), k.scalar(eps))), k.scalar(lr)))
        return k.store(p), k.store(m), k.store(v)
    return adam


def _linear_kernel(case):
    """SiLU(x W + b): the product rounded to its type, bias and activation in fp32."""
    dt = _DVM[case["dtype"]]

    @dvm.kernel(ktype="mix", dynamic=True)
    def linear(k, x, w, b):
        h = k.cast(k.matmul(k.load(x, dt), k.load(w, dt), False, case["weight_out_in"]), dvm.float32)
        h = k.add(h, k.load(b, dvm.float32))
        return k.store(k.cast(k.div(h, k.add(k.exp(k.mul(h, -1.0)), 1.0)), dt))
    return linear


def _linear_backward_kernel(case):
    dt = _DVM[case["dtype"]]

    @dvm.kernel(ktype="split", dynamic=True)
    def linear_backward(k, x, w, dy):
        x, w, dy = k.load(x, dt), k.load(w, dt), k.load(dy, dt)
        return (k.store(k.matmul(dy, w, False, True)), k.store(k.matmul(x, dy, True, False)),
                k.store(k.sum(k.cast(dy, dvm.float32), (0,), False)))
    return linear_backward


def _attention_kernel(case):
    dt, scale = _DVM[case["dtype"]], 1.0 / math.sqrt(case["d"])

    @dvm.kernel(ktype="mix", dynamic=True)
    def attention(k, q, key, value):
        s = k.cast(k.mul(k.matmul(k.load(q, dt), k.load(key, dt), False, True), scale), dvm.float32)
        e = k.exp(k.sub(s, k.max(s, (3,), True)))
        p = k.cast(k.div(e, k.sum(e, (3,), True)), dt)
        out = k.matmul(p, k.load(value, dt), False, False)
        return k.store(k.permute(out, (0, 2, 1, 3)) if case["seq_first"] else out)
    return attention


_KERNELS = {"add": _add_kernel, "batchnorm": _batchnorm_kernel, "rmsnorm": _rmsnorm_kernel, "softmax": _softmax_kernel, "adam": _adam_kernel,
            "linear": _linear_kernel, "linear_backward": _linear_backward_kernel, "attention": _attention_kernel}


def _eager_gate(x, gate, up, weight):
    """out = x + silu(gate * rmsnorm(x)) * up, plain torch."""
    h = x.float()
    rstd = torch.rsqrt((h * h).sum(-1, keepdim=True) * (1.0 / x.shape[-1]) + 1e-6)
    n = (h * rstd * weight).to(x.dtype)
    return x + torch.nn.functional.silu(gate * n) * up


# ---- inputs ----

def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, dtype="float32", scale=1.0):
        return (torch.randn(shape, device="cuda", generator=gen) * scale).to(_TORCH[dtype])

    op, dt = case["op"], case.get("dtype", "float32")
    if op == "add":
        args = [normal(case["rows"], case["cols"], dtype=dt), normal(case["rows"], case["cols"], dtype=dt)]
    elif op == "batchnorm":
        c = case["c"]
        args = [normal(case["n"], c, case["h"], case["w"]), torch.rand((1, c, 1, 1), device="cuda", generator=gen) + 0.5, normal(1, c, 1, 1, scale=0.1)]
    elif op == "rmsnorm":
        shape = (case["rows"], case["hidden"])
        args = [normal(*shape, dtype=dt), normal(*shape, dtype=dt), 1.0 + normal(case["hidden"], scale=0.1)]
    elif op == "softmax":
        args = [normal(case["rows"], case["cols"], dtype=dt, scale=2.0)]  # logits
    elif op == "adam":
        n = case["numel"]
        args = [normal(n, scale=0.02), normal(n, scale=1e-3), normal(n, scale=1e-4), normal(n, scale=1e-3) ** 2, 1e-3, 1e-8]
    elif op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        w = normal(*((n, k) if case["weight_out_in"] else (k, n)), dtype=dt, scale=1.0 / math.sqrt(k))
        args = [normal(m, k, dtype=dt), w, normal(n, scale=0.3)]
    elif op == "linear_backward":
        m, n, k = case["m"], case["n"], case["k"]
        args = [normal(m, k, dtype=dt), normal(k, n, dtype=dt, scale=1.0 / math.sqrt(k)), normal(m, n, dtype=dt)]
    elif op == "attention":
        args = []
        for tokens in (case["queries"], case["keys"], case["keys"]):
            if case["seq_first"]:  # [batch, tokens, heads, d] in memory, handed over with the heads in front
                args.append(normal(case["batch"], tokens, case["heads"], case["d"], dtype=dt).permute(0, 2, 1, 3))
            else:
                args.append(normal(case["batch"], case["heads"], tokens, case["d"], dtype=dt))
    else:
        shape = (case["rows"], case["hidden"])
        args = [normal(*shape, dtype=dt) for _ in range(3)] + [1.0 + normal(case["hidden"], scale=0.1)]
        return {"fusion": dvm.lazy_fusion(), "args": args}
    return {"kernel": _KERNELS[op](case), "args": args}


def run(state):
    if "fusion" in state:
        with state["fusion"]:
            out = _eager_gate(*state["args"])
        return out
    return state["kernel"](*state["args"])


# ---- what a pass cannot do without ----

def work(case):
    op, size = case["op"], _SIZE[case.get("dtype", "float32")]
    if op == "add":
        n = case["rows"] * case["cols"]
        return {"bytes": 3 * n * size, "flops": n}
    if op == "batchnorm":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": 8 * n + 8 * case["c"], "flops": 5 * n}
    if op == "rmsnorm":
        n = case["rows"] * case["hidden"]
        return {"bytes": 3 * n * size + 4 * case["hidden"], "flops": 5 * n}
    if op == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * size, "flops": 5 * n}
    if op == "adam":
        return {"bytes": 28 * case["numel"], "flops": 13 * case["numel"]}
    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n + m * n) * size + 4 * n, "flops": 2 * m * n * k}
    if op == "linear_backward":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n) * size + m * n * size + 4 * n, "flops": 4 * m * n * k + m * n}
    if op == "attention":
        heads, q, kv, d = case["batch"] * case["heads"], case["queries"], case["keys"], case["d"]
        return {"bytes": heads * (2 * q + 2 * kv) * d * size, "flops": 4 * heads * q * kv * d}
    n = case["rows"] * case["hidden"]
    return {"bytes": 4 * n * size + 4 * case["hidden"], "flops": 12 * n}


# Relative errors of the results against the same graphs in 64-bit floats, times about four: seen over the listed cases
# and forty drawn ones were up to 9.1e-8 (softmax), 3.2e-4 (attention in fp16), 2.6e-3 (the eager program in bf16, which
# rounds five times).
_REL = {"float32": 4e-7, "float16": 1.3e-3, "bfloat16": 1e-2}


def tolerance(case):
    if case["op"] == "add":
        return "exact"
    return {"rel": _REL[case.get("dtype", "float32")]}
