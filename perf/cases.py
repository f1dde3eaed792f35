"""The work this library does for its users, as cases to measure.

Each case is one pass of something a program built on the library does over
and over: a Linear layer's training step, the codebook head's training step,
an attention layer forward and backward, a decode step of one transformer
block, a prompt chunk against a key/value cache. Sizes are those of the model
configurations the benchmark and the tests use (widths 256, 512 and 768, head
dims 32 and 64, 16 codebooks of 1024 classes), their ragged neighbours (token
counts and widths that are no multiple of 4, as the parity tests sweep), and
what lies between.

Calls go through the C ABI with argument lists built once, as a compiled
program holds them; buffers are torch memory, and the library runs on its
context's own stream.
"""
import ctypes
import math

import torch

from staleynet_amd import gemm
from staleynet_amd.gemm import BatchStrides, CCrossEntropyHead, HeadLayout, MatmulSpec, Precision

CLASSES = 1024  # classes of one codebook
CODEBOOKS = 16

_GPU = None


def _gpu():
    """The program's one context."""
    global _GPU
    if _GPU is None:
        _GPU = gemm.Gpu(0)
    return _GPU


# ---- the cases -----------------------------------------------------------------------------------


def listed():
    return [
        # One new token of one sequence through a 111.5M-model block: the latency of autoregressive
        # decoding (four few-row products, the cache append, attention over 701 cached positions).
        dict(name="decode_block_1", kind="decode", sequences=1, width=768, heads=12, ffn=3072, cached=701,
             capacity=1408),
        # Sixteen sequences decoded together, an odd number of cached positions.
        dict(name="decode_block_16", kind="decode", sequences=16, width=768, heads=12, ffn=3072, cached=333,
             capacity=1408),
        # The 16-codebook head for one new token: one large weight streamed for a single row.
        dict(name="decode_head_1", kind="forward", tokens=1, inputs=768, outputs=CODEBOOKS * CLASSES, bf16=False),
        # A 300-token chunk of a prompt against 401 cached positions (fused forward, ragged both ways).
        dict(name="prefill_300", kind="prefill", heads=12, queries=300, cached=401, capacity=1408, head_dim=64),
        # Training steps of one Linear (y = x W + b; dW, db; dX). The small model's FFN expansion:
        # 2048 tokens, where launches and latency count.
        dict(name="linear_2048x256x1024", kind="linear", tokens=2048, inputs=256, outputs=1024, bf16=False),
        # Ragged batch and widths: 4 sequences of 701 tokens, 250 -> 1001 columns (no 16-byte rows).
        dict(name="linear_2804x250x1001", kind="linear", tokens=2804, inputs=250, outputs=1001, bf16=False),
        # The medium model's QKV projection.
        dict(name="linear_8192x512x1536", kind="linear", tokens=8192, inputs=512, outputs=1536, bf16=False),
        # The large model's QKV projection at its full batch, fp32: the heaviest use there is.
        dict(name="linear_32768x768x2304", kind="linear", tokens=32768, inputs=768, outputs=2304, bf16=False),
        # The large model's FFN expansion with the bf16-input kernels.
        dict(name="linear_bf16_32768x768x3072", kind="linear", tokens=32768, inputs=768, outputs=3072, bf16=True),
        # The medium model's 16-codebook head: logits, 16 cross-entropies, dW and dX.
        dict(name="head_8192x512", kind="head", tokens=8192, inputs=512),
        # One attention layer's training step, probability-free, at the large model's batch.
        dict(name="attention_16x12x2048x64", kind="attention", batch=16, heads=12, time=2048, head_dim=64),
        # The same step as the reference's model issues it, products and row kernels one by one with the
        # probabilities in memory, at the medium model's batch.
        dict(name="attention_calls_8x8x1024x64", kind="attention_calls", batch=8, heads=8, time=1024, head_dim=64),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A layer width: a multiple of 64, a multiple of 4, or any number."""
    n = _log_int(rng, low, high)
    step = rng.choice([64, 64, 4, 1])
    return max(step, n // step * step)


MAX_FLOPS = 3.0e11  # a drawn fp32 case stays under the largest listed one


def draw(rng):
    kind = rng.choice(["decode", "forward", "prefill", "linear", "linear", "linear", "head", "attention", "attention",
                       "attention_calls"])
    if kind == "decode":
        head_dim = rng.choice([32, 64])
        heads = rng.choice([8, 12]) if head_dim == 64 else 8
        width = heads * head_dim
        capacity = rng.choice([512, 1024, 1408, 2048])
        return dict(kind=kind, sequences=_log_int(rng, 1, 16), width=width, heads=heads, ffn=4 * width,
                    cached=rng.randint(0, capacity - 1), capacity=capacity)
    if kind == "forward":
        return dict(kind=kind, tokens=_log_int(rng, 1, 64), inputs=_width(rng, 256, 3072),
                    outputs=_width(rng, 256, CODEBOOKS * CLASSES), bf16=False)
    if kind == "prefill":
        capacity = rng.choice([512, 1024, 1408, 2048])
        queries = _log_int(rng, 5, capacity - 1)
        return dict(kind=kind, heads=rng.choice([8, 12, 48]), queries=queries,
                    cached=rng.randint(0, capacity - queries), capacity=capacity, head_dim=rng.choice([32, 64]))
    if kind == "linear":
        case = dict(kind=kind, tokens=_log_int(rng, 256, 32768), inputs=_width(rng, 128, 3072),
                    outputs=_width(rng, 128, 3072), bf16=rng.random() < 0.3)
        while work(case)["flops"] > MAX_FLOPS:
            case["tokens"] = case["tokens"] * 2 // 3
        return case
    if kind == "head":
        case = dict(kind=kind, tokens=_log_int(rng, 256, 8192), inputs=rng.choice([256, 512, 768]))
        while work(case)["flops"] > MAX_FLOPS:
            case["tokens"] = case["tokens"] * 2 // 3
        return case
    batch = _log_int(rng, 1, 16) if kind == "attention" else _log_int(rng, 1, 8)
    time = _log_int(rng, 64, 2048 if kind == "attention" else 1024)
    if rng.random() < 0.5:
        time = max(64, time // 64 * 64)
    return dict(kind=kind, batch=batch, heads=rng.choice([8, 12]) if kind == "attention" else 8, time=time,
                head_dim=rng.choice([32, 64]))


# ---- inputs --------------------------------------------------------------------------------------


class _Inputs:
    """Seeded device tensors: N(0, 1) activations and gradients, N(0, 0.02) weights, small biases."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.generator, device="cuda", dtype=torch.float32).mul_(std)

    def tokens(self, rows):
        return torch.randint(0, CLASSES, (rows, CODEBOOKS), generator=self.generator, device="cuda",
                             dtype=torch.int32)


def _inputs(case, seed):
    """The case's inputs by name, in a fixed order from the seed."""
    r = _Inputs(seed)
    kind = case["kind"]
    if kind in ("linear", "forward"):
        m, i, o = case["tokens"], case["inputs"], case["outputs"]
        got = dict(x=r.normal(m, i), w=r.normal(i, o, std=0.02), b=r.normal(o, std=0.02))
        if kind == "linear":
            got["dy"] = r.normal(m, o)
        return got
    if kind == "head":
        m, i = case["tokens"], case["inputs"]
        return dict(x=r.normal(m, i), w=r.normal(i, CODEBOOKS * CLASSES, std=0.02), targets=r.tokens(m))
    if kind == "decode":
        s, d, h, f = case["sequences"], case["width"], case["heads"], case["ffn"]
        got = dict(x=r.normal(s, d))
        for name, i, o in (("qkv", d, 3 * d), ("out", d, d), ("up", d, f), ("down", f, d)):
            got["w_" + name] = r.normal(i, o, std=0.02)
            got["b_" + name] = r.normal(o, std=0.02)
        shape = (s, h, case["capacity"], d // h)
        got["k"], got["v"] = r.normal(*shape), r.normal(*shape)
        return got
    if kind == "prefill":
        n, h = case["heads"], case["head_dim"]
        return dict(q=r.normal(n, case["queries"], h), k=r.normal(n, case["capacity"], h),
                    v=r.normal(n, case["capacity"], h))
    b, n, t, h = case["batch"], case["heads"], case["time"], case["head_dim"]
    return dict(qkv=r.normal(b * t, 3 * n * h), d_context=r.normal(b * t, n * h))


# ---- the calls -----------------------------------------------------------------------------------


class _Program:
    """A list of library calls with their arguments, and what they leave."""

    def __init__(self, tensors):
        self.gpu = _gpu()
        self.lib = gemm.library()
        self.calls = []
        self.keep = list(tensors)  # the buffers the arguments point at
        self.outputs = None

    def empty(self, *shape):
        t = torch.empty(*shape, device="cuda", dtype=torch.float32)
        self.keep.append(t)
        return t

    def add(self, name, *args):
        """Calls sn_<name>(context, ...): tensors become (pointer, length), structures references."""
        flat = [self.gpu._ctx]
        for a in args:
            if isinstance(a, torch.Tensor):
                flat += [ctypes.c_void_p(a.data_ptr()), ctypes.c_size_t(a.numel())]
            elif isinstance(a, ctypes.Structure):
                self.keep.append(a)
                flat.append(ctypes.byref(a))
            else:
                flat.append(a)
        self.calls.append((getattr(self.lib, "sn_" + name), tuple(flat)))

    def zero(self, tensor):
        self.add("fill_zero", ctypes.c_void_p(tensor.data_ptr()), tensor.numel())

    def run(self):
        for function, args in self.calls:
            status = function(*args)
            if status != 0:
                raise gemm.GpuError(status, function.__name__)
        return self.outputs


def _split(p, packed, head_major, b, t, n, h, width, column):
    p.add("split_heads", packed, head_major, HeadLayout.dense(b, t, n, h, width, column).to_c())


def _merge(p, head_major, packed, b, t, n, h, width, column):
    p.add("merge_heads", head_major, packed, HeadLayout.dense(b, t, n, h, width, column).to_c())


def _shape(heads, queries, keys, h, offset=0):
    return gemm.CAttentionShape(heads, queries, keys, h, queries * h, keys * h, offset, h ** -0.5)


def _linear(p, case, t):
    m, i, o = case["tokens"], case["inputs"], case["outputs"]
    precision = Precision.Bf16 if case["bf16"] else Precision.F32
    y = p.empty(m, o)
    p.add("matmul_bias", MatmulSpec.new(m, o, i).with_precision(precision).to_c(), t["x"], t["w"], t["b"], y)
    if case["kind"] == "forward":
        return dict(y=y)
    dw, db, dx = p.empty(i, o), p.empty(o), p.empty(m, i)
    p.zero(dw)
    p.zero(db)
    p.add("matmul_column_sums", MatmulSpec.new(i, o, m).left_transposed().accumulate().with_precision(precision).to_c(),
          t["x"], t["dy"], dw, db)
    p.add("matmul", MatmulSpec.new(m, i, o).right_transposed().with_precision(precision).to_c(), t["dy"], t["w"], dx)
    return dict(y=y, dw=dw, db=db, dx=dx)


def _head(p, case, t):
    m, i, o = case["tokens"], case["inputs"], CODEBOOKS * CLASSES
    logits, grad, losses = p.empty(m, o), p.empty(m, o), p.empty(CODEBOOKS, m)
    dw, dx = p.empty(i, o), p.empty(m, i)
    p.add("matmul", MatmulSpec.new(m, o, i).to_c(), t["x"], t["w"], logits)
    for c in range(CODEBOOKS):
        head = CCrossEntropyHead(c * CLASSES, CLASSES, CODEBOOKS, c, 1.0 / (m * CODEBOOKS))
        p.add("cross_entropy", ctypes.c_void_p(logits.data_ptr()), m, o, ctypes.c_void_p(t["targets"].data_ptr()),
              m * CODEBOOKS, head, losses[c], ctypes.c_void_p(grad.data_ptr()), m, o)
    p.zero(dw)
    p.add("matmul", MatmulSpec.new(i, o, m).left_transposed().accumulate().to_c(), t["x"], grad, dw)
    p.add("matmul", MatmulSpec.new(m, i, o).right_transposed().to_c(), grad, t["w"], dx)
    return dict(logits=logits, losses=losses, grad=grad, dw=dw, dx=dx)


def _decode(p, case, t):
    s, d, n, f = case["sequences"], case["width"], case["heads"], case["ffn"]
    h, cached, capacity = d // n, case["cached"], case["capacity"]
    qkv, q, o = p.empty(s, 3 * d), p.empty(s, n, 1, h), p.empty(s, n, 1, h)
    context, out, up, down = p.empty(s, d), p.empty(s, d), p.empty(s, f), p.empty(s, d)
    p.add("matmul_bias", MatmulSpec.new(s, 3 * d, d).to_c(), t["x"], t["w_qkv"], t["b_qkv"], qkv)
    _split(p, qkv, q, s, 1, n, h, 3 * d, 0)
    for j, cache in ((1, t["k"]), (2, t["v"])):
        p.add("split_heads", qkv, cache, HeadLayout.dense(s, 1, n, h, 3 * d, j * d).in_cache(capacity, cached).to_c())
    p.add("causal_attention", _shape(s * n, 1, capacity, h, cached), q, t["k"], t["v"], o, None, 0)
    _merge(p, o, context, s, 1, n, h, d, 0)
    p.add("matmul_bias", MatmulSpec.new(s, d, d).to_c(), context, t["w_out"], t["b_out"], out)
    p.add("matmul_bias", MatmulSpec.new(s, f, d).to_c(), out, t["w_up"], t["b_up"], up)
    p.add("matmul_bias", MatmulSpec.new(s, d, f).to_c(), up, t["w_down"], t["b_down"], down)
    return dict(qkv=qkv, k=t["k"], v=t["v"], context=context, out=out, up=up, down=down)


def _prefill(p, case, t):
    o = p.empty(case["heads"], case["queries"], case["head_dim"])
    p.add("causal_attention", _shape(case["heads"], case["queries"], case["capacity"], case["head_dim"],
                                     case["cached"]), t["q"], t["k"], t["v"], o, None, 0)
    return dict(out=o)


def _attention(p, case, t):
    b, n, time, h = case["batch"], case["heads"], case["time"], case["head_dim"]
    width = n * h
    q, k, v, o, d_o, dq, dk, dv = (p.empty(b, n, time, h) for _ in range(8))
    context, d_qkv = p.empty(b * time, width), p.empty(b * time, 3 * width)
    shape = _shape(b * n, time, time, h)
    for j, x in enumerate((q, k, v)):
        _split(p, t["qkv"], x, b, time, n, h, 3 * width, j * width)
    if case["kind"] == "attention":
        stats = p.empty(b * n, time, 2)
        p.add("causal_attention_with_stats", shape, q, k, v, o, stats)
        _merge(p, o, context, b, time, n, h, width, 0)
        _split(p, t["d_context"], d_o, b, time, n, h, width, 0)
        p.add("causal_attention_backward", shape, q, k, v, o, d_o, stats, dq, dk, dv)
        got = dict(context=context, stats=stats, d_qkv=d_qkv)
    else:
        scale = ctypes.c_float(h ** -0.5)
        rows, tt, th = b * n * time, time * time, time * h
        probabilities, d_scores = p.empty(rows, time), p.empty(rows, time)
        scores_spec = MatmulSpec.new(time, time, h).right_transposed().batched(BatchStrides(b * n, th, th, tt))
        mix_spec = MatmulSpec.new(time, h, time).batched(BatchStrides(b * n, tt, th, th))
        key_spec = mix_spec.left_transposed()
        p.add("matmul", scores_spec.causal_output().to_c(), q, k, probabilities)
        p.add("causal_softmax", ctypes.c_void_p(probabilities.data_ptr()), rows, time, time, scale, 0)
        p.add("matmul", mix_spec.causal_left().to_c(), probabilities, v, o)
        _merge(p, o, context, b, time, n, h, width, 0)
        _split(p, t["d_context"], d_o, b, time, n, h, width, 0)
        p.add("matmul", scores_spec.causal_output().to_c(), d_o, v, d_scores)
        p.add("matmul", key_spec.causal_left().to_c(), probabilities, d_o, dv)
        p.add("softmax_backward", ctypes.c_void_p(probabilities.data_ptr()), rows, time,
              ctypes.c_void_p(d_scores.data_ptr()), rows, time)
        p.add("matmul", mix_spec.causal_left().scaled(h ** -0.5).to_c(), d_scores, k, dq)
        p.add("matmul", key_spec.causal_left().scaled(h ** -0.5).to_c(), d_scores, q, dk)
        got = dict(context=context, probabilities=probabilities, d_qkv=d_qkv)
    for j, x in enumerate((dq, dk, dv)):
        _merge(p, x, d_qkv, b, time, n, h, 3 * width, j * width)
    return got


_BUILD = dict(linear=_linear, forward=_linear, head=_head, decode=_decode, prefill=_prefill, attention=_attention,
              attention_calls=_attention)


def prepare(case, seed):
    t = _inputs(case, seed)
    program = _Program(t.values())
    program.outputs = _BUILD[case["kind"]](program, case, t)
    torch.cuda.synchronize()  # torch made the inputs on its own stream
    return program


def run(state):
    return state.run()


# ---- what a pass cannot do without ------------------------------------------------------------------


def work(case):
    """Bytes: inputs read once, results written once. Flops: multiply-adds over what a causal mask shows."""
    kind = case["kind"]
    if kind in ("linear", "forward"):
        m, i, o = case["tokens"], case["inputs"], case["outputs"]
        if kind == "forward":
            return dict(bytes=4 * (m * i + i * o + o + m * o), flops=2 * m * i * o)
        return dict(bytes=4 * (2 * m * i + 2 * i * o + 2 * o + 2 * m * o), flops=6 * m * i * o)
    if kind == "head":
        m, i, o = case["tokens"], case["inputs"], CODEBOOKS * CLASSES
        return dict(bytes=4 * (2 * m * i + 2 * i * o + 2 * m * o + 2 * m * CODEBOOKS), flops=6 * m * i * o)
    if kind == "decode":
        s, d, f = case["sequences"], case["width"], case["ffn"]
        weights = 4 * d * d + 2 * d * f
        seen = 2 * s * d * (case["cached"] + 1)
        return dict(bytes=4 * (weights + seen + 2 * s * d), flops=2 * s * weights + 2 * seen)
    if kind == "prefill":
        n, q, c, h = case["heads"], case["queries"], case["cached"], case["head_dim"]
        return dict(bytes=4 * n * h * (2 * q + 2 * (q + c)), flops=4 * n * h * (q * c + q * (q + 1) // 2))
    b, n, t, h = case["batch"], case["heads"], case["time"], case["head_dim"]
    pairs = b * n * t * (t + 1) // 2
    if kind == "attention":
        return dict(bytes=4 * b * t * n * h * 8 + 8 * b * n * t, flops=2 * 6 * pairs * h)
    return dict(bytes=4 * b * t * n * h * 8 + 4 * b * n * t * t, flops=2 * 6 * pairs * h)


def tolerance(case):
    """What the order of fp32 sums changes (2-norm): four times the 0.1e-6 to 1.6e-6 by which the outputs
    of these cases differ from the 64-bit result, rounded up for the longest sums drawn (K = 32768,
    2.3e-6). bf16 inputs are rounded alike by every implementation, so they need no more."""
    return dict(rel=1e-5)


# ---- the same in 64 bits -----------------------------------------------------------------------------


def _softmax64(s, t, offset):
    keys = torch.arange(s.shape[-1], device=s.device)
    queries = torch.arange(t, device=s.device) + offset
    return torch.softmax(s.masked_fill(keys[None, :] > queries[:, None], -math.inf), -1)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("linear", "forward"):
        rounded = (lambda v: v.bfloat16().double()) if case["bf16"] else (lambda v: v.double())
        x, w = rounded(t["x"]), rounded(t["w"])
        got = dict(y=x @ w + t["b"].double())
        if kind == "linear":
            dy = rounded(t["dy"])
            got.update(dw=x.T @ dy, db=t["dy"].double().sum(0), dx=dy @ w.T)
        return got
    if kind == "head":
        m = case["tokens"]
        x, w = t["x"].double(), t["w"].double()
        logits = x @ w
        z = logits.view(m, CODEBOOKS, CLASSES)
        target = t["targets"].long()[:, :, None]
        log_p = torch.log_softmax(z, -1)
        losses = -log_p.gather(2, target)[:, :, 0].T.contiguous()
        grad = log_p.exp_()
        grad.scatter_add_(2, target, torch.full_like(target, -1, dtype=torch.float64))
        grad = grad.view(m, -1) / (m * CODEBOOKS)
        return dict(logits=logits, losses=losses, grad=grad, dw=x.T @ grad, dx=grad @ w.T)
    if kind == "decode":
        s, d, n, cached = case["sequences"], case["width"], case["heads"], case["cached"]
        h = d // n
        layer = lambda x, name: x @ t["w_" + name].double() + t["b_" + name].double()  # noqa: E731
        qkv = layer(t["x"].double(), "qkv")
        q, k_new, v_new = (part.reshape(s, n, 1, h) for part in qkv.split(d, 1))
        k = torch.cat([t["k"][:, :, :cached].double(), k_new], 2)
        v = torch.cat([t["v"][:, :, :cached].double(), v_new], 2)
        p = torch.softmax((q * k).sum(-1) * h ** -0.5, -1)
        context = (p[..., None] * v).sum(2).reshape(s, d)
        out = layer(context, "out")
        up = layer(out, "up")
        k_cache, v_cache = t["k"].double(), t["v"].double()
        k_cache[:, :, cached], v_cache[:, :, cached] = k_new[:, :, 0], v_new[:, :, 0]
        return dict(qkv=qkv, k=k_cache, v=v_cache, context=context, out=out, up=up, down=layer(up, "down"))
    if kind == "prefill":
        outs = []
        for q, k, v in zip(t["q"].double(), t["k"].double(), t["v"].double()):
            outs.append(_softmax64(q @ k.T * case["head_dim"] ** -0.5, case["queries"], case["cached"]) @ v)
        return dict(out=torch.stack(outs))
    b, n, time, h = case["batch"], case["heads"], case["time"], case["head_dim"]
    scale = h ** -0.5
    heads = lambda x: x.view(b, time, n, h).transpose(1, 2).reshape(b * n, time, h).double()  # noqa: E731
    q, k, v = (heads(part.contiguous()) for part in t["qkv"].split(n * h, 1))
    d_o = heads(t["d_context"])
    o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
    stats = torch.empty(b * n, time, 2, device=q.device, dtype=torch.float64)
    kept = torch.empty(b * n, time, time, device=q.device, dtype=torch.float64) if kind == "attention_calls" else None
    hidden = torch.ones(time, time, device=q.device, dtype=torch.bool).triu_(1)
    for i in range(b * n):
        s = (q[i] @ k[i].T * scale).masked_fill_(hidden, -math.inf)
        stats[i, :, 0] = s.max(-1).values
        p = (s - stats[i, :, :1]).exp_()
        stats[i, :, 1] = p.sum(-1)
        p /= stats[i, :, 1:]
        if kept is not None:
            kept[i] = p
        o[i] = p @ v[i]
        dv[i] = p.T @ d_o[i]
        ds = p * (d_o[i] @ v[i].T - (d_o[i] * o[i]).sum(-1, keepdim=True))
        dq[i] = ds @ k[i] * scale
        dk[i] = ds.T @ q[i] * scale
    packed = lambda x: x.view(b, n, time, h).transpose(1, 2).reshape(b * time, n * h)  # noqa: E731
    got = dict(context=packed(o), d_qkv=torch.cat([packed(dq), packed(dk), packed(dv)], 1))
    if kind == "attention":
        got["stats"] = stats
    else:
        got["probabilities"] = kept.view(b * n * time, time)
    return got
