"""The work this library does for a program, as measurable cases.

A case is one call of a public entry point:

``matmul``     ``nya_hip_matmul`` (``fyodor_amd.hip.Kernels.matmul``) on
               device buffers: Y = X W^T for one weight matrix in the
               library's layout, a batch of fp32 activations.
``attention``  ``nya_hip_attention``: a run of prompt tokens over the cached
               keys and values, causal, optionally with a local window.
``split``      ``nya_hip_attention_split``: decode or verification tokens
               over a long cache.
``prompt``     ``fyodor_amd.model.Plan.prefill`` on a resident model: a
               prompt, with the last token's logits.
``decode``     ``Plan.token``: one token with its logits.
``verify``     ``Plan.verify``: a pending token and draft proposals in one
               batch, with every row of logits and the greedy choices.

Sizes are the ones the benchmark, the tests and the decoder shapes of this
repository use, and their neighbours. Weights are the seeded GGUF blocks of
``fyodor_amd.synth``; activations are normal with a per-channel spread, as a
decoder's normalized residual has.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from fyodor_amd import BF16, F16, F32, Q4_0, Q4_K, Q6_K, Q8_0, Compute, storage_bytes, synth
from fyodor_amd.hip import Kernels
from fyodor_amd.model import LlamaModel, LlamaShape, Plan, llama_tensors

TYPES = {"F32": F32, "F16": F16, "BF16": BF16, "Q4_0": Q4_0, "Q8_0": Q8_0, "Q4_K": Q4_K, "Q6_K": Q6_K}

# Decoder shapes of the resident plan: embedding, query heads, KV heads,
# feed-forward length. Both use Q4_K attention / gate / up and Q6_K down /
# output, and a 32000-entry vocabulary.
SHAPES = {"tinyllama-1.1b": (2048, 32, 4, 5632), "llama-8b": (4096, 32, 8, 14336)}
VOCABULARY = 32000


def listed():
    return [
        # The smallest product of a decode step: one token's key (or value)
        # projection of an 8B-class block. Bound by its launch.
        {"name": "decode-kv", "op": "matmul", "type": "Q4_K", "rows": 1024, "cols": 4096, "batch": 1},
        # The benchmark's headline: one token's feed-forward gate (or up).
        {"name": "decode-ffn", "op": "matmul", "type": "Q4_K", "rows": 14336, "cols": 4096, "batch": 1},
        # A pending token and seven draft proposals through a down product.
        {"name": "draft-8", "op": "matmul", "type": "Q4_0", "rows": 4096, "cols": 11008, "batch": 8},
        # The largest verification window (32 proposals) through a down product.
        {"name": "verify-33", "op": "matmul", "type": "Q6_K", "rows": 4096, "cols": 14336, "batch": 33},
        # A prompt chunk of the resident plan: gate (or up), then down.
        {"name": "prompt-ffn", "op": "matmul", "type": "Q4_K", "rows": 14336, "cols": 4096, "batch": 512},
        {"name": "prompt-down", "op": "matmul", "type": "Q6_K", "rows": 4096, "cols": 14336, "batch": 512},
        # The largest call: a long prompt in one product, 8-bit weights.
        {"name": "prompt-2048", "op": "matmul", "type": "Q8_0", "rows": 11008, "cols": 4096, "batch": 2048},
        # An unquantized model's projection over a prompt of odd length.
        {"name": "prompt-f16", "op": "matmul", "type": "F16", "rows": 4096, "cols": 4096, "batch": 333},
        # The last 512-token chunk of a 4096-token prompt: an 8B-class block's
        # attention.
        {"name": "attention-512", "op": "attention", "heads": 32, "kv_heads": 8, "width": 128, "first": 3584,
         "count": 512, "capacity": 4096, "window": 0},
        # One decode token's attention at the end of the same context.
        {"name": "attention-1", "op": "split", "heads": 32, "kv_heads": 8, "width": 128, "first": 4095, "count": 1,
         "capacity": 4096, "window": 0},
        # A whole model over a prompt, and one decode token of a model whose
        # weights do not fit the last-level cache (a quarter of an 8B's
        # blocks: the same work per block).
        {"name": "model-prompt", "op": "prompt", "shape": "tinyllama-1.1b", "blocks": 22, "first": 0, "count": 512},
        {"name": "model-decode", "op": "decode", "shape": "llama-8b", "blocks": 8, "first": 640, "count": 1},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choices(["matmul", "attention", "split", "prompt", "decode", "verify"], [10, 2, 1, 1, 1, 1])[0]
    if op == "matmul":
        t = rng.choices(["Q4_K", "Q6_K", "Q8_0", "Q4_0", "F16", "BF16", "F32"], [6, 4, 3, 2, 1, 1, 1])[0]
        step = 256 if t in ("Q4_K", "Q6_K") else 32 if t in ("Q8_0", "Q4_0") else 2
        cols = max(4, _log(rng, 1024, 16384) // step) * step
        rows = _log(rng, 256, 32768)
        # One token and small windows as often as prompts.
        batch = rng.choice([1, rng.randint(2, 8), rng.randint(9, 64), _log(rng, 65, 2048)])
        # At most the largest listed call's work.
        while rows * cols * batch > 11008 * 4096 * 2048:
            rows, batch = max(256, rows // 2), max(1, batch // 2 + 1)
        return {"op": op, "type": t, "rows": rows, "cols": cols, "batch": batch}
    if op in ("attention", "split"):
        heads, kv_heads, width = rng.choice([(32, 8, 128), (32, 4, 64), (16, 8, 256), (32, 32, 128)])
        capacity = _log(rng, 512, 4096)
        if op == "split":
            count = rng.choice([1, 1, rng.randint(2, 33)])
            first = rng.randint(min(320, capacity - count), capacity - count)
        else:
            count = min(capacity, _log(rng, 9, 512))
            first = rng.randint(0, capacity - count)
        return {"op": op, "heads": heads, "kv_heads": kv_heads, "width": width, "first": first, "count": count,
                "capacity": capacity, "window": rng.choice([0, 0, 1024])}
    shape, blocks = rng.choice([("tinyllama-1.1b", rng.randint(4, 22)), ("llama-8b", rng.randint(2, 4))])
    count = _log(rng, 2, 512) if op == "prompt" else 1 if op == "decode" else rng.randint(2, 33)
    return {"op": op, "shape": shape, "blocks": blocks, "first": 0 if op == "prompt" else _log(rng, 8, 1024),
            "count": count}


# ---- inputs ---------------------------------------------------------------

def _normal(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda")


def _activations(batch, cols, seed):
    spread = torch.exp(0.5 * _normal((cols,), 2 * seed + 1))
    return _normal((batch, cols), 2 * seed) * spread


def _attention_inputs(case, seed):
    row = case["kv_heads"] * case["width"]
    # Scores with a standard deviation of 2 under the 1 / sqrt(width) scale.
    q = 2.0 * _normal((case["count"], case["heads"] * case["width"]), 3 * seed)
    keys = _normal((case["capacity"], row), 3 * seed + 1)
    values = _normal((case["capacity"], row), 3 * seed + 2)
    return q, keys, values


def _tokens(case, seed):
    rng = np.random.default_rng(seed)
    return [int(t) for t in rng.integers(0, VOCABULARY, case["first"] + case["count"])]


def _llama(case, seed):
    d, heads, kv, hidden = SHAPES[case["shape"]]
    return LlamaShape(embedding=d, heads=heads, kv_heads=kv, hidden=hidden, blocks=case["blocks"],
                      context=case["first"] + case["count"] + 1, vocabulary=VOCABULARY, seed=1 + seed)


class _Model:
    """A resident plan with its cache filled up to the case's first position."""

    def __init__(self, case, seed):
        shape = _llama(case, seed)
        # The blocks share host arrays; the plan uploads each block's own copy.
        self.model = LlamaModel(shape, llama_tensors(shape, shared_blocks=True))
        self.compute = Compute("rocm")
        self.plan = Plan(self.compute, self.model, shape.context)
        self.first, self.tokens = case["first"], _tokens(case, seed)[case["first"]:]
        if self.first:
            self.plan.prefill(_tokens(case, seed)[:self.first], 0)

    def __del__(self):
        if hasattr(self, "plan"):
            self.plan.close()
        if hasattr(self, "compute"):
            self.compute.close()


_library = None


def _kernels():
    """The kernel library, with the attention entry points declared."""
    global _library
    if _library is None:
        k = Kernels()
        u, z = ctypes.c_size_t, ctypes.c_size_t
        k.lib.nya_hip_attention.argtypes = [u, z, u, u, u, u, u, z, z, z, z, z, z, ctypes.c_float, u]
        k.lib.nya_hip_attention_split.argtypes = [u, z, u, u, u, u, u, z, z, z, z, z, z, z, ctypes.c_float, u]
        _library = k
    return _library


def prepare(case, seed):
    op = case["op"]
    if op in ("prompt", "decode", "verify"):
        return op, _Model(case, seed)
    k = _kernels()
    if op == "matmul":
        t, rows, cols, batch = TYPES[case["type"]], case["rows"], case["cols"], case["batch"]
        w = torch.from_numpy(k.device_weights(synth.weights(t, rows, cols, seed), t, rows, cols)).cuda()
        x = _activations(batch, cols, seed)
        y = torch.empty((batch, rows), device="cuda")
        workspace = torch.empty(max(16, k.workspace_bytes(t, rows, cols, batch)), dtype=torch.uint8, device="cuda")
        return op, (k, w, t, rows, cols, x, y, batch, workspace)
    q, keys, values = _attention_inputs(case, seed)
    positions = torch.arange(case["first"], case["first"] + case["count"], dtype=torch.int32, device="cuda")
    out = torch.empty_like(q)
    splits, partials = 0, None
    if op == "split":
        # As the resident plan chooses them.
        splits = min(64, max(8, 512 // case["kv_heads"]))
        partials = torch.empty(case["count"] * case["heads"] * splits * (case["width"] + 2), device="cuda")
    return op, (k, q, keys, values, out, partials, positions, case["count"], case["heads"], case["kv_heads"],
                case["width"], case["capacity"], case["window"], splits, 1.0 / math.sqrt(case["width"]))


def run(state):
    op, s = state
    if op == "matmul":
        k, w, t, rows, cols, x, y, batch, workspace = s
        k.matmul(w.data_ptr(), t, rows, cols, x.data_ptr(), y.data_ptr(), batch, workspace.data_ptr(),
                 workspace.numel(), torch.cuda.current_stream().cuda_stream)
        return y
    if op in ("attention", "split"):
        k, q, keys, values, out, partials, positions, count, heads, kv_heads, width, capacity, window, splits, scale = s
        stream = torch.cuda.current_stream().cuda_stream
        if op == "attention":
            status = k.lib.nya_hip_attention(q.data_ptr(), heads * width, keys.data_ptr(), values.data_ptr(),
                                             out.data_ptr(), 0, positions.data_ptr(), count, heads, kv_heads, width,
                                             capacity, window, scale, stream)
        else:
            status = k.lib.nya_hip_attention_split(q.data_ptr(), heads * width, keys.data_ptr(), values.data_ptr(),
                                                   out.data_ptr(), partials.data_ptr(), positions.data_ptr(), count,
                                                   heads, kv_heads, width, capacity, window, splits, scale, stream)
        if status:
            raise RuntimeError(f"attention returned {status}")
        return out
    if op == "prompt":
        return s.plan.prefill(s.tokens, s.first)
    if op == "decode":
        return s.plan.token(s.tokens[0], s.first)
    ids, logits = s.plan.verify(s.tokens, s.first, logits=True)
    return {"ids": np.asarray(ids, np.int64), "logits": logits}


# ---- what a pass cannot do without ----------------------------------------

def _lengths(case):
    """(positions each token attends, cached positions any of them reads)."""
    w = case.get("window", 0)
    ends = range(case["first"], case["first"] + case["count"])
    lengths = [min(p + 1, w) if w else p + 1 for p in ends]
    return lengths, ends[-1] - max(0, ends[0] - lengths[0] + 1) + 1


def work(case):
    if case["op"] == "matmul":
        r, c, n = case["rows"], case["cols"], case["batch"]
        return {"bytes": storage_bytes(TYPES[case["type"]], r, c) + 4 * n * (r + c), "flops": 2 * r * c * n}
    lengths, span = _lengths(case)
    n = case["count"]
    if case["op"] in ("attention", "split"):
        q, kv = case["heads"] * case["width"], case["kv_heads"] * case["width"]
        return {"bytes": 4 * (2 * n * q + 2 * span * kv), "flops": 4 * q * sum(lengths)}
    d, heads, kv_heads, h = SHAPES[case["shape"]]
    kv = kv_heads * (d // heads)
    attention, gate_up = (d + 2 * kv + d) * d, 2 * h * d
    head_rows = n if case["op"] == "verify" else 1
    block = storage_bytes(Q4_K, 1, attention + gate_up) + storage_bytes(Q6_K, 1, h * d)
    return {"bytes": case["blocks"] * (block + 4 * 2 * kv * (span + n)) + storage_bytes(Q6_K, VOCABULARY, d) +
            4 * VOCABULARY * head_rows,
            "flops": case["blocks"] * (2 * n * (attention + gate_up + h * d) + 4 * d * sum(lengths)) +
            2 * VOCABULARY * d * head_rows}


def tolerance(case):
    # Four times the largest error against 64 bits seen over the listed and
    # drawn cases (1.1e-6, fp32 sums in whatever order).
    return {"rel": 5e-6}


# ---- the same in 64 bits, without the library ------------------------------

def _half(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _decode(raw, t, rows, cols):
    """[rows][cols] float64 of GGUF storage."""
    raw = torch.from_numpy(raw).cuda()
    if t == F32:
        return raw.view(torch.float32).reshape(rows, cols).double()
    if t == F16:
        return raw.view(torch.float16).reshape(rows, cols).double()
    if t == BF16:
        return raw.view(torch.bfloat16).reshape(rows, cols).double()
    if t == Q8_0:
        b = raw.reshape(-1, 34)
        return (_half(b, 0) * b[:, 2:].contiguous().view(torch.int8)).reshape(rows, cols)
    if t == Q4_0:
        b = raw.reshape(-1, 18)
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0
        return (_half(b, 0) * q).reshape(rows, cols)
    if t == Q4_K:
        b = raw.reshape(-1, 144)
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, s[:, 8:12] >> 4 | (s[:, 4:8] >> 6) << 4], 1).double()
        qs = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        return ((_half(b, 0) * sc)[..., None] * q - (_half(b, 2) * mn)[..., None]).reshape(rows, cols)
    b = raw.reshape(-1, 210)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    low = torch.cat([ql & 15, ql >> 4], 2)
    high = torch.stack([qh >> (2 * i) & 3 for i in range(4)], 2)
    q = (low | high << 4).reshape(-1, 16, 16).double() - 32.0
    sc = b[:, 192:208].contiguous().view(torch.int8)
    return ((_half(b, 208) * sc)[..., None] * q).reshape(rows, cols)


def _attend(q, keys, values, positions, heads, kv_heads, window, scale):
    """Causal attention of q [n][heads * width] over rows of keys / values."""
    n, width = q.shape[0], q.shape[1] // heads
    t = torch.arange(keys.shape[0], device=q.device)
    seen = t[None, :] <= positions[:, None]
    if window:
        seen &= t[None, :] > positions[:, None] - window
    out = torch.empty(n, heads, width, dtype=q.dtype, device=q.device)
    for h in range(heads):
        g = h // (heads // kv_heads)
        k, v = keys[:, g * width:(g + 1) * width], values[:, g * width:(g + 1) * width]
        s = (q[:, h * width:(h + 1) * width] @ k.T) * scale
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ v
    return out.reshape(n, heads * width)


def _exact_model(case, seed):
    shape = _llama(case, seed)
    # Blocks share their tensors: each is decoded once.
    weights = {name: (_decode(data, t, dims[1], dims[0]) if len(dims) > 1 else _decode(data, t, 1, dims[0])[0])
               for name, t, dims, data in llama_tensors(shape, shared_blocks=True)
               if name.startswith(("token_embd", "output", "blk.0."))}
    tokens = torch.tensor(_tokens(case, seed), device="cuda")
    n, d, heads = len(tokens), shape.embedding, shape.heads
    width = d // heads
    position = torch.arange(n, device="cuda")

    def norm(v, name):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + shape.epsilon) * weights[name]

    pairs = width // 2
    angle = position[:, None] * shape.rope_base ** (-torch.arange(pairs, device="cuda", dtype=torch.float64) / pairs)
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rotate(v):
        v = v.reshape(n, -1, pairs, 2)
        a, b = v[..., 0], v[..., 1]
        return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(n, -1)

    x = weights["token_embd.weight"][tokens]
    for _ in range(shape.blocks):
        w = lambda name: weights[f"blk.0.{name}.weight"]
        a = norm(x, "blk.0.attn_norm.weight")
        att = _attend(rotate(a @ w("attn_q").T), rotate(a @ w("attn_k").T), a @ w("attn_v").T, position, heads,
                      shape.kv_heads, 0, 1.0 / math.sqrt(width))
        x = x + att @ w("attn_output").T
        f = norm(x, "blk.0.ffn_norm.weight")
        x = x + (torch.nn.functional.silu(f @ w("ffn_gate").T) * (f @ w("ffn_up").T)) @ w("ffn_down").T
    rows = x[case["first"]:] if case["op"] == "verify" else x[-1:]
    logits = norm(rows, "output_norm.weight") @ weights["output.weight"].T
    return {"ids": None, "logits": logits} if case["op"] == "verify" else logits[0]


def exact(case, seed):
    if case["op"] == "matmul":
        t, rows, cols = TYPES[case["type"]], case["rows"], case["cols"]
        return _activations(case["batch"], cols, seed).double() @ _decode(synth.weights(t, rows, cols, seed), t, rows,
                                                                         cols).T
    if case["op"] in ("attention", "split"):
        q, keys, values = (v.double() for v in _attention_inputs(case, seed))
        positions = torch.arange(case["first"], case["first"] + case["count"], device="cuda")
        return _attend(q, keys, values, positions, case["heads"], case["kv_heads"], case["window"],
                       1.0 / math.sqrt(case["width"]))
    return _exact_model(case, seed)
