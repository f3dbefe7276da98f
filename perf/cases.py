"""What this framework is timed on: the calls a user's program makes, over the sizes it makes them at.

A case is one call of a public entry point on operands already on the GPU: a whole forward of the
24-layer model (``Qwen2.forward``), or one layer's piece of it through the C entry points that
``include/nc_hip.h`` declares (``hip.call``), in the per-token int8 mode and in the reference's own
modes (``int8``, ``int8-vnni``, ``f32``). Sizes are the model's (hidden 896, intermediate 4,864, 14
query heads over 2 KV heads of 64, vocabulary 151,936) and generic ones around them.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from nanocompile_amd import hip
from nanocompile_amd.kernels import attention_workspace_bytes, float_bits, pack_chains, pack_chains_vnni
from nanocompile_amd.models.config import Qwen2Config
from nanocompile_amd.models.qwen2 import Qwen2, inverse_frequencies

EPS = 1e-6
H, I, HEADS, KV, D, V, LAYERS = 896, 4864, 14, 2, 64, 151936, 24
QKV = (HEADS + 2 * KV) * D
BLOCK = 32                                     # int8-vnni's activation block


def listed():
    return [
        # Serving: one token through the whole model into a held cache, logits out (the greedy loop's step).
        {"name": "step past 383", "kind": "forward", "tokens": 1, "past": 383},
        # A prompt's first forward, the last row's logits out.
        {"name": "prompt 512", "kind": "forward", "tokens": 512, "past": 0},
        # The smallest call: one projection of one token (gate's shape), where latency and the launch count.
        {"name": "token linear 1", "kind": "linear", "mode": "token", "rows": 1, "n": I, "k": H, "residual": False},
        # A long prompt's (or a batch of prompts') down projection with its residual.
        {"name": "token linear 2048", "kind": "linear", "mode": "token", "rows": 2048, "n": H, "k": I,
         "residual": True},
        # Gate and up with SwiGLU over a ragged prompt.
        {"name": "swiglu 1000", "kind": "swiglu", "rows": 1000, "n": I, "k": H},
        # The norm before a projection, with its per-token quantizer.
        {"name": "norm 512", "kind": "norm", "rows": 512, "k": H},
        # A long prompt's attention (with the int8 of its result, as the o projection takes it).
        {"name": "attention 2048", "kind": "attention", "rows": 2048, "past": 0, "heads": HEADS, "kv": KV, "dim": D},
        # One token's attention deep in a long context, RoPE and the cache append included.
        {"name": "decode attention 6000", "kind": "decode_attention", "past": 6000, "heads": HEADS, "kv": KV,
         "dim": D},
        # Logits of every row of a prompt (forward's default, as perplexity is measured).
        {"name": "head 128", "kind": "linear", "mode": "f32", "rows": 128, "n": V, "k": H, "residual": False},
        # The reference's int8 mode: a prompt's gate projection (float activations, int8 weights).
        {"name": "int8 linear 128", "kind": "linear", "mode": "int8", "rows": 128, "n": I, "k": H,
         "residual": False},
        # The reference's int8-vnni mode: a prompt's down projection, its block quantizer included.
        {"name": "vnni linear 128", "kind": "linear", "mode": "vnni", "rows": 128, "n": H, "k": I,
         "residual": True},
        # The reference modes' attention over a prompt.
        {"name": "reference attention 128", "kind": "reference_attention", "rows": 128, "past": 0, "heads": HEADS,
         "kv": KV, "dim": D},
    ]


def _log(rng, low, high):
    """A whole number, its logarithm spread evenly over low .. high."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _heads(rng):
    # the model's heads, and others the kernels take: even groups, one head a group, the small widths
    return rng.choice([(HEADS, KV, D), (HEADS, KV, D), (12, 2, 64), (16, 8, 64), (8, 8, 64), (32, 4, 64), (8, 2, 32)])


def _widths(rng, k_step, k_max):
    """(n, k): the model's projections half of the time, else generic ones (k a multiple of k_step)."""
    if rng.random() < 0.5:
        return rng.choice([(QKV, H), (H, H), (I, H), (H, I)])
    return _log(rng, 64, 8192), k_step * _log(rng, max(1, 128 // k_step), k_max // k_step)


def draw(rng):
    kind = rng.choice(["forward", "token", "token", "swiglu", "norm", "attention", "decode_attention", "f32", "int8",
                       "vnni", "reference_attention"])
    if kind == "forward":
        if rng.random() < 0.5:
            return {"kind": "forward", "tokens": 1, "past": _log(rng, 1, 2048)}
        return {"kind": "forward", "tokens": _log(rng, 2, 512), "past": rng.choice([0, 0, _log(rng, 1, 512)])}
    if kind == "token":
        n, k = _widths(rng, 16, 8192)
        rows = _log(rng, 1, max(1, min(4096, (1 << 34) // (n * k))))
        return {"kind": "linear", "mode": "token", "rows": rows, "n": n, "k": k, "residual": rng.random() < 0.5}
    if kind == "swiglu":
        n, k = rng.choice([(I, H), (I, H), (_log(rng, 128, 8192), 16 * _log(rng, 8, 256))])
        return {"kind": "swiglu", "rows": _log(rng, 1, max(1, min(4096, (1 << 34) // (n * k)))), "n": n, "k": k}
    if kind == "norm":
        return {"kind": "norm", "rows": _log(rng, 1, 8192), "k": rng.choice([H, H, 4 * _log(rng, 32, 2048)])}
    if kind == "f32":
        # the float32 model's projections, and the head over a few rows to a prompt
        if rng.random() < 0.5:
            return {"kind": "linear", "mode": "f32", "rows": _log(rng, 1, 128), "n": V, "k": H, "residual": False}
        n, k = _widths(rng, 16, 8192)
        return {"kind": "linear", "mode": "f32", "rows": _log(rng, 1, 512), "n": n, "k": k,
                "residual": rng.random() < 0.5}
    if kind in ("int8", "vnni"):
        n, k = _widths(rng, 16 if kind == "int8" else BLOCK, 8192)
        return {"kind": "linear", "mode": kind, "rows": _log(rng, 1, 512), "n": n, "k": k,
                "residual": rng.random() < 0.5}
    heads, kv, dim = _heads(rng)
    if kind == "decode_attention":
        return {"kind": kind, "past": _log(rng, 1, 16000), "heads": heads, "kv": kv, "dim": dim}
    if kind == "attention":
        rows = _log(rng, 2, 2048)
        past = rng.choice([0, _log(rng, 1, 8192)])
        return {"kind": kind, "rows": rows, "past": min(past, (1 << 21) // rows), "heads": heads, "kv": kv, "dim": dim}
    rows = _log(rng, 1, 512)
    past = rng.choice([0, _log(rng, 1, 2048)])
    return {"kind": kind, "rows": rows, "past": min(past, (1 << 17) // rows), "heads": heads, "kv": kv, "dim": dim}


# -- inputs ---------------------------------------------------------------------------


class _Made:
    """Seeded arrays on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed * 2 + 1)

    def normal(self, *shape, std=1.0):
        return torch.empty(shape, device="cuda").normal_(0.0, std, generator=self.g)

    def bytes(self, *shape):
        """int8 weights as the per-row quantizer leaves normal ones: bell-shaped, each row's largest 127."""
        q = torch.empty(shape, device="cuda").normal_(0.0, 36.0, generator=self.g).round_().clamp_(-127, 127)
        q[..., 0] = 127
        return q.to(torch.int8)

    def scales(self, n):
        """Weight rows of deviation 0.02 put their scales near 0.02 * 3.5 / 127."""
        return torch.empty((n,), device="cuda").uniform_(4e-4, 7e-4, generator=self.g)

    def activations(self, rows, k):
        """Normal with one element in a hundred twenty times larger, as a residual stream has."""
        x = self.normal(rows, k)
        big = torch.empty((rows, k), device="cuda").uniform_(generator=self.g) < 0.01
        return torch.where(big, 20 * x, x)

    def tokens(self, rows, k):
        """Per-token int8 activations of such rows, and their scales."""
        x = self.normal(rows, k)
        s = x.abs().amax(1) / 127
        return (x / s[:, None]).round().to(torch.int8), s


def _host(t):
    return t.cpu().numpy()


def _model(made, tokens):
    """The model's weights as an already quantized checkpoint holds them, loaded."""
    weights = {"model.embed_tokens.weight": _host(made.normal(V, H, std=0.02)),
               "model.norm.weight": _host(1 + made.normal(H, std=0.1))}
    for i in range(LAYERS):
        p = f"model.layers.{i}"
        weights[f"{p}.input_layernorm.weight"] = _host(1 + made.normal(H, std=0.1))
        weights[f"{p}.post_attention_layernorm.weight"] = _host(1 + made.normal(H, std=0.1))
        for name, n, k in (("self_attn.q_proj", HEADS * D, H), ("self_attn.k_proj", KV * D, H),
                           ("self_attn.v_proj", KV * D, H), ("self_attn.o_proj", H, HEADS * D),
                           ("mlp.gate_proj", I, H), ("mlp.up_proj", I, H), ("mlp.down_proj", H, I)):
            weights[f"{p}.{name}.weight@int8"] = _host(made.bytes(n, k))
            weights[f"{p}.{name}.weight@scales"] = _host(made.scales(n))
            if name[-6:-5] in "qkv" and name.startswith("self_attn"):
                weights[f"{p}.{name}.bias"] = _host(made.normal(n, std=0.1))
    config = Qwen2Config(vocab_size=V, hidden_size=H, intermediate_size=I, num_hidden_layers=LAYERS,
                         num_attention_heads=HEADS, num_key_value_heads=KV, rms_norm_eps=EPS, rope_theta=1e6,
                         tie_word_embeddings=True)
    return Qwen2(config, weights, max_tokens=max(512, tokens)), weights


def _forward_inputs(case, seed):
    made = _Made(seed)
    m, past = case["tokens"], case["past"]
    model, weights = _model(made, m)
    ids = _host(torch.randint(0, V, (m,), device="cuda", generator=made.g))
    keys, values = (_host(made.normal(LAYERS, KV, past, D)) for _ in "kv")
    return model, weights, ids, keys, values


def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    if kind == "forward":
        model, _, ids, keys, values = _forward_inputs(case, seed)
        m, past = case["tokens"], case["past"]
        cache = model.new_cache(past + m + 128)        # room for the answer, as a caller's sequence has
        whole = np.zeros(cache.keys.shape, np.float32)
        for part, into in ((keys, cache.keys), (values, cache.values)):
            whole[:, :, :past] = part
            into.upload(whole)
        return {"model": model, "cache": cache, "ids": ids, "past": past}
    inputs = _operands(case, seed)
    calls, outputs = _calls(case, inputs)
    torch.cuda.synchronize()
    return {"calls": calls, "outputs": outputs, "keep": inputs}


def _operands(case, seed):
    made, kind = _Made(seed), case["kind"]
    if kind in ("linear", "swiglu"):
        m, n, k = case["rows"], case["n"], case["k"]
        if kind == "swiglu":
            xq, xs = made.tokens(m, k)
            return {"xq": xq, "xs": xs, "qg": made.bytes(n, k), "sg": made.scales(n), "qu": made.bytes(n, k),
                    "su": made.scales(n)}
        got = {"bias": made.normal(n) if n != V else None,
               "residual": made.normal(m, n) if case["residual"] else None}
        if case["mode"] == "f32":
            return {**got, "x": made.normal(m, k), "w": made.normal(n, k, std=0.02)}
        got.update(q=made.bytes(n, k), scales=made.scales(n))
        if case["mode"] == "token":
            got["xq"], got["xs"] = made.tokens(m, k)
        else:
            got["x"] = made.normal(m, k)
        return got
    if kind == "norm":
        return {"x": made.activations(case["rows"], case["k"]), "gamma": 1 + made.normal(case["k"], std=0.1)}
    heads, kv, dim, past = case["heads"], case["kv"], case["dim"], case["past"]
    rows = case.get("rows", 1)
    capacity = past + rows + (64 if kind == "decode_attention" else 0)
    got = {"qkv": made.normal(rows, (heads + 2 * kv) * dim), "keys": made.normal(kv, capacity, dim),
           "values": made.normal(kv, capacity, dim)}
    if kind == "decode_attention":
        got["inv"] = torch.from_numpy(inverse_frequencies(dim, 1e6)).cuda()
    return got


def _calls(case, x):
    """One pass as (entry point, pointers, sizes), and its outputs."""
    kind = case["kind"]
    at = lambda t: None if t is None else t.data_ptr()                                   # noqa: E731
    new = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device="cuda")   # noqa: E731
    if kind == "norm":
        m, k = case["rows"], case["k"]
        xq, xs = new(m, k, dtype=torch.int8), new(m)
        return [("nc_rms_norm_quant", [None, at(xq), at(xs), at(x["x"]), at(x["gamma"])], [m, k, float_bits(EPS)])], \
            [xq, xs]
    if kind == "swiglu":
        m, n, k = case["rows"], case["n"], case["k"]
        h = new(m, n)
        return [("nc_matmul_i8_token_swiglu", [at(h), *(at(x[s]) for s in ("xq", "xs", "qg", "sg", "qu", "su"))],
                 [m, n, k, 0])], [h]
    if kind == "linear":
        m, n, k, mode = case["rows"], case["n"], case["k"], case["mode"]
        y = new(m, n)
        tail = [at(x["bias"]), at(x["residual"])]
        if mode == "token":
            return [("nc_matmul_i8_token", [at(y), at(x["xq"]), at(x["xs"]), at(x["q"]), at(x["scales"]), *tail],
                     [m, n, k, 0])], [y]
        torch.cuda.synchronize()                       # the operands are read on another stream from here on
        if mode == "f32":
            x["packed"] = new(-(-n // 64) * 64, k)
            hip.call("nc_pack_rows64", [at(x["packed"]), at(x["w"])], [n, k])
            hip.sync()
            return [("nc_lm_head", [at(y), None, at(x["x"]), at(x["packed"]), None, *tail], [m, n, k, 0])], [y]
        pack = pack_chains if mode == "int8" else pack_chains_vnni
        packed = pack(_host(x["q"])).reshape(-1)
        x["packed"] = torch.from_numpy(packed).cuda() if packed.size else new(16, dtype=torch.int8)
        weight = [at(x["packed"]), at(x["q"]), at(x["scales"]), *tail]
        if mode == "int8":
            return [("nc_matmul_i8", [at(y), at(x["x"]), *weight], [m, n, k])], [y]
        x["xq"], x["xsb"], x["offset"] = new(m, k, dtype=torch.int8), new(m, k // BLOCK), new(m)
        blocks = [at(x["xq"]), at(x["xsb"]), at(x["offset"])]
        return [("nc_quantize_blocks", [*blocks, at(x["x"])], [m, k, BLOCK]),
                ("nc_matmul_i8_vnni", [at(y), *blocks, *weight], [m, n, k, BLOCK])], [y]
    heads, kv, dim, past = case["heads"], case["kv"], case["dim"], case["past"]
    rows = case.get("rows", 1)
    capacity = x["keys"].shape[1]
    scale = float_bits(float(np.float32(dim ** -0.5)))
    ctx = new(rows, heads * dim)
    if kind == "reference_attention":
        return [("nc_attention_index_order", [at(ctx), at(x["qkv"]), at(x["keys"]), at(x["values"]), None],
                 [rows, heads, kv, dim, past, capacity, scale])], [ctx]
    per_row = attention_workspace_bytes(heads, dim, 1, past + rows)
    bytes_ = per_row * max(1, min(rows, (64 << 20) // per_row))          # a cache's workspace: at most 64 MiB
    x["work"] = new(bytes_ // 4)
    if kind == "decode_attention":
        x["table"] = new(2, capacity, dim // 2)
        torch.cuda.synchronize()
        hip.call("nc_rope_table", [at(x["table"]), at(x["inv"])], [capacity, dim])
        hip.sync()
        return [("nc_attention_decode", [at(ctx), at(x["qkv"]), at(x["keys"]), at(x["values"]), at(x["inv"]), None,
                                         at(x["table"]), at(x["work"])],
                 [heads, kv, dim, past, capacity, scale, bytes_])], \
            [ctx, x["keys"][:, past], x["values"][:, past]]
    xq, xs = new(rows, heads * dim, dtype=torch.int8), new(rows)
    return [("nc_attention", [at(ctx), at(x["qkv"]), at(x["keys"]), at(x["values"]), None, at(x["work"]), at(xq),
                              at(xs)], [rows, heads, kv, dim, past, capacity, scale, bytes_, 0])], [ctx, xq, xs]


def run(state):
    if "model" in state:
        state["cache"].length = state["past"]          # the same step of the same sequence again
        return state["model"].forward(state["ids"], state["cache"], last_only=True)
    for name, pointers, sizes in state["calls"]:
        hip.call(name, pointers, sizes)
    return state["outputs"]


# -- what a pass cannot do without, and what it should give -----------------------------


def work(case):
    kind = case["kind"]
    if kind == "forward":
        m, past = case["tokens"], case["past"]
        layer = QKV * H + H * H + 3 * I * H
        pairs = m * past + m * (m + 1) // 2
        return {"bytes": LAYERS * (layer + 8 * (QKV + H + 3 * I) + KV * D * 8 * (past + 2 * m)) + 4 * V * (H + 1)
                + 4 * H * m,
                "flops": 2 * LAYERS * (m * layer + 2 * HEADS * D * pairs) + 2 * V * H}
    if kind == "norm":
        m, k = case["rows"], case["k"]
        return {"bytes": 5 * m * k + 4 * m + 4 * k, "flops": 6 * m * k}
    if kind == "swiglu":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": m * k + 4 * m + 2 * n * (k + 4) + 4 * m * n, "flops": 4 * m * n * k}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        each = {"token": 1, "int8": 4, "vnni": 4, "f32": 4}[case["mode"]]
        weight = n * k * 4 if case["mode"] == "f32" else n * (k + 4)
        return {"bytes": each * m * k + weight + 4 * n * (n != V) + 4 * m * n * (2 if case["residual"] else 1),
                "flops": 2 * m * n * k}
    heads, kv, dim, past = case["heads"], case["kv"], case["dim"], case["past"]
    rows = case.get("rows", 1)
    pairs = rows * past + rows * (rows + 1) // 2
    return {"bytes": 8 * rows * heads * dim + 8 * kv * (past + rows) * dim
            + (5 * rows * heads * dim - 4 * rows * heads * dim if kind == "attention" else 0),
            "flops": 4 * heads * dim * pairs}


def tolerance(case):
    # About four times what each path shows against float64; whole numbers (the int8 of a row) may
    # differ where a rounding falls the other way on a last-bit difference.
    kind = case["kind"]
    if kind == "forward":
        # int8 activations are rounded at every projection of 24 layers: a last-bit difference moves
        # some of those roundings, and a prompt's logits were 4% from the float64 model's
        return {"rel": 3e-2, "max": 0.3}
    if kind in ("attention", "decode_attention", "reference_attention"):
        return {"rel": 2e-6, "max": 5e-5, "differ": 1e-3}
    if kind == "norm":
        return {"rel": 3e-7, "max": 3e-6, "differ": 1e-3}
    if kind == "swiglu" or case["mode"] == "token":
        return {"rel": 4e-7, "max": 4e-6}      # exact whole-number sums, then a few rounded products
    if case["mode"] == "vnni":
        return {"rel": 1e-5, "max": 1e-2}      # its own rounding of an activation may move by one step
    return {"rel": 2e-6, "max": 5e-5}


def _dot(a, b):
    return a.double() @ b.double().T


def _linear_exact(case, x):
    mode = case["mode"]
    if mode == "f32":
        y = _dot(x["x"], x["w"])
    elif mode == "token":
        y = _dot(x["xq"], x["q"]) * x["xs"].double()[:, None] * x["scales"].double()
    else:
        a = x["x"].double()
        if mode == "vnni":                             # each block of 32 to int8, ties away from zero
            b = x["x"].view(a.shape[0], -1, BLOCK)
            s = b.abs().amax(2, keepdim=True) / 127
            s = torch.where(s <= 0, torch.ones_like(s), s)
            r = b / s
            r = torch.where(r < 0, -torch.floor(r.abs().double() + 0.5), torch.floor(r.double() + 0.5))
            a = (r.clamp(-127, 127) * s.double()).view(a.shape)
        y = a @ x["q"].double().T * x["scales"].double()
    if x["bias"] is not None:
        y = y + x["bias"].double()
    return y if x["residual"] is None else x["residual"].double() + y


def _attend(q, keys, values, past):
    """softmax(q k^T / sqrt(d), causal) v: q [rows, heads, d], keys and values [kv, past + rows, d]."""
    rows, heads, dim = q.shape
    kv, total = keys.shape[0], past + rows
    hidden = torch.arange(total, device=q.device)[None, :] > past + torch.arange(rows, device=q.device)[:, None]
    out = []
    for h in range(heads):
        g = h // (heads // kv)
        s = (q[:, h] @ keys[g, :total].T.contiguous()) * dim ** -0.5
        out.append(torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ values[g, :total])
    return torch.stack(out, 1).reshape(rows, heads * dim)


def _rotate(x, angles):
    half = x.shape[-1] // 2
    c, s = torch.cos(angles), torch.sin(angles)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _angles(positions, dim):
    inv = torch.from_numpy(inverse_frequencies(dim, 1e6)).cuda()
    return (positions.float()[:, None] * inv).double()           # float32 angles, as the model has them


def _quantized(x):
    s = x.abs().amax(1, keepdim=True) / 127
    s = torch.where(s <= 0, torch.ones_like(s), s)
    r = x / s
    return torch.where(r < 0, -torch.floor(r.abs() + 0.5), torch.floor(r + 0.5)).clamp(-127, 127) * s


def _forward_exact(case, seed):
    model, weights, ids, keys, values = _forward_inputs(case, seed)
    del model
    w = lambda name: torch.from_numpy(weights[name]).cuda().double()                     # noqa: E731
    past, m = case["past"], case["tokens"]

    def norm(x, gamma):
        return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * gamma

    def project(xq, name):
        y = xq @ w(f"{name}.weight@int8").T * w(f"{name}.weight@scales")
        return y + w(f"{name}.bias") if f"{name}.bias" in weights else y

    x = w("model.embed_tokens.weight")[torch.from_numpy(ids).cuda()]
    angles = _angles(past + torch.arange(m, device="cuda"), D)[:, None]
    for i in range(LAYERS):
        p = f"model.layers.{i}"
        xq = _quantized(norm(x, w(f"{p}.input_layernorm.weight")))
        q, k, v = (project(xq, f"{p}.self_attn.{n}_proj").view(m, -1, D) for n in "qkv")
        q, k = _rotate(q, angles), _rotate(k, angles)
        past_k, past_v = (torch.from_numpy(t[i]).cuda().double() for t in (keys, values))
        ctx = _attend(q, torch.cat([past_k, k.transpose(0, 1)], 1), torch.cat([past_v, v.transpose(0, 1)], 1), past)
        x = x + project(_quantized(ctx), f"{p}.self_attn.o_proj")
        xq = _quantized(norm(x, w(f"{p}.post_attention_layernorm.weight")))
        h = torch.nn.functional.silu(project(xq, f"{p}.mlp.gate_proj")) * project(xq, f"{p}.mlp.up_proj")
        x = x + project(_quantized(h), f"{p}.mlp.down_proj")
    return norm(x[-1:], w("model.norm.weight")) @ w("model.embed_tokens.weight").T


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        return _forward_exact(case, seed)
    x = _operands(case, seed)
    if kind == "linear":
        return [_linear_exact(case, x)]
    if kind == "swiglu":
        xs = x["xs"].double()[:, None]
        g = _dot(x["xq"], x["qg"]) * xs * x["sg"].double()
        return [torch.nn.functional.silu(g) * (_dot(x["xq"], x["qu"]) * xs * x["su"].double())]
    if kind == "norm":
        a = x["x"].double()
        n = a * torch.rsqrt((a * a).mean(1, keepdim=True) + EPS) * x["gamma"].double()
        return [None, n.abs().amax(1) / 127]
    heads, kv, dim, past = case["heads"], case["kv"], case["dim"], case["past"]
    rows = case.get("rows", 1)
    split = x["qkv"].double().view(rows, heads + 2 * kv, dim)
    q, keys, values = split[:, :heads], x["keys"].double(), x["values"].double()
    if kind == "decode_attention":
        angles = _angles(torch.tensor([past], device="cuda"), dim)[:, None]
        q, new_k = _rotate(q, angles), _rotate(split[:, heads:heads + kv], angles)
        keys[:, past], values[:, past] = new_k[0], split[0, heads + kv:]
        return [_attend(q, keys, values, past), keys[:, past], values[:, past]]
    ctx = _attend(q, keys, values, past)
    return [ctx] if kind == "reference_attention" else [ctx, None, ctx.abs().amax(1) / 127]
