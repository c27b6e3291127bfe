"""The work whose speed this repository is judged by: single calls of the
quantized matmul (decode and prefill, device and host entries), the other
backend operations, and one generation loop of a whole decoder.

``listed()`` names fixed cases; ``draw(rng)`` gives another case of the same
families with sizes spread over their ranges.  A case is a dict of plain
values; ``prepare`` builds what a program holds before the call (inputs made
from the seed, weights uploaded and repacked), ``run`` is one pass through the
public entry points, ``exact`` the same result from plain torch in float64,
``work`` the bytes and operations one pass cannot do without.
"""
import math

import numpy as np
import torch

import tinybrain_amd as tb

INT4_GROUP = 32       # elements per scale, along K (converter) or N (runtime)
W_STD = 0.02          # standard deviation of the weights before quantization

_backend = None


def backend():
    """The one HIPBackend of the process, as a program keeps it."""
    global _backend
    if _backend is None:
        _backend = tb.HIPBackend(0)
    return _backend


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _matmul(weight, m, n, k, x="f32", entry="device"):
    return {"op": "matmul", "weight": weight, "x": x, "entry": entry, "m": m, "n": n, "k": k}


def _attention(batch, seq, kv, heads, kv_heads, head_dim, mask=False):
    return {"op": "attention", "batch": batch, "seq": seq, "kv": kv, "heads": heads, "kv_heads": kv_heads,
            "head_dim": head_dim, "mask": mask}


def _rows(op, rows, cols):
    return {"op": op, "rows": rows, "cols": cols}


def _decode(weight, layers, hidden, heads, kv_heads, ffn, vocab, context, tokens):
    return {"op": "decode", "weight": weight, "layers": layers, "hidden": hidden, "heads": heads,
            "kv_heads": kv_heads, "ffn": ffn, "vocab": vocab, "context": context, "tokens": tokens}


def listed():
    return [
        # the smallest call of a decode step: the 1.1B attention output
        # projection of one token, converter INT4
        dict(_matmul("int4", 1, 2048, 2048), name="decode_o_int4_m1"),
        # one token's FFN projection as the host runtime calls it: numpy x in,
        # numpy y out, synchronous, per-channel INT8
        dict(_matmul("int8", 1, 5632, 2048, entry="host"), name="host_ffn_int8_m1"),
        # one token through weights the runtime quantized itself (groups along
        # N), the 1.1B FFN down projection
        dict(_matmul("int4rt", 1, 2048, 5632), name="decode_down_int4rt_m1"),
        # the LM head for a batch of eight sequences
        dict(_matmul("int4", 8, 32000, 2048), name="lm_head_int4_m8"),
        # a long prompt's FFN projection, bf16 activations, INT8 weights
        dict(_matmul("int8", 2048, 5632, 2048, x="bf16"), name="prefill_bf16_int8_m2048"),
        # a medium prompt's FFN down projection, bf16 activations, INT4 weights
        dict(_matmul("int4", 512, 2048, 5632, x="bf16"), name="prefill_bf16_int4_m512"),
        # a 7B-shaped FFN projection of a 1000-token prompt in the runtime's own
        # element type (fp32): the largest call
        dict(_matmul("int4", 1000, 11008, 4096), name="prefill_f32_int4_m1000"),
        # a short prompt of odd length, fp32, weights the runtime quantized
        dict(_matmul("int4rt", 333, 2048, 5632), name="prefill_f32_int4rt_m333"),
        # attention of a 512-token prompt, 32 query and 4 key/value heads
        dict(_attention(1, 512, 512, 32, 4, 64), name="attention_prefill_512"),
        # attention of one new token over a long cache
        dict(_attention(1, 1, 4096, 32, 4, 64), name="attention_decode_4096"),
        # softmax over the logits of 256 tokens
        dict(_rows("softmax", 256, 32000), name="softmax_logits_256"),
        # generation: four tokens of a 1.1B-shaped INT8 decoder at context 512,
        # logits to the host after each, as a sampling loop needs them
        dict(_decode("int8", 22, 2048, 32, 4, 5632, 32000, 512, 4), name="decode_1p1b_int8"),
    ]


_MAX_FLOPS = 2.0 * 1000 * 11008 * 4096   # no drawn matmul costs more than the largest listed


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    family = rng.choice(("decode", "decode", "host", "prefill_bf16", "prefill_f32", "prefill_f32",
                         "attention_prefill", "attention_decode", "rows", "decoder"))
    if family in ("decode", "host"):
        weight = rng.choice(("int4", "int8", "int4rt", "int8z"))
        step = 32 if weight == "int4rt" else 1
        return _matmul(weight, rng.choice((1, 1, 1, 2, 3, 4, 5, 6, 7, 8)), _log(rng, 512, 32000, step),
                       _log(rng, 512, 11008, 32 if weight == "int4" else 8),
                       entry="host" if family == "host" else "device")
    if family.startswith("prefill"):
        weight = rng.choice(("int4", "int8", "int4rt"))
        m, k = _log(rng, 16, 2048), _log(rng, 512, 11008, 32 if weight == "int4" else 8)
        step = 32 if weight == "int4rt" else 1
        top = max(512, min(32000, int(_MAX_FLOPS / (2.0 * m * k))) // 32 * 32)
        return _matmul(weight, m, _log(rng, 512, top, step), k, x="bf16" if family == "prefill_bf16" else "f32")
    heads, kv_heads, head_dim = rng.choice(((32, 4, 64), (32, 32, 128), (32, 8, 128), (12, 12, 64), (8, 2, 32)))
    if family == "attention_prefill":
        seq = _log(rng, 16, 1024)
        return _attention(rng.choice((1, 1, 2)), seq, seq + rng.choice((0, 0, _log(rng, 16, 1024))), heads,
                          kv_heads, head_dim, rng.random() < 0.25)
    if family == "attention_decode":
        return _attention(rng.choice((1, 1, 4, 8)), 1, _log(rng, 64, 8192), heads, kv_heads, head_dim,
                          rng.random() < 0.25)
    if family == "rows":
        op = rng.choice(("softmax", "rmsnorm", "silu", "gelu"))
        return _rows(op, _log(rng, 1, 2048), _log(rng, 512, 8192))
    hidden, heads, kv_heads, ffn = rng.choice(((2048, 32, 4, 5632), (4096, 32, 32, 11008), (1024, 16, 4, 2816)))
    return _decode(rng.choice(("int8", "int4", "int4rt")), rng.choice((2, 3, 4, 6)), hidden, heads, kv_heads, ffn,
                   rng.choice((8192, 16000, 32000)), _log(rng, 16, 512), rng.choice((1, 2, 4, 8)))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _host(t):
    return t.contiguous().cpu().numpy()


def _pack_int4(q):
    """Signed values -7..7 two per byte, even index in the high nibble."""
    q = q.reshape(-1)
    if q.numel() % 2:
        q = torch.cat([q, q.new_zeros(1)])
    u = q.to(torch.int16) & 0xF
    b = (u[0::2] << 4) | u[1::2]
    return torch.where(b > 127, b - 256, b).to(torch.int8)


def _quantized(gen, kind, n, k, std=W_STD):
    """A random weight as the runtime or the converter quantizes it, and its
    dequantized [K, N] fp32 matrix (on the GPU)."""
    if kind in ("int8", "int8z"):
        w = _normal(gen, k, n, std=std)
        if kind == "int8":                        # symmetric, one scale per output channel
            s = w.abs().amax(0) / 127.0
            q = (w / s).round().clamp(-127, 127)
            qt = tb.QuantizedTensor((k, n), _host(q.to(torch.int8)).reshape(-1), _host(s),
                                    tb.QuantizationMode.perChannel)
            return qt, q * s
        w = w + 0.25 * std                        # asymmetric: one scale and zero point
        s = (w.max() - w.min()) / 255.0
        z = (-w.min() / s - 128.0).round().clamp(-128, 127)
        q = ((w / s).round() + z).clamp(-128, 127)
        qt = tb.QuantizedTensor((k, n), _host(q.to(torch.int8)).reshape(-1), _host(s.reshape(1)),
                                tb.QuantizationMode.asymmetric, zeroPoints=_host(z.to(torch.int8).reshape(1)))
        return qt, (q - z) * s
    rows, cols = (n, k) if kind == "int4" else (k, n)      # groups run along the last axis
    w = _normal(gen, rows, cols, std=std).reshape(-1, INT4_GROUP)
    s = w.abs().amax(1) / 7.0
    q = (w / s[:, None]).round().clamp(-7, 7)
    layout = tb.Layout.NK_FLAT if kind == "int4" else tb.Layout.KN_FLAT
    qt = tb.QuantizedTensor((k, n), _host(_pack_int4(q)), _host(s), tb.QuantizationMode.int4,
                            tb.QuantizationPrecision.int4, INT4_GROUP,
                            np.zeros(s.numel(), np.int8), layout)
    d = (q * s[:, None]).reshape(rows, cols)
    return qt, d.t() if kind == "int4" else d


def _matmul_inputs(case, seed):
    gen = _generator(seed)
    x = _normal(gen, case["m"], case["k"])
    if case["x"] == "bf16":
        x = x.to(torch.bfloat16)
    qt, w = _quantized(gen, case["weight"], case["n"], case["k"])
    return x, qt, w


def _attention_inputs(case, seed):
    gen = _generator(seed)
    b, nh, nkv, hd = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    q = _normal(gen, b, case["seq"], nh * hd)
    k = _normal(gen, b, case["kv"], nkv * hd)
    v = _normal(gen, b, case["kv"], nkv * hd)
    mask = None
    if case["mask"]:                              # additive, some positions ignored
        gone = torch.rand(case["kv"], generator=gen, device="cuda") < 0.2
        gone[0] = False
        mask = torch.where(gone, -math.inf, 0.0).to(torch.float32)
    return q, k, v, mask


def _rows_inputs(case, seed):
    gen = _generator(seed)
    x = _normal(gen, case["rows"], case["cols"], std=3.0 if case["op"] == "softmax" else 1.0)
    g = torch.rand(case["cols"], generator=gen, device="cuda") + 0.5
    return x, g


def _decoder_inputs(case, seed):
    """Embeddings, norms, per layer (norms, projections) and the LM head, each
    projection as (QuantizedTensor, dequantized); then the prompt and the
    tokens of the pass.  Layers come one at a time."""
    gen = _generator(seed)
    h, ffn, v = case["hidden"], case["ffn"], case["vocab"]
    kvd = h // case["heads"] * case["kv_heads"]
    tokens = torch.randint(0, v, (case["context"] + case["tokens"],), generator=gen, device="cuda").tolist()
    emb = _normal(gen, v, h)
    norm = torch.rand(2 * case["layers"] + 1, h, generator=gen, device="cuda") + 0.5
    shapes = ((h, h), (kvd, h), (kvd, h), (h, h), (ffn, h), (ffn, h), (h, ffn))   # q k v o gate up down as (N, K)

    def layers():
        for i in range(case["layers"]):
            yield norm[2 * i], norm[2 * i + 1], [_quantized(gen, case["weight"], n, k) for n, k in shapes]

    head = _quantized(gen, case["weight"], v, h)
    return tokens, emb, norm[-1], head, layers()


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    be, op = backend(), case["op"]
    if op == "matmul":
        x, qt, _ = _matmul_inputs(case, seed)
        if case["entry"] == "host":
            be.weight(qt)                         # uploaded once, as at model load
            return {"op": "host", "x": _host(x), "w": qt, "evict": _Evict(qt)}
        return {"op": "matmul_" + case["x"], "x": x, "w": tb.DeviceWeight(be, qt)}
    if op == "attention":
        q, k, v, mask = _attention_inputs(case, seed)
        return {"op": op, "args": (q, k, v, mask, case["head_dim"], case["heads"], case["kv_heads"])}
    if op == "decode":
        tokens, emb, norm, head, layers = _decoder_inputs(case, seed)
        cfg = tb.DecoderConfig(case["layers"], case["hidden"], case["heads"], case["kv_heads"], case["ffn"],
                               case["vocab"], max_seq=case["context"] + 64)
        d = tb.Decoder(be, cfg, _host(emb), _host(norm), head[0])
        for i, (g_in, g_post, projections) in enumerate(layers):
            d.set_layer(i, _host(g_in), _host(g_post), [p[0] for p in projections])
        for t in tokens[:case["context"]]:        # the prompt fills the cache
            d.step_device(t)
        torch.cuda.synchronize()
        return {"op": op, "decoder": d, "context": case["context"], "tokens": tokens[case["context"]:]}
    x, g = _rows_inputs(case, seed)
    return {"op": op, "x": x, "g": g}


class _Evict:
    """Drops a host-entry weight from the backend with the state that holds it."""

    def __init__(self, qt):
        self.qt = qt

    def __del__(self):
        backend().evict(self.qt)


def run(state):
    be, op = backend(), state["op"]
    if op == "matmul_f32":
        return be.matmul_device(state["x"], state["w"])
    if op == "matmul_bf16":
        return be.matmul_bf16_device(state["x"], state["w"])
    if op == "host":
        return be.matmulQuantized(state["x"], state["w"])
    if op == "attention":
        return be.attention_device(*state["args"])
    if op == "softmax":
        return be.softmax_device(state["x"])
    if op == "rmsnorm":
        return be.rmsnorm_device(state["x"], state["g"])
    if op == "silu":
        return be.silu_device(state["x"])
    if op == "gelu":
        return be.gelu_device(state["x"])
    d = state["decoder"]
    d.set_position(state["context"])
    return [d.step(t) for t in state["tokens"]]


# ---------------------------------------------------------------------------
# floors, tolerances, the same in 64 bits
# ---------------------------------------------------------------------------
def _weight_bytes(kind, n, k):
    if kind == "int8":
        return n * k + 4 * n
    if kind == "int8z":
        return n * k + 5
    return n * k // 2 + 4 * (n * k // INT4_GROUP)


def work(case):
    op = case["op"]
    if op == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        x_bytes = 2 if case["x"] == "bf16" else 4
        return {"bytes": _weight_bytes(case["weight"], n, k) + x_bytes * m * k + 4 * m * n, "flops": 2 * m * n * k}
    if op == "attention":
        b, s, t, hd = case["batch"], case["seq"], case["kv"], case["head_dim"]
        return {"bytes": 4 * b * hd * (2 * s * case["heads"] + 2 * t * case["kv_heads"]),
                "flops": 4 * b * s * t * case["heads"] * hd}
    if op == "decode":
        h, ffn, v = case["hidden"], case["ffn"], case["vocab"]
        kvd = h // case["heads"] * case["kv_heads"]
        shapes = ((h, h), (kvd, h), (kvd, h), (h, h), (ffn, h), (ffn, h), (h, ffn))
        weights = case["layers"] * sum(_weight_bytes(case["weight"], n, k) for n, k in shapes)
        weights += _weight_bytes(case["weight"], v, h)
        params = case["layers"] * sum(n * k for n, k in shapes) + v * h
        cache = case["layers"] * 8 * kvd * (case["context"] + case["tokens"] / 2)
        scores = case["layers"] * 4 * h * (case["context"] + case["tokens"] / 2)
        return {"bytes": case["tokens"] * (weights + cache + 4 * v), "flops": case["tokens"] * (2 * params + scores)}
    n = case["rows"] * case["cols"]
    return {"bytes": 8 * n + (4 * case["cols"] if op == "rmsnorm" else 0), "flops": 4 * n}


def tolerance(case):
    # fp32 sums of exact products in another order, or activations held as two
    # 16-bit pieces (22 bits): 1e-7 to 7e-7 was seen between the row counts'
    # different kernels on the same inputs.  "max" is against the result's
    # root mean square, where a sum of cancelling terms shows its full error.
    if case["op"] == "decode":
        # the layers carry each rounding on
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 3e-6, "max": 3e-5}


def exact(case, seed):
    op = case["op"]
    if op == "matmul":
        x, _, w = _matmul_inputs(case, seed)
        y = x.double() @ w.double()
        return y.cpu().numpy() if case["entry"] == "host" else y
    if op == "attention":
        q, k, v, mask = _attention_inputs(case, seed)
        b, nh, nkv, hd = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
        out = torch.empty(b, case["seq"], nh, hd, dtype=torch.float64, device="cuda")
        q, k, v = (t.double().reshape(b, -1, n, hd) for t, n in ((q, nh), (k, nkv), (v, nkv)))
        for i in range(b):
            for j in range(nh):
                c = j // (nh // nkv)
                s = q[i, :, j] @ k[i, :, c].t().contiguous() / math.sqrt(hd)
                if mask is not None:
                    s = s + mask.double()
                out[i, :, j] = torch.softmax(s, -1) @ v[i, :, c].contiguous()
        return out.reshape(b, case["seq"], nh * hd)
    if op == "decode":
        return _exact_decode(case, seed)
    x, g = _rows_inputs(case, seed)
    x = x.double()
    if op == "softmax":
        e = torch.exp(x - x.amax(-1, keepdim=True))
        return e / (e.sum(-1, keepdim=True) + 1e-7)
    if op == "rmsnorm":
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g.double()
    if op == "silu":
        return x / (1.0 + torch.exp(-x))
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_decode(case, seed):
    """The pass's logits from one causal forward over prompt and tokens."""
    tokens, emb, final, head, layers = _decoder_inputs(case, seed)
    nh, nkv, hd = case["heads"], case["kv_heads"], case["hidden"] // case["heads"]
    t = len(tokens)
    i = torch.arange(0, hd, 2, dtype=torch.float32, device="cuda")
    # the angle is formed in fp32, as the runtime defines it
    angle = (torch.arange(t, dtype=torch.float32, device="cuda")[:, None]
             * torch.pow(torch.tensor(10000.0, device="cuda"), -(i / hd))[None]).double()
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(a, heads):
        a = a.reshape(t, heads, hd // 2, 2)
        return torch.stack([a[..., 0] * cos - a[..., 1] * sin, a[..., 0] * sin + a[..., 1] * cos], -1).reshape(t, heads, hd)

    def rms(a, g):
        return a / torch.sqrt((a * a).mean(-1, keepdim=True) + 1e-5) * g.double()

    causal = torch.full((t, t), -math.inf, dtype=torch.float64, device="cuda").triu(1)
    h = emb[torch.tensor(tokens, device="cuda")].double()
    for g_in, g_post, projections in layers:
        wq, wk, wv, wo, wg, wu, wd = (p[1].double() for p in projections)
        x = rms(h, g_in)
        q, k, v = rope(x @ wq, nh), rope(x @ wk, nkv), (x @ wv).reshape(t, nkv, hd)
        ctx = torch.empty(t, nh, hd, dtype=torch.float64, device="cuda")
        for j in range(nh):
            c = j // (nh // nkv)
            s = q[:, j] @ k[:, c].t().contiguous() / math.sqrt(hd) + causal
            ctx[:, j] = torch.softmax(s, -1) @ v[:, c].contiguous()
        h = h + ctx.reshape(t, nh * hd) @ wo
        x = rms(h, g_post)
        g = x @ wg
        h = h + (g / (1.0 + torch.exp(-g)) * (x @ wu)) @ wd
    y = rms(h[case["context"]:], final) @ head[1].double()
    return list(y.cpu().numpy())
