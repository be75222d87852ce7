"""The work this backend is measured on: the products, blocks and whole decode
steps that a program which serves a quantized Qwen3-style model has it do.

A case is a dict of plain values with a "kind":

  linear     one QuantMatmul: the call every other path is made of
  mlp        MLP.Forward on a batch of rows: gate, up, SiLU * up, down
  attention  Attention.ForwardCached on a piece of a prompt: q/k/v products, q/k
             norms, RoPE, the KV append, causal SDPA over the cache, o product
  moe        an expert block: the router's top-k and the routed expert MLPs
  decode     one token through all layers to its logits, fused or as the
             reference's own call sequence

Inputs are drawn on the GPU from the seed alone: uniform codes, scales
|N(0,1)| * 0.02 with the bias that centres them, activations N(0,1).
"""
import math

import torch

from janis_amd import qwen3_decode as q3
from janis_amd.engine import BF16, F16, F32, I32, U32, U8, HipBackend

HEAD_DIM = 128
EPS = 1e-6
THETA = 1e6
CODE = {torch.float32: F32, torch.float16: F16, torch.bfloat16: BF16, torch.int32: I32, torch.uint8: U8}
TORCH = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16, I32: torch.int32}


# ---- the cases -------------------------------------------------------------------

def listed():
    return [
        # the smallest call of a decode loop: the key projection of one token
        {"name": "linear_kv_1", "kind": "linear", "rows": 1, "n": 1024, "k": 4096, "group": 64, "bits": 4, "f32": False},
        # one token of an 8-billion-parameter model at a chat-length context
        {"name": "decode_512", "kind": "decode", "layers": 36, "hidden": 4096, "inter": 12288, "heads": 32, "kv": 8,
         "vocab": 151936, "ctx": 512, "fused": True, "f16": False},
        # a few of its layers and the head at a document-length context
        {"name": "decode_8k", "kind": "decode", "layers": 4, "hidden": 4096, "inter": 12288, "heads": 32, "kv": 8,
         "vocab": 151936, "ctx": 8191, "fused": True, "f16": True},
        # the same layers as a program makes them that knows only engine.Backend: F32 activations, f16 caches
        {"name": "decode_calls_1000", "kind": "decode", "layers": 4, "hidden": 4096, "inter": 12288, "heads": 32, "kv": 8,
         "vocab": 151936, "ctx": 1000, "fused": False, "f16": True},
        # expert blocks of a 30-billion-parameter model: one token, a batch of sequences, a prompt
        {"name": "moe_1", "kind": "moe", "tokens": 1, "experts": 128, "top": 8, "hidden": 2048, "inter": 768, "layers": 4},
        {"name": "moe_16", "kind": "moe", "tokens": 16, "experts": 128, "top": 8, "hidden": 2048, "inter": 768, "layers": 2},
        {"name": "moe_500", "kind": "moe", "tokens": 500, "experts": 128, "top": 8, "hidden": 2048, "inter": 768, "layers": 1},
        # an MLP for a few sequences decoded together, a short odd prompt in F32, and a long prompt
        {"name": "mlp_8", "kind": "mlp", "rows": 8, "hidden": 4096, "inter": 12288, "group": 64, "f32": False},
        {"name": "mlp_200", "kind": "mlp", "rows": 200, "hidden": 4096, "inter": 12288, "group": 64, "f32": True},
        {"name": "mlp_2048", "kind": "mlp", "rows": 2048, "hidden": 4096, "inter": 12288, "group": 64, "f32": False},
        # attention of a prompt from an empty cache (F32 activations, f16 caches), and of the next piece of a long one
        {"name": "attention_512", "kind": "attention", "tokens": 512, "past": 0, "hidden": 4096, "heads": 32, "kv": 8,
         "f32": True},
        {"name": "attention_1500_2500", "kind": "attention", "tokens": 1500, "past": 2500, "hidden": 4096, "heads": 32,
         "kv": 8, "f32": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "mlp", "mlp", "attention", "attention", "moe", "moe", "decode"))
    f32 = rng.random() < 0.4
    if kind == "linear":
        rows = 1 if rng.random() < 0.4 else _log_int(rng, 2, 64)
        group = rng.choice((64, 64, 32, 128))
        return {"kind": kind, "rows": rows, "n": _log_int(rng, 512, 24576), "k": rng.choice((1024, 2048, 2560, 4096, 6144, 12288)),
                "group": group, "bits": 8 if rows == 1 and rng.random() < 0.25 else 4, "f32": f32}
    if kind == "mlp":
        hidden, inter = rng.choice(((4096, 12288), (4096, 12288), (2048, 6144), (1024, 3072)))
        return {"kind": kind, "rows": _log_int(rng, 2, 2048), "hidden": hidden, "inter": inter,
                "group": rng.choice((64, 64, 64, 32, 128)), "f32": f32}
    if kind == "attention":
        tokens = _log_int(rng, 16, 1500)
        past = 0 if rng.random() < 0.4 else _log_int(rng, 16, 4096)
        past = min(past, max(0, 1500 * 3250 // tokens - tokens // 2))
        heads, kv = rng.choice(((32, 8), (32, 8), (16, 8), (32, 4)))
        return {"kind": kind, "tokens": tokens, "past": past, "hidden": heads * HEAD_DIM, "heads": heads, "kv": kv, "f32": f32}
    if kind == "moe":
        hidden, inter = rng.choice(((2048, 768), (2048, 768), (1024, 512), (2048, 1024)))
        return {"kind": kind, "tokens": _log_int(rng, 1, 500), "experts": rng.choice((128, 128, 64)), "top": rng.choice((8, 8, 4)),
                "hidden": hidden, "inter": inter, "layers": 1}
    fused = rng.random() < 0.6
    hidden, inter, heads = rng.choice(((4096, 12288, 32), (4096, 12288, 32), (2048, 6144, 16)))
    return {"kind": kind, "layers": rng.randint(1, 4), "hidden": hidden, "inter": inter, "heads": heads, "kv": 8,
            "vocab": 151936, "ctx": _log_int(rng, 32, 16000), "fused": fused, "f16": not fused or rng.random() < 0.5}


# ---- inputs ----------------------------------------------------------------------

def _quant(gen, n, k, group=64, bits=4, lead=()):
    """A quantized matrix (w, scales, biases) in MLX's layout."""
    dev = gen.device
    w = torch.randint(-2**31, 2**31 - 1, (*lead, n, k * bits // 32), dtype=torch.int32, device=dev, generator=gen)
    s = torch.randn((*lead, n, k // group), device=dev, generator=gen).abs_().mul_(0.02 * 2.0 ** (4 - bits)).to(torch.bfloat16)
    b = s.float() * -float(1 << (bits - 1)) + 1e-3 * torch.randn(s.shape, device=dev, generator=gen)
    return w, s, b.to(torch.bfloat16)


def _normal(gen, shape, dtype, scale=1.0, mean=0.0):
    return (torch.randn(shape, device=gen.device, generator=gen) * scale + mean).to(dtype)


def _capacity(tokens):
    return (tokens + HipBackend.KV_STEP - 1) // HipBackend.KV_STEP * HipBackend.KV_STEP


def _inputs(c, seed):
    """Everything a pass reads, as torch tensors on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    act = torch.float32 if c.get("f32") else torch.bfloat16
    if c["kind"] == "linear":
        return {"x": _normal(gen, (c["rows"], c["k"]), act), "w": _quant(gen, c["n"], c["k"], c["group"], c["bits"])}
    if c["kind"] == "mlp":
        H, I, g = c["hidden"], c["inter"], c["group"]
        return {"x": _normal(gen, (c["rows"], H), act), "gate": _quant(gen, I, H, g), "up": _quant(gen, I, H, g),
                "down": _quant(gen, H, I, g)}
    if c["kind"] == "attention":
        H, Hq, Hk, T, D = c["hidden"], c["heads"], c["kv"], c["tokens"], HEAD_DIM
        cache = torch.float16 if c["f32"] else torch.bfloat16
        cap = _capacity(c["past"] + T)
        d = {"x": _normal(gen, (1, T, H), act), "q": _quant(gen, Hq * D, H), "k": _quant(gen, Hk * D, H),
             "v": _quant(gen, Hk * D, H), "o": _quant(gen, H, Hq * D), "q_norm": _normal(gen, (D,), torch.bfloat16, 0.1, 1.5),
             "k_norm": _normal(gen, (D,), torch.bfloat16, 0.1, 1.5)}
        for name in ("k_cache", "v_cache"):
            d[name] = torch.zeros((1, Hk, cap, D), dtype=cache, device=gen.device)
            d[name][:, :, :c["past"]] = _normal(gen, (1, Hk, c["past"], D), cache, 1.5)
        return d
    if c["kind"] == "moe":
        E, H, I = c["experts"], c["hidden"], c["inter"]
        return {"x": _normal(gen, (c["tokens"], H), torch.bfloat16),
                "layers": [{"logits": _normal(gen, (c["tokens"], E), torch.float32), "gate": _quant(gen, I, H, lead=(E,)),
                            "up": _quant(gen, I, H, lead=(E,)), "down": _quant(gen, H, I, lead=(E,))}
                           for _ in range(c["layers"])]}
    H, I, Hq, Hk, D = c["hidden"], c["inter"], c["heads"], c["kv"], HEAD_DIM
    cache = torch.float16 if c["f16"] else torch.bfloat16
    cap = _capacity(c["ctx"] + 1)
    d = {"token": torch.randint(0, c["vocab"], (1,), dtype=torch.int32, device=gen.device, generator=gen),
         "embed": _quant(gen, c["vocab"], H), "head": _quant(gen, c["vocab"], H),
         "norm": _normal(gen, (H,), torch.bfloat16, 0.05, 1.0), "layers": []}
    for _ in range(c["layers"]):
        L = {"qkv": _quant(gen, (Hq + 2 * Hk) * D, H), "o": _quant(gen, H, Hq * D), "gate_up": _quant(gen, 2 * I, H),
             "down": _quant(gen, H, I)}
        for name, n in (("in_norm", H), ("post_norm", H), ("q_norm", D), ("k_norm", D)):
            L[name] = _normal(gen, (n,), torch.bfloat16, 0.05, 1.0)
        for name in ("k_cache", "v_cache"):
            L[name] = torch.zeros((1, Hk, cap, D), dtype=cache, device=gen.device)
            L[name][:, :, :c["ctx"]] = _normal(gen, (1, Hk, c["ctx"], D), cache)
        d["layers"].append(L)
    return d


# ---- a pass ----------------------------------------------------------------------

_engine = []


def _backend():
    """The program's one backend and the stream it works on."""
    if not _engine:
        b, s = HipBackend(0), torch.cuda.Stream()
        b.SetStream(s.cuda_stream)
        _engine.extend((b, s))
    return _engine


def _wrap(b, t, code=None):
    if isinstance(t, tuple):
        w, s, bias = t
        return _wrap(b, w, U32), _wrap(b, s), _wrap(b, bias)
    return b.Wrap(t.data_ptr(), tuple(t.shape), CODE[t.dtype] if code is None else code, keep=t)


def _in_arena(arena, t):
    """The torch view of an engine tensor whose memory lies in `arena`."""
    off = t.ptr - arena.data_ptr()
    return arena[off:off + t.nbytes].view(TORCH[t.dtype]).view(t.shape)


def _arena_bytes(c):
    if c["kind"] == "linear":
        return c["rows"] * c["n"] * 4 + 4096
    if c["kind"] == "mlp":
        return c["rows"] * (4 * c["inter"] + 2 * c["hidden"]) * 4 + 4096
    if c["kind"] == "attention":
        return c["tokens"] * (8 * c["heads"] + 12 * c["kv"]) * HEAD_DIM * 4 + c["tokens"] * c["hidden"] * 4 + 65536
    if c["kind"] == "moe":
        return c["layers"] * (c["tokens"] * (c["hidden"] * 4 + c["top"] * 8) + 4096)
    return 8 * c["vocab"] * 4 + c["layers"] * 64 * 4 * (c["inter"] + c["hidden"]) + (1 << 20)


def _linear(c, b, s):
    return {"y": b.QuantMatmul(s["x"], *s["w"], True, c["group"], c["bits"])}


def _mlp(c, b, s):
    g = c["group"]
    gate, up = b.QuantMatmul(s["x"], *s["gate"], True, g, 4), b.QuantMatmul(s["x"], *s["up"], True, g, 4)
    return {"y": b.QuantMatmul(b.SiLUMul(gate, up), *s["down"], True, g, 4)}


def _attention(c, b, s):
    T, Hq, Hk, D, past = c["tokens"], c["heads"], c["kv"], HEAD_DIM, c["past"]
    x = s["x"]
    q = b.Reshape(b.QuantMatmul(x, *s["q"], True, 64, 4), 1, T, Hq, D)
    k = b.Reshape(b.QuantMatmul(x, *s["k"], True, 64, 4), 1, T, Hk, D)
    v = b.Reshape(b.QuantMatmul(x, *s["v"], True, 64, 4), 1, T, Hk, D)
    q, k = b.RMSNorm(q, s["q_norm"], EPS), b.RMSNorm(k, s["k_norm"], EPS)
    q = b.RoPE(b.Transpose(q, 0, 2, 1, 3), D, False, THETA, 1.0, past)
    k = b.RoPE(b.Transpose(k, 0, 2, 1, 3), D, False, THETA, 1.0, past)
    keys, values = q3.kv_cache_update(b, s["layer"], past, k, b.Transpose(v, 0, 2, 1, 3))
    att = b.SDPA(q, keys, values, D ** -0.5, T > 1)
    att = b.Reshape(b.Transpose(att, 0, 2, 1, 3), 1, T, Hq * D)
    return {"y": b.QuantMatmul(att, *s["o"], True, 64, 4)}


def _moe(c, b, s):
    out = {}
    for i, L in enumerate(s["layers"]):
        idx, scores = b.MoeRoute(L["logits"], c["top"], True)
        y = b.MoeSwiGLU(s["x"], L["gate"], L["up"], L["down"], idx, scores, 64, 4)
        out.update({"y%d" % i: y, "experts%d" % i: idx, "scores%d" % i: scores})
    return out


def _decode(c, b, s):
    logits, token = q3.decode_step(b, s["model"], s["token"], c["ctx"], fused=c["fused"])
    return {"logits": logits, "token": token}


PASS = {"linear": _linear, "mlp": _mlp, "attention": _attention, "moe": _moe, "decode": _decode}


def _captured(c):
    """Whether a program replays the pass as a graph: the loops over tokens of a
    fixed batch are captured once, prompts (each of a length of its own) and
    single calls are not."""
    return c["kind"] == "decode" or (c["kind"] == "moe" and c["tokens"] <= 16) or (c["kind"] == "mlp" and c["rows"] <= 16)


def prepare(case, seed):
    b, stream = _backend()
    d = _inputs(case, seed)
    s = {"case": case, "held": d, "arena": torch.empty(_arena_bytes(case), dtype=torch.uint8, device="cuda")}
    if case["kind"] == "moe":
        s["x"] = _wrap(b, d["x"])
        s["layers"] = [{name: _wrap(b, t) for name, t in L.items()} for L in d["layers"]]
    elif case["kind"] == "decode":
        cfg = q3.Qwen3Config(hidden=case["hidden"], inter=case["inter"], n_heads=case["heads"], n_kv=case["kv"],
                             vocab=case["vocab"], layers=case["layers"], eps=EPS, theta=THETA)
        layers = [q3.Qwen3Layer(**{name: _wrap(b, t) for name, t in L.items()}) for L in d["layers"]]
        s["model"] = q3.Qwen3Model(cfg, _wrap(b, d["embed"]), layers, _wrap(b, d["norm"]), _wrap(b, d["head"]))
        s["token"] = _wrap(b, d["token"])
    else:
        s.update({name: _wrap(b, t) for name, t in d.items()})
        if case["kind"] == "attention":
            s["layer"] = q3.Qwen3Layer(qkv=None, o=None, gate_up=None, down=None, in_norm=None, post_norm=None,
                                       q_norm=s["q_norm"], k_norm=s["k_norm"], k_cache=s["k_cache"], v_cache=s["v_cache"])
    s["room"] = _wrap(b, s["arena"])
    s["graph"] = None
    stream.wait_stream(torch.cuda.current_stream())
    if _captured(case):
        with torch.cuda.stream(stream):
            s["out"] = _pass(s)  # sizes the workspace, which a capture may not
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            s["out"] = _pass(s)
        s["graph"] = g
    return s


def _pass(s):
    c, b = s["case"], _engine[0]
    with b.use_arena(s["room"]):
        out = PASS[c["kind"]](c, b, s)
    out = {name: _in_arena(s["arena"], t) for name, t in out.items()}
    # the caches are updated in place
    if c["kind"] == "attention":
        end = c["past"] + c["tokens"]
        out["keys"], out["values"] = (s["held"][n][:, :, c["past"]:end] for n in ("k_cache", "v_cache"))
    if c["kind"] == "decode":
        for i, L in enumerate(s["held"]["layers"][:4]):
            out["key%d" % i], out["value%d" % i] = (L[n][:, :, c["ctx"]] for n in ("k_cache", "v_cache"))
    return out


def run(state):
    if state["graph"] is None:
        return _pass(state)
    with torch.cuda.stream(_engine[1]):
        state["graph"].replay()
    return state["out"]


# ---- what a pass cannot do without -------------------------------------------------

def _matrix_bytes(n, k, group=64, bits=4):
    return n * k * bits / 8 + 4 * n * (k // group)


def work(c):
    ab = 4 if c.get("f32") else 2
    if c["kind"] == "linear":
        return {"bytes": _matrix_bytes(c["n"], c["k"], c["group"], c["bits"]) + ab * c["rows"] * (c["n"] + c["k"]),
                "flops": 2 * c["rows"] * c["n"] * c["k"]}
    if c["kind"] == "mlp":
        H, I = c["hidden"], c["inter"]
        return {"bytes": 2 * _matrix_bytes(I, H, c["group"]) + _matrix_bytes(H, I, c["group"]) + 2 * ab * c["rows"] * H,
                "flops": 6 * c["rows"] * H * I}
    if c["kind"] == "attention":
        H, Q, KV, T, past = c["hidden"], c["heads"] * HEAD_DIM, c["kv"] * HEAD_DIM, c["tokens"], c["past"]
        weights = _matrix_bytes(Q + 2 * KV, H) + _matrix_bytes(H, Q)
        pairs = T * past + T * (T + 1) // 2
        return {"bytes": weights + 2 * ab * T * H + 2 * 2 * KV * (past + T),
                "flops": 2 * T * H * (2 * Q + 2 * KV) + 4 * pairs * Q}
    if c["kind"] == "moe":
        H, I, T, E, K = c["hidden"], c["inter"], c["tokens"], c["experts"], c["top"]
        used = E * (1 - (1 - K / E) ** T)
        one = 2 * _matrix_bytes(I, H) + _matrix_bytes(H, I)
        return {"bytes": c["layers"] * (used * one + T * (6 * H + 4 * E + 8 * K)), "flops": c["layers"] * 6 * T * K * H * I}
    H, I, Q, KV = c["hidden"], c["inter"], c["heads"] * HEAD_DIM, c["kv"] * HEAD_DIM
    shapes = [(Q + 2 * KV, H), (H, Q), (2 * I, H), (H, I)] * c["layers"] + [(c["vocab"], H)]
    return {"bytes": sum(_matrix_bytes(n, k) for n, k in shapes) + c["layers"] * 4 * KV * (c["ctx"] + 1) + 4 * c["vocab"],
            "flops": sum(2 * n * k for n, k in shapes) + c["layers"] * 4 * Q * (c["ctx"] + 1)}


def tolerance(c):
    """About four times the distance to exact() that was measured: bf16 (or
    bf16-rounded) inputs of every product, fp32 sums, and bf16 or f16 results
    where those are written (products 0.0017, an MLP 0.0039, attention 0.0089
    with bf16 caches and 0.0056 with f16, experts 0.0018, a decode step's rows
    0.0023 and logits 0.0004)."""
    if c["kind"] == "linear":
        return {"rel": 8e-3, "max": 0.04}
    if c["kind"] == "mlp":
        return {"rel": 1.6e-2, "max": 0.1}
    if c["kind"] == "attention":
        return {"rel": 3.5e-2, "max": 0.25}
    if c["kind"] == "moe":
        return {"rel": 8e-3, "max": 0.05}
    return {"rel": 1.2e-2, "max": 0.08}


# ---- the same in 64 bits -----------------------------------------------------------

def _dense(m, bits=4):
    """A quantized matrix (w, scales, biases) as [..., n, k] float64."""
    w, s, b = m
    k = w.shape[-1] * 32 // bits
    shifts = torch.arange(0, 32, bits, device=w.device, dtype=torch.int32)
    q = (w.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)
    q = q.reshape(*s.shape, k // s.shape[-1]).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(*w.shape[:-1], k)


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _rope(x, pos):
    """x [..., T, D] rotated at positions pos [T]."""
    half = x.shape[-1] // 2
    inv = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    a = pos.double().unsqueeze(-1) * inv
    p, q = x[..., :half], x[..., half:]
    return torch.cat((p * a.cos() - q * a.sin(), p * a.sin() + q * a.cos()), -1)


def _attend(q, k, v, past):
    """q [Hq, T, D], k/v [Hk, past + T, D]: causal over the cache."""
    G, T, S = q.shape[0] // k.shape[0], q.shape[1], k.shape[1]
    late = torch.arange(S, device=q.device) > past + torch.arange(T, device=q.device).unsqueeze(-1)
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        p = (q[h] @ k[h // G].T * HEAD_DIM ** -0.5).masked_fill_(late, -math.inf).softmax(-1)
        out[h] = p @ v[h // G]
    return out


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    if c["kind"] == "linear":
        return {"y": d["x"].double() @ _dense(d["w"], c["bits"]).T}
    if c["kind"] == "mlp":
        x = d["x"].double()
        return {"y": (_silu(x @ _dense(d["gate"]).T) * (x @ _dense(d["up"]).T)) @ _dense(d["down"]).T}
    if c["kind"] == "attention":
        T, Hq, Hk, D, past = c["tokens"], c["heads"], c["kv"], HEAD_DIM, c["past"]
        x = d["x"][0].double()
        q, k, v = ((x @ _dense(d[n]).T).view(T, h, D) for n, h in (("q", Hq), ("k", Hk), ("v", Hk)))
        pos = past + torch.arange(T, device=x.device)
        q = _rope(_rms(q, d["q_norm"]).transpose(0, 1), pos)
        k = _rope(_rms(k, d["k_norm"]).transpose(0, 1), pos)
        v = v.transpose(0, 1)
        old = [d[n][0, :, :past].double() for n in ("k_cache", "v_cache")]
        att = _attend(q, torch.cat((old[0], k), 1), torch.cat((old[1], v), 1), past)
        return {"y": (att.transpose(0, 1).reshape(T, Hq * D) @ _dense(d["o"]).T).unsqueeze(0), "keys": k.unsqueeze(0),
                "values": v.unsqueeze(0)}
    if c["kind"] == "moe":
        x, out = d["x"].double(), {}
        for i, L in enumerate(d["layers"]):
            p, idx = L["logits"].double().softmax(-1).topk(c["top"], -1)
            p = p / p.sum(-1, keepdim=True)
            y = torch.zeros((c["tokens"], c["hidden"]), dtype=torch.float64, device=x.device)
            for e in idx.unique().tolist():
                t, slot = (idx == e).nonzero(as_tuple=True)
                g, u, dn = (_dense(tuple(m[e] for m in L[n])) for n in ("gate", "up", "down"))
                y.index_add_(0, t, p[t, slot].unsqueeze(-1) * ((_silu(x[t] @ g.T) * (x[t] @ u.T)) @ dn.T))
            out.update({"y%d" % i: y, "experts%d" % i: None, "scores%d" % i: p})
        return out
    H, I, Hq, Hk, D, ctx = c["hidden"], c["inter"], c["heads"], c["kv"], HEAD_DIM, c["ctx"]
    out, token = {"token": None}, int(d["token"])
    h = _dense(tuple(t[token:token + 1] for t in d["embed"]))
    pos = torch.tensor([ctx], device=h.device)
    for i, L in enumerate(d["layers"]):
        qkv = (_rms(h, L["in_norm"]) @ _dense(L["qkv"]).T).view(Hq + 2 * Hk, 1, D)
        q = _rope(_rms(qkv[:Hq], L["q_norm"]), pos)
        k = _rope(_rms(qkv[Hq:Hq + Hk], L["k_norm"]), pos)
        v = qkv[Hq + Hk:]
        keys, values = (torch.cat((L[n][0, :, :ctx].double(), new), 1) for n, new in (("k_cache", k), ("v_cache", v)))
        h = h + _attend(q, keys, values, ctx).reshape(1, Hq * D) @ _dense(L["o"]).T
        gu = _rms(h, L["post_norm"]) @ _dense(L["gate_up"]).T
        h = h + (_silu(gu[:, :I]) * gu[:, I:]) @ _dense(L["down"]).T
        if i < 4:
            out["key%d" % i], out["value%d" % i] = k.transpose(0, 1).reshape(1, Hk, D), v.transpose(0, 1).reshape(1, Hk, D)
    x, w = _rms(h, d["norm"]), d["head"]
    step = 16384  # rows of the head at a time
    out["logits"] = torch.cat([x @ _dense(tuple(t[r:r + step] for t in w)).T for r in range(0, c["vocab"], step)], -1)
    return out
