"""The performance cases of the framework: the calls its users make, through the public host API (we.py, block.py).

listed() names one case per kind of call, from a single int4 decode row to a whole double-stream block; draw() gives
further cases of the same ranges. One Graph (context) serves every case of a process and owns the device buffers, as in
a user's program; inputs are made with torch and copied into them on the GPU, and results are torch views of them.
"""
import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "web-engine_amd"))

import block  # noqa: E402
import we  # noqa: E402

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1, "int4": 0.5}
GROUP = 64  # int4 scale group
FP8_RMS = 96.0  # normal weights at this scale use the e4m3 range (448 at 4.7 sigma)


def listed():
    return [
        # one token of a language model's largest projection: the smallest call, weight-bandwidth and launch bound
        {"name": "int4_decode", "kind": "linear", "m": 1, "n": 18944, "k": 3584, "x": "f16", "w": "int4", "bias": False,
         "gelu": False, "lora": 0},
        # the same projection on a prompt
        {"name": "int4_prefill", "kind": "linear", "m": 509, "n": 18944, "k": 3584, "x": "f16", "w": "int4",
         "bias": False, "gelu": False, "lora": 0},
        # a small batch of rows through a square projection (the time / pooled-text embedders of a DiT)
        {"name": "linear_small", "kind": "linear", "m": 64, "n": 3072, "k": 3072, "x": "bf16", "w": "fp8", "bias": True,
         "gelu": False, "lora": 0},
        # a LoRA-adapted projection in the reference's own activation type
        {"name": "linear_lora_f32", "kind": "linear", "m": 1024, "n": 6144, "k": 6144, "x": "f32", "w": "fp8",
         "bias": False, "gelu": False, "lora": 32},
        # the DiT MLP of the benchmark: the image tokens of a 1024 x 1024 picture
        {"name": "mlp_image", "kind": "mlp", "tokens": 4096, "hidden": 3072, "mlp": 12288, "dtype": "bf16",
         "gated": False},
        # the same MLP on a short, ragged text stream
        {"name": "mlp_text", "kind": "mlp", "tokens": 333, "hidden": 3072, "mlp": 12288, "dtype": "bf16",
         "gated": False},
        # the single-stream block's gated MLP in f32, the reference's dtype (a 512 x 512 picture and a prompt)
        {"name": "mlp_gated_f32", "kind": "mlp", "tokens": 1103, "hidden": 6144, "mlp": 16384, "dtype": "f32",
         "gated": True},
        # a fused QKV projection with bf16 weights, q / k norm and RoPE
        {"name": "qkv_bf16", "kind": "qkv", "tokens": 4096, "heads": 24, "kv_heads": 24, "x": "bf16", "w": "bf16"},
        # joint attention of the benchmark's block
        {"name": "attention_bf16", "kind": "attention", "tokens": 4608, "heads": 24, "kv_heads": 24, "dim": 128,
         "causal": False, "dtype": "bf16"},
        # grouped-query attention of the single-stream block in f32
        {"name": "attention_f32", "kind": "attention", "tokens": 1103, "heads": 48, "kv_heads": 12, "dim": 128,
         "causal": False, "dtype": "f32"},
        # a 3x3 convolution of an image decoder
        {"name": "conv3x3_f32", "kind": "conv", "height": 128, "width": 128, "cin": 384, "cout": 384, "w": "f32"},
        # the whole double-stream block of the benchmark: the largest call
        {"name": "block_double", "kind": "block", "text": 512, "rows": 64, "columns": 64},
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))) if lo > 0 else 0


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "qkv", "attention", "attention", "conv", "block"])
    if kind == "linear":
        w = rng.choice(["int4", "int4", "fp8", "fp8", "bf16"])
        x = rng.choice(["f16", "bf16"] if w == "int4" else ["bf16", "bf16", "f32"])
        lora = rng.choice([0, 0, 16, 32, 64]) if w != "int4" else 0
        return {"kind": kind, "m": _log(rng, 1, 2048), "n": 16 * _log(rng, 64, 1184), "k": 64 * _log(rng, 24, 128), "x": x,
                "w": w, "bias": rng.random() < 0.5, "gelu": rng.random() < 0.25, "lora": lora}
    if kind == "mlp":
        if rng.random() < 0.5:
            return {"kind": kind, "tokens": _log(rng, 64, 4096), "hidden": 3072, "mlp": 12288, "dtype": "bf16",
                    "gated": False}
        return {"kind": kind, "tokens": _log(rng, 64, 1152), "hidden": 64 * rng.randint(48, 96),
                "mlp": 64 * rng.randint(128, 256), "dtype": rng.choice(["f32", "bf16"]), "gated": True}
    if kind == "qkv":
        heads = rng.choice([16, 24, 32])
        return {"kind": kind, "tokens": _log(rng, 64, 4096), "heads": heads, "kv_heads": rng.choice([heads, heads // 4]),
                "x": "bf16", "w": rng.choice(["bf16", "fp8"])}
    if kind == "attention":
        heads = rng.choice([16, 24, 32])
        dtype = rng.choice(["bf16", "f16", "f32"])
        return {"kind": kind, "tokens": _log(rng, 64, 1536 if dtype == "f32" else 4608), "heads": heads,
                "kv_heads": rng.choice([heads, heads // 4]), "dim": rng.choice([64, 128, 128]),
                "causal": rng.random() < 0.5, "dtype": dtype}
    if kind == "conv":
        return {"kind": kind, "height": rng.randint(32, 128), "width": rng.randint(32, 128), "cin": 32 * rng.randint(3, 12),
                "cout": 32 * rng.randint(3, 12), "w": rng.choice(["f32", "f32", "bf16"])}
    return {"kind": kind, "text": rng.randint(64, 512), "rows": rng.randint(16, 64), "columns": rng.randint(16, 64)}


# ------------------------------------------------------------------------------------------------------- inputs

_graph = None


def _the_graph():
    global _graph
    if _graph is None:
        _graph = we.Graph(0)
    return _graph


class _Device:
    """A buffer of the graph that holds a tensor's bytes; `t` is its torch view, which keeps it alive."""

    def __init__(self, graph, nbytes):
        self.graph, self.buf = graph, graph.buffer(nbytes)
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (self.buf.ptr, False), "version": 2}

    def __del__(self):
        if self.graph.ctx is not None:
            self.graph.free(self.buf)


def _empty(graph, shape, dtype):
    n = math.prod(shape) * torch.empty(0, dtype=dtype).element_size()
    return torch.as_tensor(_Device(graph, n), device="cuda").view(dtype).reshape(shape)


def _resident(graph, v):
    """v (tensors in dicts and lists) with every tensor in a buffer of the graph"""
    if isinstance(v, torch.Tensor):
        t = _empty(graph, tuple(v.shape), v.dtype)
        graph.sync()  # a fresh buffer is zeroed on the graph's stream
        t.copy_(v)
        return t
    if isinstance(v, dict):
        return {k: _resident(graph, x) for k, x in v.items()}
    if isinstance(v, (list, tuple)):
        return [_resident(graph, x) for x in v]
    return v


class _Inputs:
    """Seeded tensors of one case, made on `device`."""

    def __init__(self, seed, device="cuda"):
        self.device = device
        self.g = torch.Generator(device=device)
        self.g.manual_seed(seed)

    def normal(self, *shape, rms=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=self.device) * rms).to(dtype)

    def weight(self, dtype, n, k):
        """(stored tensor, its per-tensor scale, int4 scales): rows of about unit output for unit inputs"""
        if dtype == "int4":
            q = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), generator=self.g, device=self.device, dtype=torch.int64)
            s = (torch.randn(n, k // GROUP, generator=self.g, device=self.device) * 0.01).abs()
            return q.to(torch.int32), 1.0, s.to(torch.float16)
        if dtype == "fp8":
            w = (torch.randn(n, k, generator=self.g, device=self.device) * FP8_RMS).clamp_(-448, 448)
            return w.to(torch.float8_e4m3fn), 1.0 / (FP8_RMS * math.sqrt(k)), None
        return self.normal(n, k, rms=k ** -0.5, dtype=TORCH[dtype]), 1.0, None

    def linear(self, dtype, n, k, bias=False):
        w, scale, scales = self.weight(dtype, n, k)
        return {"dtype": dtype, "n": n, "k": k, "w": w, "scale": scale, "scales": scales,
                "bias": self.normal(n, rms=0.1) if bias else None, "lora": None}


def _ptr(t):
    return None if t is None else t.data_ptr()


def _handle(lin):
    """the we.Linear a program keeps for a layer"""
    lora = None if lin["lora"] is None else tuple(_handle(p) for p in lin["lora"])
    return we.Linear(_ptr(lin["w"]), lin["dtype"], lin["scale"], lin["n"], lin["k"], bias=_ptr(lin["bias"]), lora=lora,
                     scales=_ptr(lin["scales"]), group=GROUP)


def _dense(lin):
    """a layer's weights in f64, with its scale"""
    if lin["dtype"] == "int4":
        n, k = lin["n"], lin["k"]
        sh = torch.arange(0, 32, 4, device=lin["w"].device, dtype=torch.int32)
        q = (lin["w"].unsqueeze(-1) >> sh) & 15
        q = torch.where(q > 7, q - 16, q).reshape(n, k // GROUP, GROUP).double()
        return (q * lin["scales"].double().unsqueeze(-1)).reshape(n, k)
    w = lin["w"]
    return (w.float() if lin["dtype"] == "fp8" else w).double() * lin["scale"]


def _apply(x, lin):
    y = x @ _dense(lin).t()
    if lin["bias"] is not None:
        y = y + lin["bias"].double()
    if lin["lora"] is not None:
        down, up = lin["lora"]
        y = y + (x @ _dense(down).t()) @ _dense(up).t()
    return y


def _rope(tokens, head_dim=128, theta=10000.0):
    """interleaved RoPE tables f64 of a square-ish image grid, as block.rope_for_image makes them"""
    cols = max(1, int(math.isqrt(tokens)))
    pos = block.positions(0, (tokens + cols - 1) // cols, cols)[:tokens, 1:]
    cos, sin, _ = block.rope_tables(pos, (head_dim // 2, head_dim // 2), theta)
    return torch.from_numpy(cos), torch.from_numpy(sin)


def _data(case, seed, device="cuda"):
    """the values a program holds before the call, as tensors"""
    i = _Inputs(seed, device)
    kind = case["kind"]
    if kind == "linear":
        lin = i.linear(case["w"], case["n"], case["k"], case["bias"])
        if case["lora"]:
            up = i.linear("bf16", case["n"], case["lora"])
            up["scale"] = 0.5  # alpha / rank
            lin["lora"] = (i.linear("bf16", case["lora"], case["k"]), up)
        return {"x": i.normal(case["m"], case["k"], dtype=TORCH[case["x"]]), "lin": lin}
    if kind == "mlp":
        H, M = case["hidden"], case["mlp"]
        return {"x": i.normal(case["tokens"], H, dtype=TORCH[case["dtype"]]),
                "gate": i.linear("fp8", M, H) if case["gated"] else None, "up": i.linear("fp8", M, H),
                "down": i.linear("fp8", H, M)}
    if kind == "qkv":
        H = case["heads"] * 128
        cos, sin = _rope(case["tokens"])
        return {"x": i.normal(case["tokens"], H, dtype=TORCH[case["x"]]),
                "lin": i.linear(case["w"], (case["heads"] + 2 * case["kv_heads"]) * 128, H),
                "norm_q": i.normal(128, rms=0.1), "norm_k": i.normal(128, rms=0.1), "cos": cos.to(device).contiguous(),
                "sin": sin.to(device).contiguous()}
    if kind == "attention":
        t, d, dt = case["tokens"], case["dim"], TORCH[case["dtype"]]
        return {"q": i.normal(t, case["heads"], d, dtype=dt), "k": i.normal(t, case["kv_heads"], d, dtype=dt),
                "v": i.normal(t, case["kv_heads"], d, dtype=dt)}
    if kind == "conv":
        w = i.normal(case["cout"], 9 * case["cin"], rms=(9 * case["cin"]) ** -0.5, dtype=TORCH[case["w"]])
        return {"x": i.normal(case["height"] * case["width"], case["cin"]), "w": w}
    cfg = block.DIT_DOUBLE_BLOCK
    H, M, dt = cfg.hidden, cfg.mlp, torch.bfloat16
    d = {"tvec": i.normal(6 * H, rms=0.5), "x": [], "streams": []}
    for tokens in (case["text"], case["rows"] * case["columns"]):
        d["x"].append(i.normal(tokens, H, dtype=dt))
        d["streams"].append({"qkv": i.linear("fp8", 3 * H, H), "proj": i.linear("fp8", H, H), "up": i.linear("fp8", M, H),
                             "down": i.linear("fp8", H, M), "norm1": i.normal(H, rms=0.1), "norm2": i.normal(H, rms=0.1),
                             "norm_q": i.normal(128, rms=0.1), "norm_k": i.normal(128, rms=0.1),
                             "table": i.normal(6 * H, rms=0.5)})
    return d


class _Block:
    """a DoubleBlock with its RoPE tables, whose device buffers go back with it"""

    def __init__(self, graph, case):
        self.graph = graph
        self.body = block.DoubleBlock(graph, block.DIT_DOUBLE_BLOCK, case["text"], case["rows"] * case["columns"])
        self.rope = block.rope_for_image(graph, case["rows"], case["columns"])

    def __del__(self):
        if self.graph.ctx is not None:
            self.body.free()
            self.graph.free(self.rope.cos)
            self.graph.free(self.rope.sin)


def prepare(case, seed):
    g = _the_graph()
    s = {"case": case, "graph": g, **_resident(g, _data(case, seed))}
    kind = case["kind"]
    if kind == "linear":
        s["layer"] = _handle(s["lin"])
        s["y"] = _empty(g, (case["m"], case["n"]), s["x"].dtype)
    elif kind == "mlp":
        s["layers"] = {name: _handle(s[name]) for name in ("gate", "up", "down") if s[name] is not None}
        s["u"] = _empty(g, (case["tokens"], case["mlp"]), s["x"].dtype)
        s["y"] = _empty(g, tuple(s["x"].shape), s["x"].dtype)
    elif kind == "qkv":
        s["y"] = _empty(g, (case["tokens"], s["lin"]["n"]), s["x"].dtype)
        s["params"] = we.matmul_params(case["tokens"], s["lin"]["n"], s["lin"]["k"], s["lin"]["scale"], graph=g)
    elif kind == "attention":
        s["y"] = _empty(g, tuple(s["q"].shape), s["q"].dtype)
    elif kind == "conv":
        s["y"] = _empty(g, (s["x"].shape[0], case["cout"]), torch.float32)
        s["params"] = we.conv3x3_params(case["height"], case["width"], case["cin"], case["cout"], graph=g)
    else:
        s["block"] = _Block(g, case)
        s["weights"] = [block.StreamWeights(*(_handle(w[n]) for n in ("qkv", "proj", "up", "down")),
                                            *(_ptr(w[n]) for n in ("norm1", "norm2", "norm_q", "norm_k", "table")))
                        for w in s["streams"]]
        s["y"] = [_empty(g, tuple(x.shape), x.dtype) for x in s["x"]]
    torch.cuda.synchronize()  # torch's copies are on its own stream
    return s


def run(s):
    g, case = s["graph"], s["case"]
    kind = case["kind"]
    if kind == "linear":
        dt = we.DTYPES[case["x"]]
        if case["lora"]:  # the LoRA path leaves its temporaries to the caller's mark / release
            mark = g.mark()
            we.linear(g, _ptr(s["x"]), s["layer"], case["m"], dt, dt, gelu_tanh=case["gelu"], out=_ptr(s["y"]))
            g.release(mark)
        else:
            we.linear(g, _ptr(s["x"]), s["layer"], case["m"], dt, dt, gelu_tanh=case["gelu"], out=_ptr(s["y"]))
        return s["y"]
    if kind == "mlp":
        dt, L, t = we.DTYPES[case["dtype"]], s["layers"], case["tokens"]
        x, u, y = _ptr(s["x"]), _ptr(s["u"]), _ptr(s["y"])
        if case["gated"]:
            we.linear(g, x, L["gate"], t, dt, dt, out=u)
            we.linear(g, x, L["up"], t, dt, dt, swiglu_gate=u, out=u)
        else:
            we.linear(g, x, L["up"], t, dt, dt, gelu_tanh=True, out=u)
        we.linear(g, u, L["down"], t, dt, dt, out=y)
        return s["y"]
    if kind == "qkv":
        dt = we.DTYPES[case["x"]]
        g.matmul_qk_norm_rope(s["params"], dt, _ptr(s["x"]), we.DTYPES[case["w"]], _ptr(s["lin"]["w"]), dt, _ptr(s["y"]),
                              case["heads"], case["kv_heads"], 1e-6, 1.0, _ptr(s["norm_q"]), _ptr(s["norm_k"]), 0,
                              _ptr(s["cos"]), _ptr(s["sin"]))
        return s["y"]
    if kind == "attention":
        g.attention(case["tokens"], case["heads"], case["kv_heads"], case["dim"], case["causal"], we.DTYPES[case["dtype"]],
                    _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), _ptr(s["y"]))
        return s["y"]
    if kind == "conv":
        g.matmul(s["params"], we.F32, _ptr(s["x"]), we.DTYPES[case["w"]], _ptr(s["w"]), we.F32, _ptr(s["y"]))
        return s["y"]
    s["block"].body.forward(s["weights"][0], s["weights"][1], _ptr(s["x"][0]), _ptr(s["x"][1]), _ptr(s["tvec"]),
                            s["block"].rope, _ptr(s["y"][0]), _ptr(s["y"][1]))
    return {"text": s["y"][0], "image": s["y"][1]}


# ------------------------------------------------------------------------------------------------- what it takes

def _linear_bytes(dtype, n, k):
    return n * k * BYTES[dtype] + (n * k // GROUP * 2 if dtype == "int4" else 0)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k, r = case["m"], case["n"], case["k"], case["lora"]
        return {"bytes": (m * k + m * n) * BYTES[case["x"]] + _linear_bytes(case["w"], n, k) + 2 * r * (n + k) +
                (4 * n if case["bias"] else 0), "flops": 2 * m * (n * k + r * (n + k))}
    if kind == "mlp":
        t, H, M, n = case["tokens"], case["hidden"], case["mlp"], 3 if case["gated"] else 2
        return {"bytes": 2 * t * H * BYTES[case["dtype"]] + n * H * M, "flops": 2 * t * n * H * M}
    if kind == "qkv":
        t, H, n = case["tokens"], case["heads"] * 128, (case["heads"] + 2 * case["kv_heads"]) * 128
        return {"bytes": t * (H + n) * BYTES[case["x"]] + _linear_bytes(case["w"], n, H) + 8 * 64 * t, "flops": 2 * t * n * H}
    if kind == "attention":
        t, h, kv, d = case["tokens"], case["heads"], case["kv_heads"], case["dim"]
        return {"bytes": 2 * t * d * (h + kv) * BYTES[case["dtype"]],
                "flops": 4 * t * t * d * h * (0.5 if case["causal"] else 1)}
    if kind == "conv":
        p, ci, co = case["height"] * case["width"], case["cin"], case["cout"]
        return {"bytes": 4 * p * (ci + co) + 9 * ci * co * BYTES[case["w"]], "flops": 18 * p * ci * co}
    H, M = block.DIT_DOUBLE_BLOCK.hidden, block.DIT_DOUBLE_BLOCK.mlp
    t = case["text"] + case["rows"] * case["columns"]
    weights = 4 * H * H + 2 * H * M
    return {"bytes": 2 * weights + 4 * t * H + 2 * 4 * 6 * H, "flops": 2 * t * weights + 4 * t * t * H}


def tolerance(case):
    """Relative errors of correct implementations: f32 results differ by the order of their sums, 16-bit results by the
    roundings of stored values (the result; inside an MLP or block, the intermediates; in attention the
    probabilities)."""
    kind = case["kind"]
    dtype = {"linear": case.get("x"), "qkv": case.get("x"), "conv": "f32", "block": "bf16"}.get(kind, case.get("dtype"))
    if dtype == "f32":
        return {"rel": 1e-5}
    if kind == "linear":
        return {"rel": 1.5e-3 if dtype == "f16" else 8e-3}
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------------------ the results in 64 bits

def _rms(x, weight, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + weight.double())


def _rotate(x, cos, sin):
    """x [t, heads, 128], interleaved pairs; cos, sin [t, 64]"""
    c, s = cos.double().unsqueeze(1), sin.double().unsqueeze(1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], dim=-1).flatten(-2)


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _attend(q, k, v, causal):
    """[t, heads, d] in f64, one head at a time"""
    t, heads, d = q.shape
    out = torch.empty_like(q)
    mask = torch.ones(t, t, dtype=torch.bool, device=q.device).triu(1) if causal else None
    for h in range(heads):
        g = h // (heads // k.shape[1])
        s = q[:, h].contiguous() @ k[:, g].t().contiguous() / math.sqrt(d)
        if causal:
            s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, g].contiguous()
    return out


def exact(case, seed):
    d = _data(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = _apply(d["x"].double(), d["lin"])
        return _gelu(y) if case["gelu"] else y
    if kind == "mlp":
        x = d["x"].double()
        if case["gated"]:
            gate = _apply(x, d["gate"])
            u = gate * torch.sigmoid(gate) * _apply(x, d["up"])
        else:
            u = _gelu(_apply(x, d["up"]))
        return _apply(u, d["down"])
    if kind == "qkv":
        y = _apply(d["x"].double(), d["lin"])
        for first, heads, norm in ((0, case["heads"], d["norm_q"]), (case["heads"], case["kv_heads"], d["norm_k"])):
            part = y[:, first * 128:(first + heads) * 128].reshape(-1, heads, 128)
            y[:, first * 128:(first + heads) * 128] = _rotate(_rms(part, norm, 1e-6), d["cos"], d["sin"]).flatten(1)
        return y
    if kind == "attention":
        return _attend(d["q"].double(), d["k"].double(), d["v"].double(), case["causal"])
    if kind == "conv":
        h, w, ci = case["height"], case["width"], case["cin"]
        padded = torch.zeros(h + 2, w + 2, ci, dtype=torch.float64, device=d["x"].device)
        padded[1:-1, 1:-1] = d["x"].double().reshape(h, w, ci)
        y = torch.zeros(h * w, case["cout"], dtype=torch.float64, device=d["x"].device)
        taps = d["w"].double().reshape(case["cout"], 9, ci)
        for t in range(9):
            y += padded[t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(h * w, ci) @ taps[:, t].t().contiguous()
        return y
    cfg = block.DIT_DOUBLE_BLOCK
    H, heads = cfg.hidden, cfg.heads
    pos = block.positions(0, case["rows"], case["columns"])[:, 1:]
    cos, sin, _ = block.rope_tables(pos, (64, 64), 10000.0)
    cos, sin = (torch.from_numpy(t).to(d["tvec"].device) for t in (cos, sin))
    mods, parts = [], []
    for s in (0, 1):
        w, x = d["streams"][s], d["x"][s].double()
        mod = (d["tvec"].double() + w["table"].double()).reshape(6, H)
        mods.append(mod)
        h = _rms(x, w["norm1"], cfg.eps) * (1 + mod[0]) + mod[1]
        q, k, v = _apply(h, w["qkv"]).reshape(-1, 3, heads, 128).unbind(1)
        q, k = _rms(q, w["norm_q"], cfg.eps), _rms(k, w["norm_k"], cfg.eps)
        if s == 1:
            q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
        parts.append((q, k, v))
    o = _attend(*(torch.cat([parts[0][i], parts[1][i]]) for i in range(3)), False).flatten(1)
    outs = []
    for s, rows in ((0, slice(0, case["text"])), (1, slice(case["text"], None))):
        w, mod = d["streams"][s], mods[s]
        x1 = d["x"][s].double() + mod[2] * _apply(o[rows], w["proj"])
        h = _rms(x1, w["norm2"], cfg.eps) * (1 + mod[3]) + mod[4]
        outs.append(x1 + mod[5] * _apply(_gelu(_apply(h, w["up"])), w["down"]))
    return {"text": outs[0], "image": outs[1]}
