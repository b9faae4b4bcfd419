"""The work this framework does for its users, as cases to be timed: GGUF weights rebuilt (plain and with a LoRA), GGUF
linears from one activation row to a whole video latent, the int8 W8A8 linear and the int8 MLP / QKV of a DiT block
with its fused quantiser operations, and a forward whose blocks stream from host memory.

``listed()`` gives the fixed cases, ``draw(rng)`` another one of the same ranges, ``prepare(case, seed)`` what a program
holds before the call, ``run(state)`` one pass, ``work(case)`` the bytes and operations it cannot do without,
``tolerance(case)`` how far another correct implementation may be, ``exact(case, seed)`` the result in float64 (the
quantisation steps that define the int8 path, and the rounding of a weight to its dequantised bf16 value, are part of
what is computed and kept)."""
import importlib
import math
import types

import torch

_PKG = "comfyui-weightferry_amd"


def _mod(name):
    return importlib.import_module(f"{_PKG}.{name}")


# GGML types: bytes and values per block
_BLOCK = {3: (20, 32), 7: (24, 32), 8: (34, 32), 12: (144, 256), 13: (176, 256), 14: (210, 256)}
_FUSED = (12, 13, 14, 8)


# ------------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # a 14B DiT's FFN weight rebuilt for one layer call (ComfyUI-GGUF does it for every layer of every step)
        {"name": "dequant_q4_k_ffn", "kind": "dequant", "qtype": 12, "n": 13824, "k": 5120},
        # the smallest call: one attention weight of a 2B DiT, where the launch and the host path count
        {"name": "dequant_q5_1_attn", "kind": "dequant", "qtype": 7, "n": 2048, "k": 2048},
        # an FFN weight of a 2B DiT with one rank-32 LoRA, the factors on the host as ComfyUI-GGUF keeps them
        {"name": "lora_q5_1_ffn", "kind": "lora", "qtype": 7, "n": 8192, "k": 2048, "rank": 32},
        # one row: timestep embedding and modulation layers of a 14B DiT
        {"name": "linear_q4_k_1_row", "kind": "linear", "qtype": 12, "rows": 1, "n": 5120, "k": 5120, "bias": True},
        # a short text context (77 tokens), a size that fits no tile
        {"name": "linear_q6_k_77_rows", "kind": "linear", "qtype": 14, "rows": 77, "n": 5120, "k": 5120, "bias": True},
        # the 512-token text context of the cross-attention's k and v
        {"name": "linear_q5_k_512_rows", "kind": "linear", "qtype": 13, "rows": 512, "n": 5120, "k": 5120,
         "bias": True},
        # one 832 x 480 latent frame (1560 tokens) through the FFN's second layer, 8-bit weights
        {"name": "linear_q8_0_1560_rows", "kind": "linear", "qtype": 8, "rows": 1560, "n": 5120, "k": 13824,
         "bias": True},
        # a 4096-token latent through the FFN's first layer
        {"name": "linear_q4_k_4096_rows", "kind": "linear", "qtype": 12, "rows": 4096, "n": 13824, "k": 5120,
         "bias": True},
        # the int8 linear on a short context, plain per-token activations
        {"name": "int8_plain_256_rows", "kind": "int8", "rows": 256, "n": 5120, "k": 5120, "convrot": False,
         "bias": True},
        # the int8 ConvRot linear on a whole video latent: the largest call
        {"name": "int8_convrot_16384_rows", "kind": "int8", "rows": 16384, "n": 5120, "k": 5120, "convrot": True,
         "bias": False},
        # the MLP of an int8 2B DiT block at 896 x 1472 with classifier-free guidance (2 x 56 x 92 / 2 tokens): LayerNorm
        # and modulation inside the first quantiser, GELU inside the second, the gated residual in the last epilogue
        {"name": "int8_mlp_5152_rows", "kind": "int8_mlp", "batch": 2, "rows": 2576, "width": 2048, "hidden": 8192,
         "op": "lnmod"},
        # a forward with six 2B-DiT-sized Q4_K blocks streamed from page-locked host memory through two slots
        {"name": "streamed_6_blocks", "kind": "stream", "blocks": 6, "dim": 2048, "heads": 16, "ffn": 8192,
         "rows": 1024, "context": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dequant", "lora"] + ["linear"] * 6 + ["int8"] * 3 + ["int8_mlp", "int8_qkv", "stream"])
    width = lambda: 256 * _log_int(rng, 4, 54)                                        # noqa: E731 -- 1024 .. 13824
    out = lambda: rng.choice([_log_int(rng, 1000, 13824), 16 * _log_int(rng, 64, 864)])   # noqa: E731 -- any, or whole
    if kind == "dequant":
        return {"kind": kind, "qtype": rng.choice(sorted(_BLOCK)), "n": out(), "k": width()}
    if kind == "lora":
        return {"kind": kind, "qtype": rng.choice(sorted(_BLOCK)), "n": 16 * _log_int(rng, 64, 320),
                "k": 256 * _log_int(rng, 4, 20), "rank": rng.choice([4, 16, 32, 64])}
    if kind == "linear":
        case = {"kind": kind, "qtype": rng.choice([12, 13, 14, 8, 12, 13, 14, 8, 7]), "rows": _log_int(rng, 1, 4096),
                "n": out(), "k": width(), "bias": rng.random() < 0.7}
        most = 4096 * 13824 * 5120
    elif kind == "int8":
        convrot = rng.random() < 0.5
        case = {"kind": kind, "rows": _log_int(rng, 3, 16384), "n": out(),
                "k": width() if convrot else rng.choice([width(), 64 * _log_int(rng, 16, 216)]), "convrot": convrot,
                "bias": not convrot and rng.random() < 0.5}
        most = 16384 * 5120 * 5120
    elif kind == "int8_mlp":
        op = rng.choice(["lnmod", "mod"])
        width_ = rng.choice([1024, 2048, 4096]) if op == "lnmod" else 256 * rng.randint(4, 20)
        return {"kind": kind, "batch": rng.choice([1, 2]), "rows": _log_int(rng, 64, 4096) // 2 * 2, "width": width_,
                "hidden": 256 * rng.randint(8, 32), "op": op}
    elif kind == "int8_qkv":
        op = rng.choice(["lnmod", "mod"])
        width_ = rng.choice([1024, 2048, 4096]) if op == "lnmod" else 256 * rng.randint(4, 20)
        return {"kind": kind, "batch": rng.choice([1, 2]), "rows": _log_int(rng, 64, 4096), "width": width_, "op": op}
    else:
        return {"kind": kind, "blocks": rng.randint(3, 6), "dim": rng.choice([1024, 1536, 2048]), "heads": 16,
                "ffn": 1024 * rng.randint(4, 8), "rows": _log_int(rng, 128, 1024), "context": rng.randint(77, 512)}
    while case["rows"] * case["n"] * case["k"] > most:
        case["rows"] = case["rows"] // 2 + 1
    return case


# ----------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(torch.bfloat16)


def _gguf(g, qtype, n, k):
    """Random GGML blocks for an [n, k] weight of about N(0, 0.02)'s size: every quant and scale code at random, the
    float16 scales within a factor of three of each other."""
    size, per = _BLOCK[qtype]
    nb = n * k // per
    raw = torch.randint(0, 256, (nb, size), generator=g, device="cuda", dtype=torch.uint8)

    def scale(at, typical, sign=1.0):
        v = (torch.rand(nb, generator=g, device="cuda") + 0.5) * typical * sign
        raw[:, at:at + 2] = v.half().view(torch.uint8).view(nb, 2)
    if qtype in (12, 13):
        scale(0, 1.0e-4 if qtype == 12 else 5.0e-5)
        scale(2, 8.0e-4)
    elif qtype == 14:
        scale(208, 1.0e-5)
    elif qtype == 8:
        scale(0, 3.0e-4)
    elif qtype in (3, 7):
        step = 5.0e-3 if qtype == 3 else 2.5e-3
        scale(0, step)
        scale(2, step * (7.5 if qtype == 3 else 15.5), -1.0)
    return raw.view(-1)


class _Int8Weight:
    """The fields of ComfyUI's quantised int8 ConvRot weight that the int8 path reads."""

    def __init__(self, w_q, scale):
        self._layout_cls, self._qdata = "TensorWiseINT8Layout", w_q
        self._params = types.SimpleNamespace(scale=scale, convrot=True, transposed=False, convrot_groupsize=256)
        self.shape, self.dtype = w_q.shape, torch.bfloat16


class _Linear:
    """ComfyUI's quantised linear: its forward hands input, weight and bias to ``_forward``."""

    def __init__(self, weight):
        self.weight, self.bias = weight, None

    def _forward(self, input, weight, bias):
        raise RuntimeError("the int8 path declined this layer")

    def __call__(self, x):
        return self._forward(x, self.weight, self.bias)


def _int8_weight(g, n, k):
    w_q = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    return w_q, torch.rand(n, generator=g, device="cuda") * 2.0e-4 + 2.0e-4


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    t = types.SimpleNamespace(case=case)
    if kind in ("dequant", "lora", "linear"):
        t.raw = _gguf(g, case["qtype"], case["n"], case["k"])
    if kind == "lora":
        t.up = _randn(g, case["n"], case["rank"], std=0.05).cpu()
        t.down = _randn(g, case["rank"], case["k"], std=0.05).cpu()
        t.factor = 0.75
    if kind in ("linear", "int8"):
        t.x = _randn(g, case["rows"], case["k"])
        t.bias = _randn(g, case["n"], std=0.02) if case["bias"] else None
    if kind == "int8":
        t.w_q, t.ws = _int8_weight(g, case["n"], case["k"])
    if kind in ("int8_mlp", "int8_qkv"):
        b, w = case["batch"], case["width"]
        height = 2 if case["rows"] % 2 == 0 else 1
        t.x = _randn(g, b, 1, height, case["rows"] // height, w, std=1.5, mean=0.1)
        t.scale, t.shift, t.gate = (_randn(g, b, 1, 1, 1, w, std=s) for s in (0.2, 0.2, 0.5))
        t.norm = torch.nn.LayerNorm(w, elementwise_affine=False, eps=1e-6)
        t.src = t.x if case["op"] == "lnmod" else t.norm(t.x)
        shapes = [(case["hidden"], w), (w, case["hidden"])] if kind == "int8_mlp" else [(w, w)] * 3
        t.weights = [_int8_weight(g, n, k) for n, k in shapes]
    if kind == "stream":
        d, f = case["dim"], case["ffn"]
        t.x, t.ctx = _randn(g, 1, case["rows"], d), _randn(g, 1, case["context"], d)
        shapes = [(d, d)] * 8 + [(f, d), (d, f)]
        t.weights = [[(_gguf(g, 12, n, k), _randn(g, n, std=0.01), n, k) for n, k in shapes]
                     for _ in range(case["blocks"])]
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "lora":
        t.loras = [(t.up, t.down, t.factor)]
    elif case["kind"] in ("int8_mlp", "int8_qkv"):
        t.layers = [_Linear(_Int8Weight(w_q, ws)) for w_q, ws in t.weights]
    elif case["kind"] == "stream":
        model = _mod("streaming.synthetic").WanLikeStack(case["blocks"], case["dim"], case["heads"], case["ffn"], 12)
        for block, weights in zip(model.blocks, t.weights):
            for lin, (raw, bias, _n, _k) in zip(block.linears(), weights):
                lin.weight.data.copy_(raw)
                lin.bias.data.copy_(bias)
        t.weights = None
        t.model = _mod("streaming.dit_node").apply_streaming(model, device=torch.device("cuda", 0), prefetch_slots=2,
                                                             profile=False)
    return t


# --------------------------------------------------------------------------------------------------- one pass
def _taken(y):
    if y is None:
        raise RuntimeError("the library declined this call")
    return y


def run(t):
    with torch.no_grad():
        return _run(t)


def _run(t):
    case = t.case
    kind = case["kind"]
    if kind == "dequant":
        return _taken(_mod("enhancers.gguf_dequant").dequantize(t.raw, case["qtype"], (case["n"], case["k"]), None,
                                                                torch.bfloat16))
    if kind == "lora":
        return _taken(_mod("enhancers.gguf_dequant").dequantize_lora(t.raw, case["qtype"], (case["n"], case["k"]), None,
                                                                     torch.bfloat16, t.loras))
    if kind == "linear":
        return _taken(_mod("enhancers.fused_gguf").linear(t.x, t.raw, case["qtype"], (case["n"], case["k"]), t.bias))
    fi = _mod("enhancers.fused_int8")
    if kind == "int8":
        return _taken(fi.int8_linear(t.x, t.w_q, t.ws, t.bias, convrot=case["convrot"]))
    if kind == "stream":
        return t.model(t.x, t.ctx)
    norm = t.norm if case["op"] == "lnmod" else None
    if kind == "int8_qkv":
        with fi._Overrides(t.layers):
            fi._set_pre(t.src, case["op"], t.scale, t.shift, norm=norm)
            try:
                flat = t.src.view(case["batch"], case["rows"], case["width"])
                return [layer(flat) for layer in t.layers]
            finally:
                fi._clear_pre()
    first, second = t.layers
    state = _mod("enhancers.fused_state")._tls
    with fi._Overrides([first, (second, fi._residual_forward)]):
        fi._set_pre(t.src, case["op"], t.scale, t.shift, norm=norm)
        try:
            h = first(t.src)
            fi._clear_pre()
            fi._set_pre(h, "gelu")
            state.res = {"x": t.x, "gate": t.gate, "done": False, "same": False}
            return [h, second(h)]
        finally:
            state.res = None
            fi._clear_pre()


# ------------------------------------------------------------------------------------------------------- work
def _weight_bytes(case):
    size, per = _BLOCK[case["qtype"]]
    return case["n"] * case["k"] // per * size


def work(case):
    kind = case["kind"]
    if kind == "dequant":
        return {"bytes": _weight_bytes(case) + 2 * case["n"] * case["k"], "flops": 2 * case["n"] * case["k"]}
    if kind == "lora":
        n, k, r = case["n"], case["k"], case["rank"]
        return {"bytes": _weight_bytes(case) + 2 * n * k + 2 * r * (n + k), "flops": 2 * n * k * r}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _weight_bytes(case) + 2 * m * (n + k) + 2 * n * case["bias"], "flops": 2 * m * n * k}
    if kind == "int8":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k + 2 * m * (n + k) + 4 * n + 2 * n * case["bias"], "flops": 2 * m * n * k}
    if kind in ("int8_mlp", "int8_qkv"):
        m, w = case["batch"] * case["rows"], case["width"]
        if kind == "int8_qkv":
            return {"bytes": 3 * w * w + 8 * m * w + 12 * w, "flops": 6 * m * w * w}
        f = case["hidden"]
        return {"bytes": 2 * f * w + 2 * m * (2 * w + f) + 2 * m * f + 4 * (f + w), "flops": 4 * m * f * w}
    m, c, d, f = case["rows"], case["context"], case["dim"], case["ffn"]
    weights = (8 * d * d + 2 * d * f) // 256 * 144
    flops = 2 * d * d * (6 * m + 2 * c) + 4 * m * d * f + 4 * m * (m + c) * d
    return {"bytes": case["blocks"] * weights + 4 * m * d + 2 * c * d, "flops": case["blocks"] * flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "lora":
        # the difference's float32 sum in another order moves few bf16 roundings, by one step each (6e-6 measured)
        return {"rel": 3.0e-5, "max": 1.6e-2}
    if kind == "linear":
        # the same for a product's float32 sum (1.0e-4 measured, at one row)
        return {"rel": 4.0e-4, "max": 1.6e-2}
    if kind == "stream":
        # such roundings travel through the blocks that follow (3.8e-3 measured between two forms of the linears)
        return {"rel": 1.5e-2}
    # a format's rounding chain; integer sums between a fixed quantiser and a fixed epilogue: whole bits
    return "exact"


# ------------------------------------------------------------------------------------------- float64 results
def _dense(raw, qtype, n, k, dt):
    """The [n, k] weight of GGML blocks with every step of the format's formula in ``dt``."""
    size, per = _BLOCK[qtype]
    b = raw.view(-1, size)
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).to(dt)          # noqa: E731 -- [nb, 1]
    if qtype == 8:
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).to(dt)
    elif qtype in (3, 7):
        qs = b[:, -16:]
        q = torch.cat([qs & 15, qs >> 4], dim=1)
        if qtype == 7:
            q = q | (((b[:, 4:8].unsqueeze(2) >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1) << 4).view(-1, 32)
        w = half(0) * q.to(dt) + half(2)
    elif qtype in (12, 13):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1)
        qs = b[:, -128:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], dim=2).view(-1, 8, 32)
        if qtype == 13:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (((b[:, 16:48].unsqueeze(1) >> bit) & 1) << 4)
        step = (half(0) * sc.to(dt)).unsqueeze(2)
        w = step * q.to(dt) - (half(2) * mn.to(dt)).unsqueeze(2)
    else:
        ql, qh = b[:, :128].view(-1, 2, 1, 64), b[:, 128:192].view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], dim=2).view(-1, 2, 4, 32)
        shift = torch.arange(0, 8, 2, device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (lo | (((qh >> shift) & 3) << 4)).to(torch.int8).view(-1, 16, 16) - 32
        step = half(208) * b[:, 192:208].contiguous().view(torch.int8).to(dt)
        w = step.unsqueeze(2) * q.to(dt)
    return w.reshape(n, k)


def _weight(raw, qtype, n, k):
    """The weight a layer multiplies by: float16 steps, rounded to bf16."""
    return _dense(raw, qtype, n, k, torch.float16).to(torch.bfloat16).double()


def _linear64(x, raw, qtype, n, k, bias):
    y = x.double() @ _weight(raw, qtype, n, k).t()
    return y if bias is None else y + bias.double()


def _rotate(x):
    """The ConvRot rotation of float32 rows: per 256-group, radix-4 butterflies of stride 1, 4, 16, 64, over 16."""
    m, k = x.shape
    v = x.view(m, k // 256, 4, 4, 4, 4)                  # digits of stride 64, 16, 4, 1
    for dim in (5, 4, 3, 2):
        a, b, c, d = v.unbind(dim)
        v = torch.stack([a + b + c - d, a + b - c + d, a - b + c + d, -a + b + c + d], dim=dim)
    return v.reshape(m, k) * 0.0625


def _quantise(x, convrot):
    """(int8 rows as float64, float64 scales [m, 1]) of bf16 rows, by the quantiser's float32 and bf16 steps."""
    y = x.float()
    if convrot:
        y = _rotate(y)
    scale = (y.abs().amax(dim=1, keepdim=True).clamp(max=3.38953139e38) / 127.0).clamp(min=1.0e-30)
    step = scale.to(torch.bfloat16).float()
    q = (y.to(torch.bfloat16).float() / step).to(torch.bfloat16).float().round().clamp(-128, 127)
    return q.double(), scale.double()


def _int8_64(x, w_q, ws, convrot, bias=None):
    q, s = _quantise(x, convrot)
    y = (q @ w_q.double().t()) * s * ws.double()
    return y if bias is None else y + bias.double()


def _stack64(t):
    def norm(v):
        return torch.nn.functional.layer_norm(v, (v.shape[-1],))

    heads = t.case["heads"]

    def attend(q, k, v):
        q, k, v = (u.view(u.shape[0], heads, -1).transpose(0, 1) for u in (q, k, v))
        p = torch.softmax(torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1]), dim=-1)
        return torch.matmul(p, v.contiguous()).transpose(0, 1).reshape(q.shape[1], -1)
    x, ctx = t.x[0].double(), t.ctx[0].double()
    for block in t.weights:
        lin = [lambda v, w=w: _linear64(v, w[0], 12, w[2], w[3], w[1]) for w in block]
        h = norm(x)
        x = x + lin[3](attend(lin[0](h), lin[1](h), lin[2](h)))
        h = norm(x)
        x = x + lin[7](attend(lin[4](h), lin[5](ctx), lin[6](ctx)))
        h = norm(x)
        x = x + lin[9](torch.nn.functional.gelu(lin[8](h), approximate="tanh"))
    return x.unsqueeze(0)


def exact(case, seed):
    with torch.no_grad():
        return _exact(case, _inputs(case, seed))


def _exact(case, t):
    kind = case["kind"]
    if kind == "dequant":
        return _dense(t.raw, case["qtype"], case["n"], case["k"], torch.float64)
    if kind == "lora":
        w = _dense(t.raw, case["qtype"], case["n"], case["k"], torch.float64)
        return w + t.factor * (t.up.cuda().double() @ t.down.cuda().double())
    if kind == "linear":
        return _linear64(t.x, t.raw, case["qtype"], case["n"], case["k"], t.bias)
    if kind == "int8":
        return _int8_64(t.x, t.w_q, t.ws, case["convrot"], t.bias)
    if kind == "stream":
        return _stack64(t)
    # the operations before a quantiser round to bf16 where the block's own tensors would
    v = t.src
    if case["op"] == "lnmod":
        v = torch.nn.functional.layer_norm(v.double(), (case["width"],), eps=1e-6).to(torch.bfloat16)
    v = v * (1 + t.scale) + t.shift
    rows = v.reshape(-1, case["width"])
    if kind == "int8_qkv":
        return [_int8_64(rows, w_q, ws, True).view(case["batch"], case["rows"], -1) for w_q, ws in t.weights]
    h = _int8_64(rows, *t.weights[0], True)
    a = torch.nn.functional.gelu(h.to(torch.bfloat16).double()).to(torch.bfloat16)
    y = _int8_64(a, *t.weights[1], True).to(torch.bfloat16).double().view(t.x.shape)
    return [h.view(*t.x.shape[:-1], case["hidden"]), t.x.double() + t.gate.double() * y]
