"""What compact_amd is measured on: the work a user's program has it do, each
case through the package's public entry points.

A case is a dict of plain values:

kind "ffn"    a SwiGLU MLP (plain nn.Linear projections or LoRA / DoRA
              wrappers) whose forward is FlashFFNv3; `train` "full" (weights
              train), "adapter" (frozen base), or "none" (inference forward
              under no_grad)
kind "topk"   a FlashFFN module (top-K activation compression), full fine-tune
kind "codec"  the codec kernels as an autograd Function of a user's own calls
              them: K1 (SiLU * up + quantise both), then K2 (dequantise +
              SwiGLU backward + h_mid)

Inputs follow BASELINE's distributions: x, grad_y ~ N(0, 1), weights
~ N(0, 0.02), LoRA A kaiming-uniform, B ~ N(0, 0.01), alpha = 2 r.
"""

import math

import torch
import torch.nn as nn

import compact_amd as cpt
from compact_amd.model_patch import LoraLinear

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _ffn(name, batch, seq, d_model, d_ff, cache, group, train, dtype="bf16", adapter="none",
         rank=0, outliers=0.0):
    return {"name": name, "kind": "ffn", "batch": batch, "seq": seq, "d_model": d_model,
            "d_ff": d_ff, "cache": cache, "group": group, "train": train, "dtype": dtype,
            "adapter": adapter, "rank": rank, "outliers": outliers}


def listed():
    return [
        # one generation step of a patched TinyLlama with its adapters: 4
        # sequences, one token each (launch latency and weight streaming)
        _ffn("generate_4_tokens", 4, 1, 2048, 5632, "int4", 64, "none", adapter="lora", rank=8),
        # scoring one ragged prompt with a patched Llama-7B (evaluation)
        _ffn("score_333_tokens_7b", 1, 333, 4096, 11008, "int8", 128, "none"),
        # a small LoRA fine-tuning batch (GLUE-length sequences), no cache kept
        _ffn("lora_4x128_recompute", 4, 128, 2048, 5632, "recompute", 64, "adapter",
             adapter="lora", rank=8),
        # a LoRA fine-tuning batch padded to its longest sequence (ragged)
        _ffn("lora_16x113_int4", 16, 113, 2048, 5632, "int4", 64, "adapter", adapter="lora",
             rank=8),
        # one MLP of the TinyLlama full fine-tune step
        _ffn("full_8x1024_int8", 8, 1024, 2048, 5632, "int8", 128, "full"),
        # Llama-7B MLP, full fine-tune: the headline configuration
        _ffn("full_7b_8x1024_int8", 8, 1024, 4096, 11008, "int8", 128, "full"),
        # Llama-7B MLP, LoRA with int4 codes and 1% outlier channels
        _ffn("lora_7b_8x1024_int4_outliers", 8, 1024, 4096, 11008, "int4", 64, "adapter",
             adapter="lora", rank=16, outliers=0.01),
        # single-precision full fine-tune of a TinyLlama MLP
        _ffn("full_fp32_4x512_int8", 4, 512, 2048, 5632, "int8", 128, "full", dtype="fp32"),
        # half-precision LoRA fine-tune
        _ffn("lora_fp16_4x512_int4", 4, 512, 2048, 5632, "int4", 64, "adapter", dtype="fp16",
             adapter="lora", rank=8),
        # DoRA fine-tune of a Llama-7B MLP
        _ffn("dora_7b_2x1024_int4", 2, 1024, 4096, 11008, "int4", 64, "adapter", adapter="dora",
             rank=16),
        # the top-K compressed FFN (kept fraction 0.3), full fine-tune
        {"name": "topk_4x512", "kind": "topk", "batch": 4, "seq": 512, "d_model": 2048,
         "d_ff": 5632, "keep": 0.3, "dtype": "bf16"},
        # the codec kernels alone on a wide MLP's activations
        {"name": "codec_2048x14336_int8", "kind": "codec", "rows": 2048, "d_ff": 14336, "bits": 8,
         "group": 128},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------

_FLOP_CAP = 18.0 * 8192 * 4096 * 11008      # the listed Llama-7B full fine-tune


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dims(rng, most=4096):
    """(d_model, d_ff): a named model's dims, or any multiples of 64 / 128."""
    named = [d for d in ((2048, 5632), (4096, 11008), (4096, 14336), (1024, 2816))
             if d[0] <= most]
    if rng.random() < 0.6:
        return rng.choice(named)
    h = 64 * _log_int(rng, 8, most // 64)
    return h, 128 * max(8, min(112, int(round(h * rng.uniform(2.0, 3.6) / 128))))


def draw(rng):
    kind = rng.choice(["ffn"] * 8 + ["fp32", "fp16", "dora", "topk", "codec"])
    if kind == "codec":
        return {"kind": "codec", "rows": _log_int(rng, 1, 8192), "d_ff": _dims(rng)[1],
                "bits": rng.choice([4, 8]), "group": rng.choice([32, 64, 128])}
    if kind == "topk":
        h, d = _dims(rng, 2048)
        return {"kind": "topk", "batch": 1, "seq": _log_int(rng, 1, 4096), "d_model": h, "d_ff": d,
                "keep": rng.choice([0.1, 0.3, 0.5]), "dtype": "bf16"}
    h, d = _dims(rng, 2048 if kind in ("fp32", "fp16") else 4096)
    train = rng.choice(["none", "full", "adapter", "adapter"])
    adapter = "none" if train == "full" else rng.choice(["lora", "lora", "none"])
    most = 16384
    if kind == "fp32":
        most = 2048
    elif kind == "fp16":
        most = 4096
    elif kind == "dora":
        most, adapter = 4096, "dora"
        train = rng.choice(["none", "adapter"])
    n = _log_int(rng, 1, min(most, int(_FLOP_CAP / (18.0 * h * d))))
    batch = rng.choice([1, 1, 2, 4, 8])
    batch, seq = (batch, n // batch) if n >= 8 * batch else (1, n)
    cache, group = rng.choice([("int4", 64), ("int8", 128), ("int8", 64), ("bf16", 64),
                               ("recompute", 64), ("int4", 32)])
    outl = 0.01 if (kind == "ffn" and cache in ("int4", "int8") and rng.random() < 0.25) else 0.0
    case = _ffn("", batch, seq, h, d, cache, group, train,
                dtype=kind if kind in ("fp32", "fp16") else "bf16", adapter=adapter,
                rank=0 if adapter == "none" else rng.choice([8, 16, 32]), outliers=outl)
    del case["name"]
    return case


# ---------------------------------------------------------------------------
# inputs and one pass
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _normal(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device=_device()) * std).to(dtype)


class _Mlp(nn.Module):
    """A LLaMA-style MLP's projections (its forward is replaced by FlashFFNv3)."""


class _Magnitude(nn.Module):
    """PEFT's DoRA layer: the magnitude vector as `.weight`."""

    def __init__(self, m):
        super().__init__()
        self.weight = nn.Parameter(m)


def _linear(w):
    lin = nn.Linear(1, 1, bias=False, device="meta")
    lin.in_features, lin.out_features = w.shape[1], w.shape[0]
    lin.weight = nn.Parameter(w)
    return lin


def _projection(case, g, w):
    lin = _linear(w)
    if case["adapter"] == "none":
        lin.weight.requires_grad_(case["train"] == "full")
        return lin
    r, dt = case["rank"], w.dtype
    wrap = LoraLinear(lin, r, 2.0 * r)
    bound = 1.0 / math.sqrt(w.shape[1])
    with torch.no_grad():
        a = (torch.rand((r, w.shape[1]), generator=g, device=w.device) * 2 - 1) * bound
        wrap.lora_A["default"].weight.copy_(a.to(dt))
        wrap.lora_B["default"].weight.copy_(_normal(g, (w.shape[0], r), 0.01, dt))
        if case["adapter"] == "dora":
            ba = wrap.lora_B["default"].weight.float() @ wrap.lora_A["default"].weight.float()
            norm = (w.float() + 2.0 * ba).norm(dim=1)
            jitter = torch.randn(w.shape[0], generator=g, device=w.device)
            wrap.lora_magnitude_vector = nn.ModuleDict(
                {"default": _Magnitude((norm * (1 + 0.1 * jitter)).to(dt))})
    return wrap


def _weights(case, g):
    """gate, up and down weights, in the order both prepare and exact draw them."""
    h, d, dt = case["d_model"], case["d_ff"], DTYPES[case["dtype"]]
    return [_normal(g, s, 0.02, dt) for s in ((d, h), (d, h), (h, d))]


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "codec":
        shape = (case["rows"], case["d_ff"])
        # gate and up activations of N(0, 1) inputs and N(0, 0.02) weights
        return {"case": case, "gate": _normal(g, shape, 1.28, torch.bfloat16),
                "up": _normal(g, shape, 1.28, torch.bfloat16),
                "dh": _normal(g, shape, 1.28, torch.bfloat16)}
    h, dt = case["d_model"], DTYPES[case["dtype"]]
    x = _normal(g, (case["batch"], case["seq"], h), 1.0, dt)
    gy = _normal(g, (case["batch"], case["seq"], h), 1.0, dt)
    ws = _weights(case, g)
    if case["kind"] == "topk":
        mlp = cpt.FlashFFN(8, 8, k_fraction=case["keep"]).to(_device())
        for p, w in zip((mlp.gate_proj, mlp.up_proj, mlp.down_proj), ws):
            p.weight = nn.Parameter(w)
    else:
        mlp = _Mlp()
        for name, w in zip(("gate_proj", "up_proj", "down_proj"), ws):
            setattr(mlp, name, _projection(case, g, w))
        mlp = cpt.FlashFFNv3(mlp, case["cache"], case["group"], True, case["outliers"])
    train = case.get("train", "full") != "none"
    names, params = [], []
    if train:
        x.requires_grad_()
        for n, p in mlp.named_parameters():
            if p.requires_grad:
                names.append(n)
                params.append(p)
    return {"case": case, "mlp": mlp, "x": x, "gy": gy, "names": names, "params": params,
            "train": train}


def run(state):
    case = state["case"]
    if case["kind"] == "codec":
        bits, group = case["bits"], case["group"]
        h_mid, qg, sg, qu, su = cpt.triton_silu_mul_quant(state["gate"], state["up"], bits, group)
        dg, du, hm = cpt.triton_dequant_swiglu_backward(state["dh"], qg, sg, qu, su, bits, group,
                                                        want_h_mid=True)
        return {"h_mid": h_mid, "q_gate": qg, "s_gate": sg, "q_up": qu, "s_up": su,
                "grad_gate": dg, "grad_up": du, "h_mid_hat": hm}
    if not state["train"]:
        with torch.no_grad():
            return {"y": state["mlp"](state["x"])}
    y = state["mlp"](state["x"])
    grads = torch.autograd.grad(y, [state["x"]] + state["params"], state["gy"])
    out = {"y": y, "grad_x": grads[0]}
    out.update(zip(state["names"], grads[1:]))
    return out


# ---------------------------------------------------------------------------
# the least work, the tolerances, the values in 64 bits
# ---------------------------------------------------------------------------

def work(case):
    if case["kind"] == "codec":
        el = case["rows"] * case["d_ff"]
        code = case["bits"] / 8.0 + 2.0 / case["group"]
        return {"bytes": el * (3 * 2 + 4 * 2 + 2 * code), "flops": 20.0 * el}
    n, h, d = case["batch"] * case["seq"], case["d_model"], case["d_ff"]
    e = 4 if case["dtype"] == "fp32" else 2
    train = case.get("train", "full")
    flops, nbytes = 6.0 * n * h * d, e * (3.0 * h * d + 2.0 * n * h)
    if train != "none":
        flops += 6.0 * n * h * d
        nbytes += e * 2.0 * n * h
    if train == "full":
        flops += 6.0 * n * h * d
        nbytes += e * 3.0 * h * d
    r = case.get("rank", 0)
    if r:
        thin = 3.0 * (h + d) * r
        flops += 2.0 * n * thin * (1 if train == "none" else 3)
        nbytes += e * thin * (1 if train == "none" else 2)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "codec":
        # the codes are whole numbers of given inputs; the floats one rounding to bf16
        return {"rel": 2e-3, "max": 2e-2, "differ": 0.0}
    if case["kind"] == "topk":
        return {"rel": 1e-2, "max": 0.5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5 if case["cache"] in ("bf16", "recompute") else 3e-4, "max": 0.1}
    return {"rel": 1e-2 if case["cache"] in ("bf16", "recompute", "int8") else 2e-2, "max": 0.5}


def _codes(h, bits, group):
    """(codes, fp16 scales widened) of the per-group absmax codec on h, float32 [N, D]."""
    qmax = 2.0 ** (bits - 1) - 1
    t = h.view(h.shape[0], -1, group)
    scale = (t.abs().amax(-1, keepdim=True) / qmax).to(torch.float16)
    safe = torch.where(scale > 0, scale.float(), torch.ones_like(scale, dtype=torch.float32))
    return (t / safe).round().clamp(-qmax, qmax), scale


def _payload(codes, bits):
    q = codes.reshape(codes.shape[0], -1)
    if bits == 8:
        return q.to(torch.int8)
    q = (q + 8).to(torch.uint8)
    return q[:, 0::2] | (q[:, 1::2] << 4)


def _cached(case, h):
    """What the backward sees of h (float64) through the case's cache."""
    dt = DTYPES[case["dtype"]]
    if case["cache"] not in ("int4", "int8"):
        return h
    hr = h.to(dt)
    k = int(case["d_ff"] * case["outliers"])
    keep = None
    t = hr.float()
    if k:
        rows = case["seq"]
        keep = t[:rows].double().square().sum(0).topk(k).indices
        t = t.clone()
        t[:, keep] = 0
    codes, scale = _codes(t, 4 if case["cache"] == "int4" else 8, case["group"])
    deq = (codes * scale.float()).view_as(t).to(dt).double()
    if k:
        deq[:, keep] = hr[:, keep].double()
    return deq


def _value(v, grad_of):
    """v's value with the gradient of grad_of."""
    return grad_of + (v - grad_of).detach()


def _exact_codec(case, seed):
    s = prepare(case, seed)
    bits, group = case["bits"], case["group"]
    out, deq = {}, []
    for key in ("gate", "up"):
        codes, scale = _codes(s[key].float(), bits, group)
        out["q_" + key], out["s_" + key] = _payload(codes, bits), scale.squeeze(-1)
        deq.append((codes * scale.float()).view_as(s[key]).to(torch.bfloat16).double())
    silu = torch.nn.functional.silu
    g, u = (t.requires_grad_() for t in deq)
    hm = silu(g) * u
    dg, du = torch.autograd.grad(hm, (g, u), s["dh"].double())
    out.update(h_mid=silu(s["gate"].double()) * s["up"].double(), grad_gate=dg, grad_up=du,
               h_mid_hat=hm.detach())
    return out


def exact(case, seed):
    if case["kind"] == "codec":
        return _exact_codec(case, seed)
    s = prepare(case, seed)
    x = s["x"].detach().double().reshape(-1, case["d_model"])
    gy = s["gy"].double().reshape(-1, case["d_model"])
    leaf = {n: p.detach().double().requires_grad_(s["train"] and p.requires_grad)
            for n, p in s["mlp"].named_parameters()}
    x.requires_grad_(s["train"])
    pre = "" if case["kind"] == "topk" else "mlp."

    def factors(proj):
        base = pre + proj
        if base + ".weight" in leaf:
            return leaf[base + ".weight"], None, None, None
        return (leaf[base + ".base_layer.weight"], leaf[base + ".lora_A.default.weight"],
                leaf[base + ".lora_B.default.weight"],
                leaf.get(base + ".lora_magnitude_vector.default.weight"))

    def raw(t, f, thin=None):
        out = t @ f[0].t()
        if f[1] is not None:
            xa = t @ f[1].t()
            out = out + 2.0 * ((xa if thin is None else _value(thin, xa)) @ f[2].t())
        return out

    def column_norm(f):
        return (f[0] + 2.0 * f[2] @ f[1]).norm(dim=1).detach()

    silu = torch.nn.functional.silu
    gate, up, down = (factors(p) for p in ("gate_proj", "up_proj", "down_proj"))
    h, seen = [], []
    for f in (gate, up):
        t = raw(x, f)
        if f[3] is not None:
            c = f[3] / column_norm(f)
            t = c.detach() * t
            v = _cached(case, t.detach())
            # grad_m = sum grad_h * (the cached h) / m
            seen.append(_value(v, t) + (f[3] - f[3].detach()) * (v / f[3].detach()))
        else:
            v = t.detach() if case["kind"] == "topk" else _cached(case, t.detach())
            seen.append(_value(v, t))
        h.append(t.detach())
    h_mid = silu(h[0]) * h[1]
    hat = silu(seen[0]) * seen[1]
    if case["kind"] == "topk":
        k = max(1, int(case["d_ff"] * case["keep"]))
        order = h_mid.to(DTYPES[case["dtype"]]).abs().sort(
            dim=-1, descending=True, stable=True)
        idx = order.indices[:, :k]
        sparse = torch.zeros_like(h_mid).scatter_(-1, idx, h_mid.gather(-1, idx))
        w = down[0]
        y_hat = hat @ w.detach().t() + sparse @ (w - w.detach()).t()
        y = h_mid @ w.detach().t()
    else:
        thin = None if down[1] is None else (h_mid @ down[1].t()).detach()
        y_hat = raw(hat, down, thin)
        y = raw(h_mid, down).detach()
        if down[3] is not None:
            c = down[3] / column_norm(down)
            y_hat, y = c * y_hat, c.detach() * y
    shape = s["x"].shape
    out = {"y": y.detach().view(shape)}
    if s["train"]:
        want = [leaf[n] for n in s["names"]]
        grads = torch.autograd.grad(y_hat, [x] + want, gy)
        out["grad_x"] = grads[0].view(shape)
        out.update(zip(s["names"], grads[1:]))
    return out
