"""Performance cases: the work a user of this framework runs, through its public entry points.

Every case is one call on device-resident inputs. A program is prepared once
(`HipDevice.prepare`), as a serving loop does, and a pass runs it with
`Executable.execute_static` on the caller's tensors; the whole-model case drives
`llama.LlamaMachine`, the captured decode step. Sizes are those of the shipped configurations
(Llama-3.2-1B widths: hidden 2048, ffn 8192, 32/8 heads of 64, vocabulary 128256) and of the
tests' ragged shapes, with batch sizes and lengths over the range between them.

Kinds:
  proj     RMSNorm-fused projection (x / rms(x) · g) · W, bf16, W [out, in] or K-major [in, out]
  int4     x · dequant(W)ᵀ, packed 4-bit weights with bf16 scale and zero point per group
  prefill  GQA causal FlashAttention over a prompt, RoPE on Q and K, optional sliding window
  decode   one query token per head against a K/V cache, RoPE on q, prefix mask at `position`
  attn32   single-head causal attention in float32
  llama    one decode step of the whole model over a filled cache (logits, token and caches)
"""
from __future__ import annotations

import math

import torch

from sanic_amd import configs, ir
from sanic_amd.backend import HipDevice
from sanic_amd.llama import LlamaMachine

EPS = 1e-5
THETA = 500000.0

_device = None


def _dev() -> HipDevice:
    """The process's one device handle, as a program opens it."""
    global _device
    if _device is None:
        torch.cuda.init()
        _device = HipDevice(0)
    return _device


# ── the cases ────────────────────────────────────────────────────────────────

def listed():
    return [
        # one token through a projection whose weight is stored K-major: the smallest bf16 call
        {"name": "proj_1_kmajor", "kind": "proj", "m": 1, "k": 2048, "n": 8192, "kmajor": True},
        # a decode batch: eight sequences, one token each, weights as checkpoints store them
        {"name": "proj_8", "kind": "proj", "m": 8, "k": 2048, "n": 8192, "kmajor": False},
        # a short prompt of an odd length through the same layer
        {"name": "proj_200", "kind": "proj", "m": 200, "k": 2048, "n": 8192, "kmajor": False},
        # a prefill chunk: the configuration's GEMM size
        {"name": "proj_512_kmajor", "kind": "proj", "m": 512, "k": 2048, "n": 8192, "kmajor": True},
        # one token through 4-bit weights: the smallest call of all
        {"name": "int4_1", "kind": "int4", "m": 1, "k": 2048, "n": 8192, "g": 64},
        # a decode batch of sixteen through 4-bit weights
        {"name": "int4_16", "kind": "int4", "m": 16, "k": 2048, "n": 8192, "g": 64},
        # a prefill chunk through 4-bit weights
        {"name": "int4_128", "kind": "int4", "m": 128, "k": 2048, "n": 8192, "g": 64},
        # a long prompt, full causal attention
        {"name": "prefill_4096", "kind": "prefill", "s": 4096, "nh": 32, "nkv": 8, "window": 0},
        # a prompt of a length nobody rounded, with a sliding window
        {"name": "prefill_1000_window", "kind": "prefill", "s": 1000, "nh": 32, "nkv": 8, "window": 256},
        # one token's attention over a full 4096-entry cache
        {"name": "decode_4096", "kind": "decode", "cap": 4096, "pos": 4095, "nh": 32, "nkv": 8},
        # the framework's first example, single-head float32 attention, at a longer sequence
        {"name": "attn32_1024", "kind": "attn32", "s": 1024, "d": 64},
        # the headline: one decode step of the whole model at 2048 tokens of context
        {"name": "llama_2048", "kind": "llama", "pos": 2048, "cap": 2080},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "proj", "int4", "int4", "prefill", "prefill", "decode", "attn32"])
    if kind == "proj":
        # hidden and ffn widths are multiples of 64 as a rule, vocabularies and cut shards need not be
        k = 64 * _log(rng, 8, 32) if rng.random() < 0.8 else 8 * _log(rng, 64, 256)
        n = 64 * _log(rng, 8, 128) if rng.random() < 0.7 else _log(rng, 300, 8192)
        return {"kind": kind, "m": _log(rng, 1, 512), "k": k, "n": n, "kmajor": rng.random() < 0.4}
    if kind == "int4":
        g = rng.choice([32, 64, 64, 128])
        n = 64 * _log(rng, 8, 128) if rng.random() < 0.7 else _log(rng, 300, 8192)
        return {"kind": kind, "m": _log(rng, 1, 128), "k": 128 * _log(rng, 4, 16), "n": n, "g": g}
    if kind == "prefill":
        nkv = rng.choice([1, 2, 4, 8])
        # long prompts come in padded buckets; short ones in any length
        s = 128 * _log(rng, 8, 32) if rng.random() < 0.4 else _log(rng, 40, 1000)
        window = 0 if rng.random() < 0.6 else _log(rng, 64, 1024)
        return {"kind": kind, "s": s, "nh": nkv * rng.choice([1, 2, 4]), "nkv": nkv, "window": window}
    if kind == "decode":
        cap = _log(rng, 100, 8192)
        nkv = rng.choice([2, 4, 8])
        return {"kind": kind, "cap": cap, "pos": min(cap - 1, int(cap * rng.uniform(0.3, 1.0))),
                "nh": nkv * rng.choice([1, 4, 8]), "nkv": nkv}
    return {"kind": kind, "s": _log(rng, 32, 1024), "d": rng.choice([32, 64, 64])}


# ── inputs ───────────────────────────────────────────────────────────────────

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    t = torch.empty(shape, device="cuda", dtype=torch.float32)
    return t.normal_(mean, std, generator=g).to(dtype)


def _inputs(case, seed):
    """The case's input tensors by program buffer name, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "proj":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": _normal(g, (m, k)), "g": _normal(g, (k,), 0.02, 1.0),
                "W": _normal(g, (k, n) if case["kmajor"] else (n, k), 0.02)}
    if kind == "int4":
        m, k, n, gr = case["m"], case["k"], case["n"], case["g"]
        s = (torch.rand((n, k // gr), generator=g, device="cuda") * 0.019 + 0.001).to(torch.bfloat16)
        return {"x": _normal(g, (m, k)), "S": s, "Z": (8.0 * s.float()).to(torch.bfloat16),
                "Wq": torch.randint(0, 256, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8)}
    if kind == "prefill":
        s, nh, nkv = case["s"], case["nh"], case["nkv"]
        return {"Q": _normal(g, (nh, s, 64)), "K": _normal(g, (nkv, s, 64)), "V": _normal(g, (nkv, s, 64))}
    if kind == "decode":
        nh, nkv, cap = case["nh"], case["nkv"], case["cap"]
        return {"q": _normal(g, (nh, 64)), "k_cache": _normal(g, (nkv, cap, 64)), "v_cache": _normal(g, (nkv, 64, cap)),
                "position": torch.full((1,), float(case["pos"]), device="cuda")}
    if kind == "attn32":
        shape = (case["s"], case["d"])
        return {name: _normal(g, shape, dtype=torch.float32) for name in ("Q", "K", "V")}
    shape = _llama_shape(case)
    out = {}
    for name, shp in shape.weight_shapes():
        out[name] = _normal(g, shp, 0.02, 1.0) if name.endswith("norm.weight") else _normal(g, shp, 0.02)
    for layer in range(shape.layers):
        # the cache as a prompt left it: rows before `pos` written, the rest zero
        for which, std, shp in (("key", 1.0, (shape.kv_heads, shape.capacity, shape.head_dim)),
                                ("value", 0.5, (shape.kv_heads, shape.head_dim, shape.capacity))):
            t = _normal(g, shp, std)
            if which == "key":
                t[:, case["pos"]:, :] = 0
            else:
                t[:, :, case["pos"]:] = 0
            out[f"cache.{layer}.{which}"] = t
    out["token"] = torch.randint(0, shape.vocab, (1,), generator=g, device="cuda")
    return out


def _llama_shape(case):
    return configs.LlamaShape(capacity=case["cap"])


def _program(case):
    kind = case["kind"]
    if kind == "proj":
        return configs.rmsnorm_projection(M=case["m"], K=case["k"], N=case["n"], eps=EPS, kmajor=case["kmajor"])
    if kind == "int4":
        return configs.int4_matmul(M=case["m"], K=case["k"], N=case["n"], G=case["g"])
    if kind == "prefill":
        return configs.flash_prefill(NH=case["nh"], NKV=case["nkv"], S=case["s"], window=case["window"], theta=THETA)
    if kind == "decode":
        return configs.decode_attention(NH=case["nh"], NKV=case["nkv"], HD=64, cap=case["cap"], theta=THETA)
    return configs.direct_attention(S=case["s"], D=case["d"])


_TORCH = {ir.F32: torch.float32, ir.BF16: torch.bfloat16}


class _DeviceView:
    """A device buffer the framework owns, for torch to view without a copy."""

    def __init__(self, buf, shape, typestr):
        self._keep = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "strides": None,
                                         "data": (buf.device_ptr, False), "version": 2}


def _view(buf, shape, dtype):
    if dtype == torch.bfloat16:
        return torch.as_tensor(_DeviceView(buf, shape, "<i2"), device="cuda").view(torch.bfloat16)
    return torch.as_tensor(_DeviceView(buf, shape, "<f4" if dtype == torch.float32 else "<i4"), device="cuda")


def prepare(case, seed):
    dev = _dev()
    tensors = _inputs(case, seed)
    if case["kind"] == "llama":
        return _prepare_llama(dev, case, tensors)
    prog = _program(case)
    out = prog.buffers[-1]
    tensors[out.name] = torch.empty(out.shape, device="cuda", dtype=_TORCH[out.dtype])
    binds = {name: dev.wrap(t.data_ptr(), t.numel() * t.element_size()) for name, t in tensors.items()}
    torch.cuda.synchronize()
    return {"exe": dev.prepare(prog), "binds": binds, "tensors": tensors, "out": tensors[out.name]}


def _prepare_llama(dev, case, tensors):
    shape = _llama_shape(case)
    names = [name for name, _ in shape.weight_shapes()]
    weights = {n: dev.wrap(tensors[n].data_ptr(), tensors[n].numel() * 2) for n in names}
    torch.cuda.synchronize()
    m = LlamaMachine(dev, weights, shape)
    outs = {"logits": _view(m.logits, (shape.vocab,), torch.float32), "token": _view(m.token, (1,), torch.int32)}
    for layer in range(shape.layers):
        for which in ("key", "value"):
            name = f"cache.{layer}.{which}"
            outs[name] = _view(m.bind[name], m.prog.by_name[name].shape, torch.bfloat16)
            outs[name].copy_(tensors[name])
    token = int(tensors["token"].item())
    torch.cuda.synchronize()
    return {"machine": m, "weights": [tensors[n] for n in names], "token": token, "pos": case["pos"], "outs": outs}


def run(state):
    if "machine" in state:
        m = state["machine"]
        m.set_position(state["pos"])
        m.step(state["token"])
        return state["outs"]
    state["exe"].execute_static(state["binds"])
    return state["out"]


# ── what a pass cannot do without ────────────────────────────────────────────

def _pairs(s, window):
    """Visible (query, key) pairs of one head."""
    if not window or window >= s:
        return s * (s + 1) // 2
    return window * (window + 1) // 2 + (s - window) * window


def work(case):
    kind = case["kind"]
    if kind == "proj":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * (m * k + k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "int4":
        m, k, n, g = case["m"], case["k"], case["n"], case["g"]
        return {"bytes": n * k // 2 + 4 * n * (k // g) + 2 * m * k + 2 * m * n, "flops": 2 * m * k * n}
    if kind == "prefill":
        s, nh, nkv = case["s"], case["nh"], case["nkv"]
        return {"bytes": 2 * 64 * s * (2 * nh + 2 * nkv), "flops": 4 * 64 * nh * _pairs(s, case["window"])}
    if kind == "decode":
        p = case["pos"] + 1
        return {"bytes": 2 * 64 * (2 * case["nkv"] * p + 2 * case["nh"]), "flops": 4 * 64 * case["nh"] * p}
    if kind == "attn32":
        s, d = case["s"], case["d"]
        return {"bytes": 4 * 4 * s * d, "flops": 4 * d * _pairs(s, 0)}
    shape = _llama_shape(case)
    kv = 2 * shape.layers * 2 * shape.kv_heads * shape.head_dim * (case["pos"] + 1)
    # every weight once; of the embedding table the tied head reads every row
    return {"bytes": shape.weight_bytes() + kv + 4 * shape.vocab,
            "flops": shape.weight_bytes() + 4 * shape.layers * shape.heads * shape.head_dim * (case["pos"] + 1)}


def tolerance(case):
    return {
        # bf16 output of 32-bit sums: the store's rounding (2^-9 relative at most)
        "proj": {"rel": 6e-3},
        "int4": {"rel": 6e-3},
        # rotated keys and softmax weights pass through bf16 besides the output
        "prefill": {"rel": 1.2e-2},
        "decode": {"rel": 8e-3},
        # 32-bit throughout
        "attn32": {"rel": 2e-6},
        # 32-bit activations over 16 layers; the step's own K/V rows are stored in bf16
        "llama": {"rel": 8e-4, "differ": 0.01},
    }[case["kind"]]


# ── the same in 64 bits ──────────────────────────────────────────────────────

def _rope64(x, pos, inv):
    """Rotate-half RoPE of x [..., rows, 64] with row i at pos[i]."""
    ang = pos[:, None] * inv[None, :]
    c, s = torch.cos(ang), torch.sin(ang)
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _inv_freq(half):
    i = torch.arange(half, device="cuda", dtype=torch.float64)
    return THETA ** (-i / half)


def _llama3_inv_freq(half):
    """The Llama-3 frequency schedule: factor 32, low/high 1 and 4, original context 8192."""
    inv = _inv_freq(half)
    wavelen = 2 * math.pi / inv
    smooth = (8192.0 / wavelen - 1.0) / 3.0
    mid = (1 - smooth) * inv / 32.0 + smooth * inv
    return torch.where(wavelen > 8192.0, inv / 32.0, torch.where(wavelen < 2048.0, inv, mid))


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    f = torch.float64
    if kind == "proj":
        x, g, w = t["x"].to(f), t["g"].to(f), t["W"].to(f)
        y = (x * g) @ (w if case["kmajor"] else w.t().contiguous())
        return y / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS)
    if kind == "int4":
        n, k, gr = case["n"], case["k"], case["g"]
        q = torch.stack((t["Wq"] & 15, t["Wq"] >> 4), dim=-1).to(f).view(n, k // gr, gr)
        w = (q * t["S"].to(f)[..., None] - t["Z"].to(f)[..., None]).view(n, k)
        return t["x"].to(f) @ w.t().contiguous()
    if kind == "prefill":
        s, nh, nkv, window = case["s"], case["nh"], case["nkv"], case["window"]
        pos = torch.arange(s, device="cuda", dtype=f)
        inv = _inv_freq(32)
        qi, ki = pos[:, None], pos[None, :]
        hidden = ki > qi
        if window:
            hidden = hidden | (ki < qi - (window - 1))
        out = torch.empty((nh, s, 64), device="cuda", dtype=f)
        for h in range(nh):
            q = _rope64(t["Q"][h].to(f), pos, inv)
            k = _rope64(t["K"][h // (nh // nkv)].to(f), pos, inv)
            sc = (q @ k.t().contiguous() / 8.0).masked_fill_(hidden, -math.inf)
            out[h] = torch.softmax(sc, dim=-1) @ t["V"][h // (nh // nkv)].to(f)
        return out
    if kind == "decode":
        nh, nkv, p = case["nh"], case["nkv"], case["pos"] + 1
        q = _rope64(t["q"].to(f)[:, None, :], torch.full((1,), float(case["pos"]), device="cuda", dtype=f), _inv_freq(32))
        q = q.view(nkv, nh // nkv, 64)
        k, v = t["k_cache"][:, :p].to(f), t["v_cache"][:, :, :p].to(f)
        w = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) / 8.0, dim=-1)
        return torch.bmm(w, v.transpose(1, 2).contiguous()).reshape(nh, 64)
    if kind == "attn32":
        q, k, v = (t[n].to(f) for n in ("Q", "K", "V"))
        sc = q @ k.t().contiguous() / math.sqrt(case["d"])
        sc = sc.masked_fill(torch.ones_like(sc, dtype=torch.bool).triu(1), -math.inf)
        return torch.softmax(sc, dim=-1) @ v
    return _exact_llama(case, t)


def _exact_llama(case, t):
    f = torch.float64
    shape, pos = _llama_shape(case), case["pos"]
    nh, nkv, hd = shape.heads, shape.kv_heads, shape.head_dim
    at = torch.full((1,), float(pos), device="cuda", dtype=f)
    inv = _llama3_inv_freq(hd // 2)

    def norm(x, w):
        return x / torch.sqrt((x * x).mean() + EPS) * t[w].to(f)

    x = t["model.embed_tokens.weight"][int(t["token"].item())].to(f)
    out = {}
    for layer in range(shape.layers):
        pre = f"model.layers.{layer}."
        h = norm(x, pre + "input_layernorm.weight")
        q, k, v = (t[pre + f"self_attn.{n}_proj.weight"].to(f) @ h for n in "qkv")
        q = _rope64(q.view(nh, 1, hd), at, inv).view(nkv, nh // nkv, hd)
        kc, vc = t[f"cache.{layer}.key"].to(f), t[f"cache.{layer}.value"].to(f)
        kc[:, pos] = _rope64(k.view(nkv, 1, hd), at, inv)[:, 0]
        vc[:, :, pos] = v.view(nkv, hd)
        out[f"cache.{layer}.key"], out[f"cache.{layer}.value"] = kc, vc
        w = torch.softmax(torch.bmm(q, kc[:, :pos + 1].transpose(1, 2).contiguous()) / math.sqrt(hd), dim=-1)
        o = torch.bmm(w, vc[:, :, :pos + 1].transpose(1, 2).contiguous()).reshape(-1)
        x = x + t[pre + "self_attn.o_proj.weight"].to(f) @ o
        h = norm(x, pre + "post_attention_layernorm.weight")
        gate, up = t[pre + "mlp.gate_proj.weight"].to(f) @ h, t[pre + "mlp.up_proj.weight"].to(f) @ h
        x = x + t[pre + "mlp.down_proj.weight"].to(f) @ (gate * torch.sigmoid(gate) * up)
    out["logits"] = t["model.embed_tokens.weight"].to(f) @ norm(x, "model.norm.weight")
    out["token"] = out["logits"].argmax().view(1).to(torch.int32)
    return out
