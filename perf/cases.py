"""The work a user of libmimg has it do, as cases that can be timed and checked.

A case is a plain dict; `kind` names the public entry point it goes through:

  linear     one quantized linear layer on device buffers: `op` "a8" is
             dequant_matmul_a8 (activations quantized in blocks of `block`),
             "f32" is dequant_matmul (float32 activations), both in the
             reference's float order; "a8_tiled" and "f32_tiled" are the
             matrix-core forms a caller opts into
  layer_set  the seven linears of one decoder layer at one row, inputs
             independent (mimg.linear_a8_set_dev)
  ffn        the feed-forward block of a decoder layer as the decoder calls
             it: norm, gate and up, swiglu, down
  attention  attention over the key-value cache, a prompt or a decode batch
  host       one linear layer on host arrays, the Go shim's call
  generate   greedy generation by a whole decoder: prompt, then one replayed
             step per token

Weights are normal draws with the spread of trained layers, encoded here by
plain range quantizers, so that they can be decoded without the library.
Shapes are the two model shapes of the decode benchmarks (embedding 2048 and
4096, FFN 8192 and 14336, 32 query and 8 key-value heads, vocabulary 128256),
the prompt lengths 19 and 181 of the reference's published runs, and odd
sizes between.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mimir-model_amd"))
# torch and the library share one HIP runtime: the one torch has loaded
os.environ.setdefault("MIMG_HIP_RUNTIME", os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))

import decoder  # noqa: E402
import mimg  # noqa: E402

DT = {"q4_k": mimg.Q4_K, "q6_k": mimg.Q6_K, "q8_0": mimg.Q8_0}
BLOCK = {"q4_k": 256, "q6_k": 256, "q8_0": 32}  # weight elements a block
EPS = 1e-5
STD = 0.02  # spread of the weights


# ---- the cases ---------------------------------------------------------------

def linear(op, dt, n, k, rows, block=256, bias=False):
    return dict(kind="linear", op=op, dt=dt, n=n, k=k, rows=rows, block=block, bias=bias)


def listed():
    return [
        # the key projection of the small model for one token: launches and latency
        dict(linear("a8", "q4_k", 512, 2048, 1), name="k_proj_1row"),
        # one token's linears of a large model's layer: weights streamed once
        dict(kind="layer_set", embed=4096, kv=1024, ffn=14336, name="layer_set_1row"),
        # down projection for a decode batch of eight sequences
        dict(linear("a8", "q6_k", 4096, 14336, 8), name="down_8rows"),
        # gate projection for a short prompt
        dict(linear("a8", "q4_k", 14336, 4096, 64), name="gate_64rows"),
        # gate projection for a long prompt: the largest product
        dict(linear("a8", "q4_k", 14336, 4096, 2048), name="gate_2048rows"),
        # a Q8_0 model's up projection for the reference's 181-token prompt
        # (dequant_matmul_a8.v1 in the reference's order)
        dict(linear("a8", "q8_0", 14336, 4096, 181, block=32), name="up_q8_0_181rows"),
        # float32 activations (dequant_matmul.v1), the small model's down
        # projection for the same prompt
        dict(linear("f32", "q6_k", 2048, 8192, 181), name="down_f32_181rows"),
        # a whole feed-forward block for a 512-token prompt
        dict(kind="ffn", embed=4096, ffn=14336, rows=512, name="ffn_512rows"),
        # prompt attention, 512 tokens into an empty cache
        dict(kind="attention", heads=32, kv_heads=8, d=128, context=768, slots=1, rows=512, f16=True,
             name="attention_prompt_512"),
        # decode attention, eight sequences deep into their contexts
        dict(kind="attention", heads=32, kv_heads=8, d=128, context=2048, slots=8, rows=8, f16=True,
             name="attention_decode_8x2048"),
        # the executor's fast path: pageable host arrays in and out
        dict(kind="host", op="a8", dt="q4_k", n=14336, k=4096, rows=1, block=256, name="host_gate_1row"),
        # the small model end to end: a 32-token prompt and 24 tokens
        dict(kind="generate", layers=16, embed=2048, ffn=8192, heads=32, kv_heads=8, vocab=128256, weights="q4_k_m",
             a8=True, cache_f16=True, slots=1, prompt=32, new=24, name="generate_1b"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _step(v, step, lo):
    return max(lo, v // step * step)


def _linear_sizes(rng, dt, max_rows, flops):
    """Rows and [N, K], K whole blocks of 256; odd N and rows among them."""
    k = _step(_log(rng, 512, 14336), 256, 512)
    n = _log(rng, 256, 16384)
    if rng.random() < 0.7:
        n = _step(n, 64, 256)
    rows = _log(rng, 1, max_rows)
    while 2.0 * rows * n * k > flops:
        rows = max(1, rows // 2)
    return rows, n, k


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["layer_set", "ffn", "attention", "attention", "host", "generate"])
    if kind == "linear":
        op = rng.choice(["a8", "a8", "a8", "a8_b32", "f32", "f32_tiled", "a8_tiled"])
        if op == "a8":
            dt = rng.choice(["q4_k", "q6_k"])
            rows, n, k = _linear_sizes(rng, dt, 2048, 2.4e11)
            return linear("a8", dt, n, k, rows, 256, rng.random() < 0.25)
        dt = rng.choice(["q4_k", "q6_k", "q8_0"])
        rows, n, k = _linear_sizes(rng, dt, 512, 3e10)
        if op == "a8_b32":
            return linear("a8", dt, n, k, rows, 32, rng.random() < 0.25)
        return linear(op, dt, n, k, rows, 32 if op == "a8_tiled" else 256, rng.random() < 0.25)
    if kind == "layer_set":
        e = _step(_log(rng, 512, 8192), 256, 512)
        return dict(kind="layer_set", embed=e, kv=max(64, e // rng.choice([1, 2, 4, 8])),
                    ffn=_step(_log(rng, 1024, 16384), 256, 1024))
    if kind == "ffn":
        return dict(kind="ffn", embed=_step(_log(rng, 512, 4096), 256, 512), ffn=_step(_log(rng, 1024, 14336), 256, 1024),
                    rows=_log(rng, 1, 512))
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        c = dict(kind="attention", heads=kv * rng.choice([1, 2, 4, 8]), kv_heads=kv, d=rng.choice([64, 128]),
                 context=_log(rng, 64, 4096), f16=rng.random() < 0.6)
        if rng.random() < 0.5:
            return dict(c, slots=1, rows=min(_log(rng, 2, 512), c["context"]))
        s = rng.randint(1, 8)
        return dict(c, slots=s, rows=s)
    if kind == "host":
        op = rng.choice(["a8", "a8", "f32"])
        dt = rng.choice(["q4_k", "q6_k", "q8_0"])
        rows, n, k = _linear_sizes(rng, dt, 256, 3e10)
        return dict(kind="host", op=op, dt=dt, n=n, k=k, rows=rows, block=32 if dt == "q8_0" else 256)
    e = rng.choice([1024, 2048])
    slots = rng.choice([1, 1, 2, 3, 4, 6, 8])
    return dict(kind="generate", layers=rng.randint(2, 8), embed=e, ffn=_step(_log(rng, 2048, 8192), 256, 2048),
                heads=e // 64, kv_heads=rng.choice([4, 8]), vocab=_step(_log(rng, 8192, 65536), 64, 8192),
                weights=rng.choice(["q4_k_m", "q4_k_m", "q8_0"]), a8=rng.random() < 0.7, cache_f16=rng.random() < 0.5,
                slots=slots, prompt=_log(rng, 4, 192), new=rng.randint(4, 24))


# ---- block encoders and decoders (spec/dtypes.md:124-246) ----------------------

def _f16_bytes(v):
    return v.half().contiguous().view(torch.uint8).reshape(*v.shape, 2)


def encode(dt, w):
    """float32 [n, k] -> block bytes [n, row bytes], by plain range quantizers."""
    n, k = w.shape
    if dt == "q8_0":
        x = w.reshape(n, k // 32, 32)
        d = (x.abs().amax(-1) / 127).half().float()
        q = torch.round(x / d[..., None].clamp_min(1e-12)).clamp(-127, 127).to(torch.int8)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], -1).reshape(n, -1).contiguous()
    if dt == "q6_k":
        x = w.reshape(n, k // 256, 16, 16)
        s = x.abs().amax(-1) / 31
        d = (s.amax(-1) / 127).half().float()
        sc = torch.round(s / d[..., None].clamp_min(1e-12)).clamp(1, 127)
        q = (torch.round(x / (d[..., None] * sc).clamp_min(1e-12)[..., None]).clamp(-32, 31) + 32).to(torch.uint8)
        q = q.reshape(n, k // 256, 2, 4, 32)
        lo = q & 15
        ql = torch.cat([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], -1)
        hi = q >> 4
        qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
        return torch.cat([ql.reshape(n, -1, 128), qh.reshape(n, -1, 64), sc.to(torch.int8).view(torch.uint8),
                          _f16_bytes(d)], -1).reshape(n, -1).contiguous()
    x = w.reshape(n, k // 256, 8, 32)
    low = x.amin(-1).clamp_max(0)
    s, m = (x.amax(-1) - low) / 15, -low
    d, dmin = (s.amax(-1) / 63).half().float(), (m.amax(-1) / 63).half().float()
    sc = torch.round(s / d[..., None].clamp_min(1e-12)).clamp(1, 63)
    mn = torch.round(m / dmin[..., None].clamp_min(1e-12)).clamp(0, 63)
    q = torch.round((x + (dmin[..., None] * mn)[..., None]) / (d[..., None] * sc).clamp_min(1e-12)[..., None])
    q = q.clamp(0, 15).to(torch.uint8).reshape(n, k // 256, 4, 2, 32)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    scales = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    return torch.cat([_f16_bytes(d), _f16_bytes(dmin), scales, (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(n, -1, 128)],
                     -1).reshape(n, -1).contiguous()


def _f16_at(b):
    return b.contiguous().view(torch.float16).double()[..., 0]


def decode(dt, raw, n, k):
    """Block bytes -> float64 [n, k]."""
    if dt == "q8_0":
        b = raw.reshape(n, k // 32, 34)
        return (_f16_at(b[..., :2])[..., None] * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if dt == "q6_k":
        b = raw.reshape(n, k // 256, 210)
        ql, qh = b[..., :128].reshape(n, -1, 2, 2, 32), b[..., 128:192].reshape(n, -1, 2, 32)
        q = torch.stack([(ql[..., p & 1, :] >> (4 * (p >> 1))) & 15 | ((qh >> (2 * p)) & 3) << 4 for p in range(4)], -2)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        v = (q.double() - 32).reshape(n, k // 256, 16, 16) * sc[..., None]
        return (v * _f16_at(b[..., 208:])[..., None, None]).reshape(n, k)
    b = raw.reshape(n, k // 256, 144)
    s = b[..., 4:16]
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    qs = b[..., 16:].reshape(n, -1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], -2).reshape(n, -1, 8, 32).double()
    d, dmin = _f16_at(b[..., :2])[..., None, None], _f16_at(b[..., 2:4])[..., None, None]
    return (d * sc[..., None] * q - dmin * mn[..., None]).reshape(n, k)


def _row_bytes(dt, k):
    return mimg.row_bytes(DT[dt], k)


class Draws:
    """Seeded values on the GPU; the same calls give the same values."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std)

    def raw(self, dt, n, k):
        return encode(dt, self.normal(n, k, std=STD))

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int64)


def _register(dt, raw, n, k):
    torch.cuda.synchronize()  # the encoded bytes are ready
    return mimg.Weight((raw.data_ptr(), raw.numel()), DT[dt], n, k, device=True)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _workspace(rows, k):
    return _empty(mimg.a8_workspace_bytes(rows, k), dtype=torch.uint8)


# ---- linear --------------------------------------------------------------------

def _linear_inputs(c, seed):
    r = Draws(seed)
    return (r.raw(c["dt"], c["n"], c["k"]), r.normal(c["rows"], c["k"]),
            r.normal(c["n"], std=0.1) if c["bias"] else None)


def _prepare_linear(c, seed):
    raw, x, bias = _linear_inputs(c, seed)
    return dict(c, w=_register(c["dt"], raw, c["n"], c["k"]), x=x, b=bias, y=_empty(c["rows"], c["n"]),
                ws=_workspace(c["rows"], c["k"]))


def _run_linear(s):
    x, y, b, st = s["x"].data_ptr(), s["y"].data_ptr(), s["b"].data_ptr() if s["bias"] else None, s["stream"]
    if s["op"] == "a8":
        mimg.linear_a8_dev(s["w"], x, s["rows"], b, s["block"], y, s["ws"].data_ptr(), s["ws"].numel(), st)
    elif s["op"] == "f32":
        mimg.linear_f32_dev(s["w"], x, s["rows"], b, y, st)
    elif s["op"] == "f32_tiled":
        mimg.linear_f32_mfma_dev(s["w"], x, s["rows"], b, y, st)
    else:
        mimg.quantize_act_dev(x, s["rows"], s["k"], 32, s["ws"].data_ptr(), s["ws"].numel(), st)
        mimg.matmul_a8_quantized_b32_tiled_dev(s["w"], x, s["rows"], b, y, s["ws"].data_ptr(), s["ws"].numel(), st)
    return s["y"]


def _quantized(x, block):
    """The 8-bit activations' values in 64 bits: round(127 x / amax) * amax / 127 a block."""
    b = x.double().reshape(x.shape[0], -1, block)
    amax = b.abs().amax(-1, keepdim=True)
    q = torch.round(b * 127 / amax.clamp_min(1e-300))
    return (q * (amax / 127)).reshape(x.shape)


def _exact_linear(c, seed):
    raw, x, bias = _linear_inputs(c, seed)
    w = decode(c["dt"], raw, c["n"], c["k"])
    y = (x.double() if c["op"].startswith("f32") else _quantized(x, c["block"])) @ w.T
    return y if bias is None else y + bias.double()


# ---- layer_set -------------------------------------------------------------------

def _set_groups(c):
    e, kv, f = c["embed"], c["kv"], c["ffn"]
    return [(e, [("q4_k", e), ("q4_k", kv), ("q6_k", kv)]), (e, [("q4_k", e)]), (e, [("q4_k", f), ("q4_k", f)]),
            (f, [("q6_k", e)])]


def _set_inputs(c, seed):
    r = Draws(seed)
    return [(r.normal(1, k), [(dt, n, r.raw(dt, n, k)) for dt, n in mats]) for k, mats in _set_groups(c)]


def _prepare_set(c, seed):
    groups, xs, ys = [], [], []
    for x, mats in _set_inputs(c, seed):
        ws = [_register(dt, raw, n, x.shape[1]) for dt, n, raw in mats]
        y = [_empty(1, n) for _, n, _ in mats]
        xs.append(x)
        ys += y
        groups.append((ws, x.data_ptr(), None, [t.data_ptr() for t in y]))
    ws = _empty(mimg.linear_a8_set_workspace_bytes(groups), dtype=torch.uint8)
    return dict(c, groups=groups, xs=xs, ys=ys, ws=ws)


def _run_set(s):
    mimg.linear_a8_set_dev(s["groups"], s["ws"].data_ptr(), s["ws"].numel(), s["stream"])
    return s["ys"]


def _exact_set(c, seed):
    return [_quantized(x, 256) @ decode(dt, raw, n, x.shape[1]).T
            for x, mats in _set_inputs(c, seed) for dt, n, raw in mats]


# ---- ffn -------------------------------------------------------------------------

def _ffn_inputs(c, seed):
    r, e, f = Draws(seed), c["embed"], c["ffn"]
    return dict(gate=r.raw("q4_k", f, e), up=r.raw("q4_k", f, e), down=r.raw("q6_k", e, f), x=r.normal(c["rows"], e),
                scale=1 + r.normal(e, std=0.1))


def _prepare_ffn(c, seed):
    i, e, f, t = _ffn_inputs(c, seed), c["embed"], c["ffn"], c["rows"]
    return dict(c, x=i["x"], scale=i["scale"], gate=_register("q4_k", i["gate"], f, e), up=_register("q4_k", i["up"], f, e),
                down=_register("q6_k", i["down"], e, f), h=_empty(t, e), g=_empty(t, f), u=_empty(t, f), sw=_empty(t, f),
                y=_empty(t, e), ws=_workspace(t, max(e, f)))


def _run_ffn(s):
    """The calls of the decoder's feed-forward block (one launch for gate, up
    and swiglu at up to eight rows, separate ones above)."""
    t, e, f, st = s["rows"], s["embed"], s["ffn"], s["stream"]
    ws, nws = s["ws"].data_ptr(), s["ws"].numel()
    h, g, u, sw = (s[k].data_ptr() for k in ("h", "g", "u", "sw"))
    mimg.rms_norm_quant_dev(s["x"].data_ptr(), None, s["scale"].data_ptr(), EPS, t, e, h, 256, ws, nws, st)
    if t <= 8:
        mimg.matmul_a8_quantized_swiglu_dev([s["gate"], s["up"]], h, t, None, 256, sw, 16, ws, nws, st)
        mimg.quantize_act_dev(sw, t, f, 256, ws, nws, st)
    else:
        mimg.matmul_a8_quantized_group_dev([s["gate"], s["up"]], h, t, None, 256, [g, u], ws, nws, st)
        mimg.swiglu_quant_dev(g, u, sw, t, f, 16, 256, ws, nws, st)
    mimg.matmul_a8_quantized_group_dev([s["down"]], sw, t, None, 256, [s["y"].data_ptr()], ws, nws, st)
    return dict(y=s["y"], h=s["h"], sw=s["sw"])


def _exact_ffn(c, seed):
    i, e, f = _ffn_inputs(c, seed), c["embed"], c["ffn"]
    x = i["x"].double()
    h = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * i["scale"].double()
    a = _quantized(h, 256)
    g, u = a @ decode("q4_k", i["gate"], f, e).T, a @ decode("q4_k", i["up"], f, e).T
    sw = g * torch.sigmoid(g) * u
    return dict(y=_quantized(sw, 256) @ decode("q6_k", i["down"], e, f).T, h=h, sw=sw)


# ---- attention ---------------------------------------------------------------------

def _attention_inputs(c, seed):
    r, hk, d, total = Draws(seed), c["kv_heads"], c["d"], c["slots"] * c["context"]
    q = r.normal(c["rows"], c["heads"], d)
    dtype = torch.float16 if c["f16"] else torch.float32
    k, v = r.normal(hk, total, d).to(dtype), r.normal(hk, total, d).to(dtype)
    if c["slots"] == c["rows"] and c["rows"] <= 8:  # a decode batch, a query a slot
        start = torch.arange(c["slots"], device="cuda", dtype=torch.int64) * c["context"]
        end = start + r.ints(3 * c["context"] // 4, c["context"], c["rows"])
    else:  # a prompt from the cache's first entry
        start = torch.zeros(c["rows"], device="cuda", dtype=torch.int64)
        end = torch.arange(c["rows"], device="cuda", dtype=torch.int64)
    return q, k, v, start, end


def _prepare_attention(c, seed):
    q, k, v, start, end = _attention_inputs(c, seed)
    hk, total, d = v.shape
    padded = torch.zeros(hk, mimg.vcache_len(total), d, device="cuda", dtype=v.dtype)
    padded[:, :total] = v
    vb = padded.reshape(hk, -1, 8, d).transpose(2, 3).contiguous()  # blocked by eight keys
    nws = mimg.attention_workspace_bytes(c["rows"], c["heads"], c["context"])
    return dict(c, q=q, k=k, v=vb, start=start, end=end, total=total, out=torch.empty_like(q),
                ws=_empty(max(nws, 16), dtype=torch.uint8))


def _run_attention(s):
    mimg.attention_dev(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["end"].data_ptr(),
                       s["start"].data_ptr() if s["slots"] > 1 else None, s["rows"], s["heads"], s["kv_heads"], s["d"],
                       s["total"], s["context"], s["f16"], s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(),
                       s["stream"])
    return s["out"]


def _exact_attention(c, seed):
    q, k, v, start, end = _attention_inputs(c, seed)
    out = torch.empty(q.shape, device="cuda", dtype=torch.float64)
    at = torch.arange(k.shape[1], device="cuda")
    seen = (at[None, :] >= start[:, None]) & (at[None, :] <= end[:, None])
    for h in range(c["heads"]):
        kv = h // (c["heads"] // c["kv_heads"])
        s = q[:, h].double() @ k[kv].double().T / math.sqrt(c["d"])
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[kv].double()
    return out


# ---- host --------------------------------------------------------------------------

def _prepare_host(c, seed):
    raw, x, _ = _linear_inputs(dict(c, bias=False), seed)
    return dict(c, w=mimg.Weight(raw.cpu().numpy().reshape(-1), DT[c["dt"]], c["n"], c["k"]), x=x.cpu().numpy())


def _run_host(s):
    return mimg.dequant_matmul_a8(s["w"], s["x"], block=s["block"]) if s["op"] == "a8" else mimg.dequant_matmul(s["w"], s["x"])


def _exact_host(c, seed):
    return _exact_linear(dict(c, bias=False), seed).cpu().numpy()


# ---- generate ------------------------------------------------------------------------

def _matrices(c):
    e, f, kv = c["embed"], c["ffn"], c["kv_heads"] * (c["embed"] // c["heads"])
    low, high = ("q4_k", "q6_k") if c["weights"] == "q4_k_m" else ("q8_0", "q8_0")
    out = [("token_embd.weight", low, c["vocab"], e)]
    for l in range(c["layers"]):
        p = f"blk.{l}."
        out += [(p + "attn_q.weight", low, e, e), (p + "attn_k.weight", low, kv, e), (p + "attn_v.weight", high, kv, e),
                (p + "attn_output.weight", low, e, e), (p + "ffn_gate.weight", low, f, e), (p + "ffn_up.weight", low, f, e),
                (p + "ffn_down.weight", high, e, f)]
    return out + [("output.weight", high, c["vocab"], e)]


def _prepare_generate(c, seed):
    r = Draws(seed)
    tensors = {name: (DT[dt], [n, k], _register(dt, r.raw(dt, n, k), n, k)) for name, dt, n, k in _matrices(c)}
    norms = [f"blk.{l}.{n}_norm.weight" for l in range(c["layers"]) for n in ("attn", "ffn")] + ["output_norm.weight"]
    for name in norms:
        tensors[name] = (mimg.F32, [c["embed"]], np.ones(c["embed"], np.float32))
    context = (c["prompt"] + c["new"] + 63) // 64 * 64
    cfg = dict(arch="llama", layers=c["layers"], embed=c["embed"], ffn=c["ffn"], heads=c["heads"], kv_heads=c["kv_heads"],
               rope_theta=500000.0, norm_eps=EPS, context=context)
    dec = decoder.Decoder(cfg, tensors, a8=c["a8"], cache_f16=c["cache_f16"], max_rows=min(512, c["slots"] * c["prompt"]),
                          slots=c["slots"])
    prompts = r.ints(0, c["vocab"], c["slots"], c["prompt"]).cpu().numpy().astype(np.int32)
    return dict(c, dec=dec, prompts=prompts)


def _run_generate(s):
    """The tokens, and the logits of the last step."""
    ids = s["dec"].generate(s["prompts"], s["new"])
    logits = s["dec"].logits.download(np.float32, s["slots"] * s["vocab"]).reshape(s["slots"], s["vocab"])
    return dict(ids=ids, logits=logits)


# ---- the interface ---------------------------------------------------------------------

def prepare(case, seed):
    state = {"linear": _prepare_linear, "layer_set": _prepare_set, "ffn": _prepare_ffn, "attention": _prepare_attention,
             "host": _prepare_host, "generate": _prepare_generate}[case["kind"]](case, seed)
    return dict(state, stream=torch.cuda.current_stream().cuda_stream)


def run(state):
    return {"linear": _run_linear, "layer_set": _run_set, "ffn": _run_ffn, "attention": _run_attention,
            "host": _run_host, "generate": _run_generate}[state["kind"]](state)


def exact(case, seed):
    """64-bit results. None for whole generations with 8-bit activations:
    sixteen layers of rounding decisions that 64 bits take differently."""
    if case["kind"] == "generate":
        return None
    return {"linear": _exact_linear, "layer_set": _exact_set, "ffn": _exact_ffn, "attention": _exact_attention,
            "host": _exact_host}[case["kind"]](case, seed)


def _products(mats, rows):
    """Bytes and operations of products sharing nothing but their inputs."""
    return (sum(n * _row_bytes(dt, k) + 4 * rows * n for dt, n, k in mats), sum(2 * rows * n * k for _, n, k in mats))


def work(case):
    """Weights, inputs and outputs once, and two operations per product."""
    c = case
    if c["kind"] in ("linear", "host"):
        b, f = _products([(c["dt"], c["n"], c["k"])], c["rows"])
        return dict(bytes=b + 4 * c["rows"] * c["k"], flops=f)
    if c["kind"] == "layer_set":
        b, f = _products([(dt, n, k) for k, mats in _set_groups(c) for dt, n in mats], 1)
        return dict(bytes=b + 4 * sum(k for k, _ in _set_groups(c)), flops=f)
    if c["kind"] == "ffn":
        e, n, t = c["embed"], c["ffn"], c["rows"]
        mats = [("q4_k", n, e), ("q4_k", n, e), ("q6_k", e, n)]
        return dict(bytes=sum(m * _row_bytes(dt, k) for dt, m, k in mats) + 4 * t * (3 * e + n), flops=6 * t * e * n)
    if c["kind"] == "attention":
        esz = 2 if c["f16"] else 4
        decode_batch = c["slots"] == c["rows"] and c["rows"] <= 8
        keys = c["slots"] * c["context"] * 7 // 8 if decode_batch else c["rows"]  # read once
        pairs = keys if decode_batch else c["rows"] * (c["rows"] + 1) // 2
        return dict(bytes=2 * c["kv_heads"] * keys * c["d"] * esz + 8 * c["rows"] * c["heads"] * c["d"],
                    flops=4 * pairs * c["heads"] * c["d"])
    per_pass = sum(n * _row_bytes(dt, k) for _, dt, n, k in _matrices(c)[1:])
    head = 2 * c["vocab"] * c["embed"]
    rows = c["slots"] * (c["prompt"] + c["new"] - 1)
    flops = rows * (sum(2 * n * k for _, _, n, k in _matrices(c)[1:]) - head) + c["slots"] * c["new"] * head
    return dict(bytes=c["new"] * per_pass, flops=flops)


def tolerance(case):
    """Float32 sums of 32-bit products: rel about four times the difference to
    the 64-bit results. The ffn's two quantizers round a few of the values on
    a tie the other way; a generation carries such steps through its layers."""
    if case["kind"] == "generate":
        return {"rel": 2e-2, "max": 0.3, "differ": 0.01}
    if case["kind"] == "ffn":
        return {"rel": 1e-3, "max": 5e-2}
    if case["kind"] == "attention":
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 4e-6, "max": 1e-4}
