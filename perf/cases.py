"""Performance cases of the library: what a program that serves the hybrid model has it do.

A case is a dict of plain values. `prepare` makes what such a program holds before the call
(uploaded weights, device buffers, caches, workspaces), `run` is one pass through the public
entry points of `uq` / `uq.layer` / `uq.ops` on the default stream, `work` the bytes and
operations that pass cannot do without, `exact` the same outputs in 64-bit torch arithmetic.

The shapes are those of the synthetic hybrid model that bench.py and the tests run (32 layers,
width 4096, FFN 12288, 16 query heads of 256 over 4 KV heads, 16 / 32 GatedDeltaNet heads of 128,
vocabulary 152064): attention layers' own projections and down projection are Q6_K, the rest
Q4_K. `draw` varies them.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unltd-inference_amd"))

import uq  # noqa: E402
from uq import layer as L  # noqa: E402
from uq import ops as O  # noqa: E402

Q8_0, Q4K, Q6K = int(uq.DType.Q8_0), int(uq.DType.Q4K), int(uq.DType.Q6K)
BLOCK = {Q8_0: (32, 34), Q4K: (256, 144), Q6K: (256, 210)}  # weights and bytes of a block
NAME = {"q4k": Q4K, "q6k": Q6K, "q80": Q8_0}
MODEL = dict(n_embd=4096, n_ff=12288, n_qk_heads=16, n_v_heads=32, head_dim_linear=128, conv_kernel=4,
             n_head=16, n_head_kv=4, head_dim=256, n_rot=64)
EPS = 1e-6


def listed():
    return [
        # one projection of a decoded token, the smallest call a decode loop makes: latency counts
        {"name": "gemv q4k 4096x4096", "kind": "gemv", "q8k": False, "dtype": "q4k", "k": 4096, "n": 4096},
        # the vocabulary head of a decoded token, the largest single weight read of a step
        {"name": "gemv q6k head", "kind": "gemv", "q8k": False, "dtype": "q6k", "k": 4096, "n": 152064},
        # the gated FFN of a decoded token, called as an operator of its own
        {"name": "ffn token", "kind": "ffn", "n": 4096, "ff": 12288, "down": "q6k"},
        # one decoded token through a GatedDeltaNet layer: three layers of four of the model
        {"name": "gdn token", "kind": "gdn_step", "q6k": False, "ff": 12288},
        # one decoded token through a full-attention layer in the middle of a conversation
        {"name": "attn token 3k", "kind": "attn_step", "pos": 3070, "ff": 12288},
        # the attention of one decoded token over a long document
        {"name": "attn decode 24k", "kind": "attn_decode", "ctx": 24001, "heads": 16, "kv": 4, "hd": 256},
        # a decoded token through one period of the model (three GatedDeltaNet layers and one of
        # attention), the final norm and the head: a whole call, logits out
        {"name": "token", "kind": "token", "pos": 511},
        # a prompt of 512 tokens through a GatedDeltaNet layer
        {"name": "gdn prefill 512", "kind": "gdn_prefill", "tokens": 512, "ff": 12288},
        # the last chunk of a prompt of 4k tokens through an attention layer
        {"name": "attn prefill 4k", "kind": "attn_prefill", "tokens": 509, "pos0": 3587, "ff": 12288},
        # a short prompt's down projection in the forward's own numerics: few rows, a ragged count
        {"name": "gemm_q8k q6k 77", "kind": "gemm", "q8k": True, "dtype": "q6k", "k": 12288, "n": 4096, "m": 77},
        # a prompt of 512 tokens through the FFN's gate projection with plain dequantized weights
        {"name": "gemm q4k 512", "kind": "gemm", "q8k": False, "dtype": "q4k", "k": 4096, "n": 12288, "m": 512},
        # a handful of sequences decoded together: a batch of 8, Q8_0, odd columns
        {"name": "gemm q80 8", "kind": "gemm", "q8k": False, "dtype": "q80", "k": 4096, "n": 5003, "m": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges, no larger than the largest listed one of its kind."""
    kind = rng.choice(["gemv", "gemv", "ffn", "gdn_step", "attn_step", "attn_decode", "token", "gdn_prefill",
                       "attn_prefill", "gemm", "gemm", "gemm"])
    if kind == "gemv":
        q8k = rng.random() < 0.5
        k = 256 * _log(rng, 1, 48)
        return {"kind": kind, "q8k": q8k, "dtype": rng.choice(["q4k", "q6k"] if q8k else ["q4k", "q6k", "q80"]), "k": k,
                "n": _log(rng, 1024, 152064 * 4096 // max(k, 4096))}
    if kind == "ffn":
        return {"kind": kind, "n": 256 * rng.randint(4, 16), "ff": 256 * rng.randint(8, 48), "down": rng.choice(["q4k", "q6k"])}
    if kind == "gdn_step":
        return {"kind": kind, "q6k": rng.random() < 0.3, "ff": 256 * rng.randint(16, 48)}
    if kind == "attn_step":
        return {"kind": kind, "pos": _log(rng, 1, 16384), "ff": 256 * rng.randint(16, 48)}
    if kind == "attn_decode":
        hd = rng.choice([64, 128, 256])
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "ctx": _log(rng, 64, 24000 * 1024 // max(hd * kv, 1024)), "heads": kv * rng.choice([1, 2, 4, 6]), "kv": kv, "hd": hd}
    if kind == "token":
        return {"kind": kind, "pos": _log(rng, 1, 4096)}
    if kind == "gdn_prefill":
        return {"kind": kind, "tokens": _log(rng, 2, 512), "ff": 256 * rng.randint(16, 48)}
    if kind == "attn_prefill":
        return {"kind": kind, "tokens": _log(rng, 2, 509), "pos0": _log(rng, 1, 3587) - 1, "ff": 256 * rng.randint(16, 48)}
    q8k = rng.random() < 0.6
    return {"kind": kind, "q8k": q8k, "dtype": rng.choice(["q4k", "q6k"] if q8k else ["q4k", "q6k", "q80"]),
            "k": 256 * rng.randint(4, 16), "n": _log(rng, 512, 12288), "m": _log(rng, 2, 512)}


# ---------------------------------------------------------------------- inputs
class Buf:
    """A torch tensor where the binding takes a device array."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, ctypes.c_void_p(t.data_ptr()), t.numel() * t.element_size()


class Inputs:
    """Seeded inputs: weights as GGUF blocks, normal activations, norm weights near one."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda")

    def norm(self, n):
        return 1.0 + 0.1 * self.normal(n)

    def blocks(self, dtype, k, n):
        """n rows of k weights: uniform quants and scales, f16 block scales |N(0, sigma)|."""
        per, size = BLOCK[dtype]
        nb = n * (k // per)
        b = torch.randint(0, 256, (nb, size), generator=self.g, device="cuda", dtype=torch.uint8)

        def f16(sigma):
            return (self.normal(nb).abs() * sigma).half().view(torch.uint8).view(nb, 2)

        if dtype == Q4K:
            b[:, 0:2], b[:, 2:4] = f16(2e-3), f16(2e-3)
        elif dtype == Q6K:
            b[:, 192:208] = torch.randint(-64, 64, (nb, 16), generator=self.g, device="cuda", dtype=torch.int8).view(torch.uint8)
            b[:, 208:210] = f16(1e-3)
        else:
            b[:, 0:2] = f16(5e-3)
        return b

    def weights(self, dtype, k, n):
        """(uploaded handle, the blocks of n rows of k weights)"""
        b = self.blocks(dtype, k, n)
        return uq.Weights(b.cpu().numpy(), dtype, k, n), b


def dims(case):
    m = dict(MODEL, n_ff=case.get("ff", MODEL["n_ff"]))
    theta = float(np.float32(1.0e7) ** np.float32(-2.0 / m["n_rot"]))
    return L.Dims(**m, theta_scale=theta, kq_scale=1.0 / math.sqrt(m["head_dim"]), rms_eps=EPS)


def gdn_shapes(d, q6k=False):
    t, nv = Q6K if q6k else Q4K, d.n_v_heads * d.head_dim_linear
    return [("attn_qkv", t, d.n_embd, d.channels), ("attn_gate", t, d.n_embd, nv), ("ssm_beta", t, d.n_embd, d.n_v_heads),
            ("ssm_alpha", t, d.n_embd, d.n_v_heads), ("ssm_out", t, nv, d.n_embd), ("ffn_gate", Q4K, d.n_embd, d.n_ff),
            ("ffn_up", Q4K, d.n_embd, d.n_ff), ("ffn_down", t, d.n_ff, d.n_embd)]


def attn_shapes(d):
    q, kv = d.n_head * d.head_dim, d.n_head_kv * d.head_dim
    return [("attn_q", Q6K, d.n_embd, 2 * q), ("attn_k", Q6K, d.n_embd, kv), ("attn_v", Q6K, d.n_embd, kv),
            ("attn_output", Q6K, q, d.n_embd), ("ffn_gate", Q4K, d.n_embd, d.n_ff), ("ffn_up", Q4K, d.n_embd, d.n_ff),
            ("ffn_down", Q6K, d.n_ff, d.n_embd)]


def layer(inp, d, kind, q6k=False):
    """(weights as the layer takes them, {name: tensor} of the same)"""
    raw, w = {}, {}
    for name, t, k, n in gdn_shapes(d, q6k) if kind == "gdn" else attn_shapes(d):
        w[name], b = inp.weights(t, k, n)
        raw[name] = (t, k, b)
    if kind == "gdn":
        vec = dict(attn_norm=inp.norm(d.n_embd), ssm_dt_bias=inp.normal(d.n_v_heads), ssm_a=-torch.exp(0.5 * inp.normal(d.n_v_heads)),
                   ssm_conv1d=0.3 * inp.normal(d.channels, d.conv_kernel), ssm_norm=inp.norm(d.head_dim_linear),
                   post_attention_norm=inp.norm(d.n_embd))
    else:
        vec = dict(attn_norm=inp.norm(d.n_embd), attn_q_norm=inp.norm(d.head_dim), attn_k_norm=inp.norm(d.head_dim),
                   post_attention_norm=inp.norm(d.n_embd))
    raw.update(vec)
    return (L.GdnWeights if kind == "gdn" else L.AttnWeights)(**w, **{k: Buf(v) for k, v in vec.items()}), raw


def gdn_state(inp, d):
    """A conv window and recurrent state as earlier tokens of a conversation leave them."""
    return 0.5 * inp.normal(d.conv_kernel, d.channels), 0.1 * inp.normal(d.n_v_heads, d.head_dim_linear, d.head_dim_linear)


def empty(*shape):
    return Buf(torch.empty(*shape, device="cuda"))


def prepare(case, seed, outputs_only=False):
    """The state of a pass. outputs_only: for `exact`, the inputs and no workspace."""
    inp, kind, s = Inputs(seed), case["kind"], {"kind": case["kind"], "case": case}
    if kind in ("gemv", "gemm"):
        t, m = NAME[case["dtype"]], case.get("m", 1)
        s["w"], b = inp.weights(t, case["k"], case["n"])
        s["raw"], s["x"], s["y"] = (t, case["k"], b if outputs_only else None), Buf(inp.normal(m, case["k"])), empty(m, case["n"])
        s["m"] = m
    elif kind == "ffn":
        n, ff = case["n"], case["ff"]
        shapes = [(Q4K, n, ff), (Q4K, n, ff), (NAME[case["down"]], ff, n)]
        both = [inp.weights(*sh) for sh in shapes]
        s["w"], s["raw"] = [h for h, _ in both], [(sh[0], sh[1], b) for sh, (_, b) in zip(shapes, both)] if outputs_only else None
        s["x"], s["out"] = Buf(inp.normal(n)), [empty(ff), empty(ff), empty(ff), empty(n)]
    elif kind == "attn_decode":
        c, q, kv = case, case["heads"] * case["hd"], case["kv"] * case["hd"]
        s["q"], s["k"], s["v"] = Buf(inp.normal(q)), Buf(inp.normal(c["ctx"], kv)), Buf(inp.normal(c["ctx"], kv))
        s["out"], s["soft"] = empty(q), empty(c["heads"], c["ctx"])
    else:
        d = s["d"] = dims(case)
        kinds = {"token": ["gdn", "gdn", "gdn", "attn"]}.get(kind, [kind.split("_")[0]])
        t = s["t"] = case.get("tokens", 1)
        s["pos0"] = case.get("pos0", case.get("pos", 0))
        s["ctx"] = s["pos0"] + t + 1
        s["layers"] = []
        for k in kinds:
            w, raw = layer(inp, d, k, case.get("q6k", False))
            kv = d.n_head_kv * d.head_dim
            a, b = gdn_state(inp, d) if k == "gdn" else (inp.normal(s["ctx"], kv), inp.normal(s["ctx"], kv))
            s["layers"].append((k, w, Buf(a), Buf(b), empty(t, d.n_embd)))
            if outputs_only:
                s.setdefault("raw", []).append(raw)
        if kind == "token":
            s["norm"] = Buf(inp.norm(d.n_embd))
            s["head"], b = inp.weights(Q6K, d.n_embd, 152064)
            s["head_raw"] = (Q6K, d.n_embd, b) if outputs_only else None
            s["xn"], s["logits"] = empty(d.n_embd), empty(152064)
        s["x"] = Buf(inp.normal(t, d.n_embd))
        ctx = s["ctx"] if "attn" in kinds else 0
        if not outputs_only:
            if kind.endswith("prefill"):
                s["ws"] = empty(L.prefill_ws_floats(d, t, n_ctx_max=ctx, **{kinds[0]: s["layers"][0][1]}))
            else:
                s["ws"] = empty(L.ws_floats(d, ctx))
    return s


# ---------------------------------------------------------------------- one pass
def run(s):
    kind, c = s["kind"], s["case"]
    if kind == "gemv":
        (uq.gemv_q8k if c["q8k"] else uq.gemv)(s["w"], s["x"], s["y"])
        return s["y"].t
    if kind == "gemm":
        (uq.gemm_q8k if c["q8k"] else uq.gemm)(s["w"], s["m"], s["x"], s["y"])
        return s["y"].t
    if kind == "ffn":
        uq.ffn_swiglu_q8k(*s["w"], s["x"], *s["out"])
        return [o.t for o in s["out"]]
    if kind == "attn_decode":
        O.attn_decode_d(s["out"], s["soft"], s["q"], s["k"], s["v"], c["ctx"], c["heads"], c["kv"], c["hd"], 1.0 / math.sqrt(c["hd"]))
        return [s["out"].t, s["soft"].t]
    d, x, ws = s["d"], s["x"], s["ws"]
    for k, w, a, b, y in s["layers"]:
        if kind == "gdn_prefill":
            L.gdn_prefill(d, w, a, b, s["t"], x, y, ws)
        elif kind == "attn_prefill":
            L.attn_prefill(d, w, a, b, s["ctx"], s["pos0"], s["t"], x, y, ws)
        elif k == "gdn":
            L.gdn_step(d, w, a, b, x, y, ws)
        else:
            L.attn_step(d, w, a, b, s["ctx"], s["pos0"], x, y, ws)
        x = y
    out = [x.t] + [v.t for _, _, a, b, _ in s["layers"] for v in (a, b)]
    if kind == "token":
        O.rmsnorm_d(s["xn"], x, s["norm"], d.n_embd, 1, EPS)
        uq.gemv_q8k(s["head"], s["xn"], s["logits"])
        out.append(s["logits"].t)
    return out


# ---------------------------------------------------------------------- work
def _size(t, k, n):
    return n * (k // BLOCK[t][0]) * BLOCK[t][1]


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        k, n, m = case["k"], case["n"], case.get("m", 1)
        return {"bytes": _size(NAME[case["dtype"]], k, n) + 4 * m * (k + n), "flops": 2 * m * k * n}
    if kind == "ffn":
        n, ff = case["n"], case["ff"]
        return {"bytes": 2 * _size(Q4K, n, ff) + _size(NAME[case["down"]], ff, n) + 4 * (2 * n + 3 * ff), "flops": 6 * n * ff}
    if kind == "attn_decode":
        kv, q = case["kv"] * case["hd"], case["heads"] * case["hd"]
        return {"bytes": 4 * (case["ctx"] * (2 * kv + case["heads"]) + 2 * q), "flops": 4 * case["ctx"] * q}
    d, t = dims(case), case.get("tokens", 1)
    pos0 = case.get("pos0", case.get("pos", 0))
    kinds = ["gdn", "gdn", "gdn", "attn"] if kind == "token" else [kind.split("_")[0]]
    b = f = 0
    for k in kinds:
        sh = gdn_shapes(d, case.get("q6k", False)) if k == "gdn" else attn_shapes(d)
        b += sum(_size(*x[1:]) for x in sh) + 8 * t * d.n_embd
        f += sum(2 * t * x[2] * x[3] for x in sh)
        if k == "gdn":  # state and window read and written
            st = d.n_v_heads * d.head_dim_linear ** 2
            b += 8 * (st + d.conv_kernel * d.channels)
            f += 7 * t * st
        else:  # the cache rows seen, those written; causal products
            kv, q = d.n_head_kv * d.head_dim, d.n_head * d.head_dim
            b += 8 * kv * (pos0 + 2 * t)
            f += 4 * q * (t * pos0 + t * (t + 1) // 2)
    if kind == "token":
        b += _size(Q6K, d.n_embd, 152064) + 4 * (3 * d.n_embd + 152064)
        f += 2 * d.n_embd * 152064
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        if case["q8k"]:
            return "exact"  # gemv_quant_q8k bit for bit, whatever the route
        return {"rel": 8e-7, "max": 2e-5}  # f32 results of 64-bit (gemm: matrix core) sums, 2e-7 off exact
    if kind == "attn_decode":
        return {"rel": 5e-7, "max": 1e-5}  # f32 weights and results, 1.3e-7 off exact
    # a layer quantizes what it computes to Q8_K: where another rounding flips one quant on the way, the FFN, whose
    # hidden values reach thousands, carries that to 2e-2 of that token's output (measured against exact: 1e-7 with
    # no flip, 1e-2 over a long prompt's tokens)
    return {"rel": 3e-2, "max": 0.5}


# ---------------------------------------------------------------------- in 64 bits
def _f16(b):
    return b.contiguous().view(torch.float16).double().squeeze(-1)


def dequant(t, k, b):
    """The blocks b as [rows][k] weights in f64."""
    nb = b.shape[0]
    if t == Q8_0:
        w = _f16(b[:, 0:2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == Q4K:
        sc = b[:, 4:16].to(torch.int32)
        lo, hi, top = sc[:, 0:4], sc[:, 4:8], sc[:, 8:12]
        scale = torch.cat([lo & 63, (top & 15) | (lo >> 6 << 4)], 1).double()
        least = torch.cat([hi & 63, (top >> 4) | (hi >> 6 << 4)], 1).double()
        q = b[:, 16:].view(nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(nb, 8, 32).double()
        w = (_f16(b[:, 0:2])[:, None] * scale)[..., None] * q - (_f16(b[:, 2:4])[:, None] * least)[..., None]
    else:
        ql, qh = b[:, 0:128].view(nb, 2, 64), b[:, 128:192].view(nb, 2, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        low = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 2)
        high = torch.stack([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, qh >> 6], 2)
        q = (low | (high << 4)).to(torch.int32).double() - 32.0
        w = (_f16(b[:, 208:210])[:, None] * sc).repeat_interleave(16, 1) * q.reshape(nb, 256)
    return w.reshape(-1, k)


def q8k(x):
    """x after Q8_K quantization (the activations' own rounding), in f64."""
    v = x.double().reshape(*x.shape[:-1], -1, 256)
    top = v.gather(-1, v.abs().argmax(-1, keepdim=True))
    scale = torch.where(top == 0, torch.zeros_like(top), -127.0 / torch.where(top == 0, torch.ones_like(top), top))
    q = torch.clamp(torch.round(scale * v), max=127.0)
    return torch.where(scale == 0, torch.zeros_like(q), q / torch.where(scale == 0, torch.ones_like(scale), scale)).reshape(x.shape).double()


def product(raw, x, quantized=True):
    """x [m][k] times the weights' rows, in f64; quantized: x through Q8_K first."""
    t, k, b = raw
    x = q8k(x) if quantized else x.double()
    rows = (1 << 26) // k
    nb = k // BLOCK[t][0]
    return torch.cat([x @ dequant(t, k, b[r * nb:(r + rows) * nb]).T for r in range(0, b.shape[0] // nb, rows)], -1)


def rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def silu(x):
    return x * torch.sigmoid(x)


def attend(q, k, v, pos0, group, scale):
    """q [t][heads][hd] over k, v [n][kv][hd], token i seeing pos0 + i + 1 rows: (out, weights)"""
    t, n = q.shape[0], k.shape[0]
    hide = torch.arange(n, device="cuda")[None, :] > pos0 + torch.arange(t, device="cuda")[:, None]
    out, soft = [], []
    for h in range(q.shape[1]):
        sc = (q[:, h] @ k[:, h // group].double().T * scale).masked_fill(hide, -math.inf)
        p = torch.softmax(sc, -1)
        out.append(p @ v[:, h // group].double())
        soft.append(p if t == 1 else None)
    return torch.stack(out, 1), torch.cat(soft, 0) if t == 1 else None


def imrope(x, d, pos):
    """every third pair of the first n_rot values turned by pos * theta^i"""
    half = d.n_rot // 2
    i = torch.arange(0, half, 3, device="cuda")
    ang = pos.double()[:, None, None] * d.theta_scale ** i.double()
    a, b, y = x[..., i], x[..., i + half], x.clone()
    y[..., i], y[..., i + half] = torch.cos(ang) * a - torch.sin(ang) * b, torch.sin(ang) * a + torch.cos(ang) * b
    return y


def ffn_exact(raw, res):
    p = rms(res, raw["post_attention_norm"])
    return res + product(raw["ffn_down"], silu(product(raw["ffn_gate"], p)) * product(raw["ffn_up"], p))


def gdn_exact(d, raw, win, state, x):
    t, hd, nv, nq, ck = x.shape[0], d.head_dim_linear, d.n_v_heads, d.n_qk_heads, d.conv_kernel
    xn = rms(x, raw["attn_norm"])
    qkv, z, beta, alpha = (product(raw[k], xn) for k in ("attn_qkv", "attn_gate", "ssm_beta", "ssm_alpha"))
    beta = torch.sigmoid(beta)
    decay = torch.exp(torch.nn.functional.softplus(alpha + raw["ssm_dt_bias"].double(), threshold=60.0) * raw["ssm_a"].double())
    seq = torch.cat([win[:ck - 1].double(), qkv])
    mix = silu(sum(seq[r:r + t] * raw["ssm_conv1d"][:, r].double() for r in range(ck)))
    q, k = (mix[:, i * nq * hd:(i + 1) * nq * hd].view(t, nq, hd) for i in (0, 1))
    q, k = (y / torch.sqrt((y * y).sum(-1, keepdim=True)).clamp(min=EPS) for y in (q, k))
    q, k, v = q.repeat(1, nv // nq, 1), k.repeat(1, nv // nq, 1), mix[:, 2 * nq * hd:].view(t, nv, hd)
    s, out = state.double(), []
    for i in range(t):
        s = s * decay[i][:, None, None]
        delta = (v[i] - (s * k[i][:, :, None]).sum(1)) * beta[i][:, None]
        s = s + k[i][:, :, None] * delta[:, None, :]
        out.append((s * q[i][:, :, None]).sum(1) / math.sqrt(hd))
    y = rms(torch.stack(out), raw["ssm_norm"]).reshape(t, -1) * silu(z)
    return ffn_exact(raw, x + product(raw["ssm_out"], y)), torch.cat([seq[t:], seq[-1:]]), s


def attn_exact(d, raw, kc, vc, pos0, x):
    t, hd, nh, nkv = x.shape[0], d.head_dim, d.n_head, d.n_head_kv
    pos = pos0 + torch.arange(t, device="cuda")
    xn = rms(x, raw["attn_norm"])
    qf = product(raw["attn_q"], xn).view(t, nh, 2, hd)
    q = imrope(rms(qf[:, :, 0], raw["attn_q_norm"]), d, pos)
    kc, vc = kc.double().view(-1, nkv, hd).clone(), vc.double().view(-1, nkv, hd).clone()
    kc[pos] = imrope(rms(product(raw["attn_k"], xn).view(t, nkv, hd), raw["attn_k_norm"]), d, pos)
    vc[pos] = product(raw["attn_v"], xn).view(t, nkv, hd)
    a, _ = attend(q, kc[:pos0 + t], vc[:pos0 + t], pos0, nh // nkv, d.kq_scale)
    y = (a * torch.sigmoid(qf[:, :, 1])).reshape(t, -1)
    return ffn_exact(raw, x + product(raw["attn_output"], y)), kc.view(kc.shape[0], -1), vc.view(vc.shape[0], -1)


def exact(case, seed):
    s, kind = prepare(case, seed, outputs_only=True), case["kind"]
    if kind in ("gemv", "gemm"):
        return product(s["raw"], s["x"].t, case["q8k"])
    if kind == "ffn":
        g, u = (product(r, s["x"].t[None])[0] for r in s["raw"][:2])
        h = silu(g) * u
        return [g, u, h, product(s["raw"][2], h[None])[0]]
    if kind == "attn_decode":
        c = case
        kv = (-1, c["kv"], c["hd"])
        out, soft = attend(s["q"].t.double().view(1, c["heads"], c["hd"]), s["k"].t.view(kv), s["v"].t.view(kv), c["ctx"] - 1,
                           c["heads"] // c["kv"], 1.0 / math.sqrt(c["hd"]))
        return [out.reshape(-1), soft]
    d, x, states = s["d"], s["x"].t.double(), []
    for (k, _, a, b, _), raw in zip(s["layers"], s["raw"]):
        x, *after = gdn_exact(d, raw, a.t, b.t, x) if k == "gdn" else attn_exact(d, raw, a.t, b.t, s["pos0"], x)
        states += after
    if kind == "token":
        return [x] + states + [product(s["head_raw"], rms(x, s["norm"].t))[0]]
    return [x] + states
