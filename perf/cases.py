"""Performance cases: the work a user of this framework has it do, through its
public entry points, from one decode token to the 4096^3 product.

listed() holds the cases, draw(rng) more of the same ranges; prepare(case,
seed) makes what a program has in hand before the call, run(state) is one
pass, work(case) the bytes and operations no implementation can do without,
tolerance(case) how far another correct implementation at the same precision
may be, and exact(case, seed) the result in 64 bits in plain torch.

Kinds:
  linear    a linear layer's forward with its fused bias and activation:
            1 row (one decode token) to 2048 (a prompt), fp32 and bf16
  train     the same layer in training: forward keeping the pre-activation,
            then the gradients of input, weight and bias
  matmul    rac_matmul, C = A B: the FAST and CORDIC MACs
  softmax   row softmax on the CORDIC exp
  norm_silu RMSNorm of the hidden states, SiLU of the feed-forward's
  rope      the rotation of Q and K
  q8_gemv   the Q8_0 product of decode: 1 to 8 rows
  attention the attention core in training: forward, then dQ, dK, dV
  generate  a decoder with a key/value cache: a prompt, then tokens one by one
"""
import math

import torch

from rac_amd import ext, rac_torch
from rac_amd.decoder import DecoderConfig, PRESETS, RACDecoder

DEV = "cuda"
MODES = {"fast": ext.MODE_FAST, "cordic": ext.MODE_CORDIC}


def listed():
    return [
        # one decode token through a 4096 x 4096 projection, the framework's
        # default MAC: latency and the weights' stream
        dict(name="linear_token", kind="linear", m=1, n=4096, k=4096, act=0, bias=False, mode="fast", iters=24,
             dtype="float32"),
        # a chat prompt through the feed-forward's first layer
        dict(name="linear_prompt", kind="linear", m=128, n=11008, k=4096, act=3, bias=True, mode="fast", iters=24,
             dtype="float32"),
        # a ragged prompt through a bf16 module's feed-forward layer
        dict(name="linear_bf16", kind="linear", m=301, n=5632, k=2048, act=2, bias=True, mode="fast", iters=24,
             dtype="bfloat16"),
        # a training step of a mid-sized layer, odd sizes (1000 rows of an
        # uneven batch)
        dict(name="train_layer", kind="train", m=1000, n=777, k=1531, act=2, mode="fast", iters=24),
        # the CORDIC product of the reference's C API example, 1024^3
        dict(name="matmul_1024", kind="matmul", m=1024, n=1024, k=1024, mode="cordic", iters=16),
        # the headline product
        dict(name="matmul_4096", kind="matmul", m=4096, n=4096, k=4096, mode="cordic", iters=16),
        # attention-sized row softmax
        dict(name="softmax_rows", kind="softmax", rows=4096, cols=4096, iters=16),
        # one layer's norm and activation over a large batch of tokens
        dict(name="norm_silu", kind="norm_silu", rows=16384, d=4096, ff=11008, iters=16),
        # Q and K of a batch of 8 prompts
        dict(name="rope_qk", kind="rope", b=8, h=32, t=4096, d=128),
        # one token through a Q8_0 feed-forward matrix
        dict(name="q8_token", kind="q8_gemv", m=1, n=11008, k=4096),
        # a training step of the attention core, a Llama block's heads
        dict(name="attention_train", kind="attention", b=1, h=32, t=2048, d=128, causal=True),
        # a whole call of the decoder: a prompt of 500, then 32 tokens
        dict(name="generate", kind="generate", d_model=2048, n_heads=32, n_kv_heads=4, d_ff=5632, n_layers=22,
             prompt=500, tokens=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "train", "train", "matmul", "matmul", "softmax", "norm_silu",
                       "rope", "q8_gemv", "attention", "generate"])
    iters = rng.choice([8, 16, 24])
    if kind == "linear":
        mode = rng.choice(["fast", "fast", "cordic"])
        return dict(kind=kind, m=_log(rng, 1, 2048), n=_log(rng, 64, 11008 if mode == "fast" else 4096),
                    k=_log(rng, 64, 4096),
                    act=rng.randrange(4), bias=rng.random() < 0.5, mode=mode, iters=iters,
                    dtype=rng.choice(["float32", "float32", "bfloat16"]))
    if kind == "train":
        return dict(kind=kind, m=_log(rng, 16, 4096), n=_log(rng, 64, 4096), k=_log(rng, 64, 4096),
                    act=rng.randrange(4), mode="fast", iters=iters)
    if kind == "matmul":
        mode = rng.choice(["fast", "cordic"])
        return dict(kind=kind, m=_log(rng, 16, 4096), n=_log(rng, 16, 4096), k=_log(rng, 16, 4096), mode=mode,
                    iters=8 if mode == "cordic" and rng.random() < 0.5 else 16)
    if kind == "softmax":
        return dict(kind=kind, rows=_log(rng, 32, 8192), cols=_log(rng, 64, 8192), iters=iters)
    if kind == "norm_silu":
        return dict(kind=kind, rows=_log(rng, 1, 16384), d=_log(rng, 256, 4096), ff=_log(rng, 512, 11008),
                    iters=iters)
    if kind == "rope":
        return dict(kind=kind, b=rng.randint(1, 8), h=rng.choice([4, 8, 12, 32]), t=_log(rng, 16, 4096),
                    d=rng.choice([32, 64, 80, 128]))
    if kind == "q8_gemv":
        return dict(kind=kind, m=rng.randint(1, 8), n=_log(rng, 256, 32000), k=32 * _log(rng, 8, 344))
    if kind == "attention":
        return dict(kind=kind, b=rng.randint(1, 2), h=rng.choice([4, 8, 12, 16]), t=_log(rng, 64, 2048),
                    d=rng.choice([32, 64, 80, 128]), causal=rng.random() < 0.75)
    preset = PRESETS["tiny"]
    return dict(kind=kind, d_model=preset.d_model, n_heads=preset.n_heads, n_kv_heads=rng.choice([2, 4, 8]),
                d_ff=preset.d_ff, n_layers=preset.n_layers, prompt=_log(rng, 2, 1500), tokens=rng.randint(4, 48))


# ── inputs ───────────────────────────────────────────────────────────────

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(shape, device=DEV, generator=g) * std


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        dt = getattr(torch, case["dtype"])
        x = _randn(g, m, k).to(dt)
        w = _randn(g, n, k, std=k ** -0.5).to(dt)
        b = _randn(g, n, std=0.1).to(dt) if case["bias"] else torch.empty(0, device=DEV, dtype=dt)
        return x, w, b
    if kind == "train":
        m, n, k = case["m"], case["n"], case["k"]
        return (_randn(g, m, k), _randn(g, n, k, std=k ** -0.5), _randn(g, n, std=0.1), _randn(g, m, n))
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return (torch.rand((m, k), device=DEV, generator=g) * 2 - 1,
                torch.rand((k, n), device=DEV, generator=g) * 2 - 1)
    if kind == "softmax":
        return (_randn(g, case["rows"], case["cols"], std=2.0),)
    if kind == "norm_silu":
        return (_randn(g, case["rows"], case["d"]), 1.0 + _randn(g, case["d"], std=0.02),
                _randn(g, case["rows"], case["ff"]))
    if kind == "rope":
        b, h, t, d = case["b"], case["h"], case["t"], case["d"]
        ang = (torch.arange(t, device=DEV, dtype=torch.float64).view(t, 1)
               * 10000.0 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d))
        return (_randn(g, b, h, t, d), _randn(g, b, h, t, d), ang.cos().float(), ang.sin().float())
    if kind == "q8_gemv":
        return _randn(g, case["m"], case["k"]), _randn(g, case["n"], case["k"], std=case["k"] ** -0.5)
    if kind == "attention":
        shape = (case["b"], case["h"], case["t"], case["d"])
        return tuple(_randn(g, *shape) for _ in range(4))
    # generate: every layer's weights, the prompt's and the tokens' vectors
    d, ff = case["d_model"], case["d_ff"]
    kvw = case["n_kv_heads"] * (d // case["n_heads"])
    layers = []
    for _ in range(case["n_layers"]):
        layers.append({"W_q": _randn(g, d, d, std=d ** -0.5), "W_k": _randn(g, kvw, d, std=d ** -0.5),
                       "W_v": _randn(g, kvw, d, std=d ** -0.5), "W_o": _randn(g, d, d, std=d ** -0.5),
                       "W_g": _randn(g, ff, d, std=d ** -0.5), "W_u": _randn(g, ff, d, std=d ** -0.5),
                       "W_d": _randn(g, d, ff, std=ff ** -0.5),
                       "rms_att": 1.0 + _randn(g, d, std=0.02), "rms_ffn": 1.0 + _randn(g, d, std=0.02)})
    return layers, _randn(g, case["prompt"], d), _randn(g, case["tokens"], d)


def prepare(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    st = dict(case=case)
    if kind == "q8_gemv":
        st["inp"] = (inp[0], ext.q8_quantize(inp[1]))
    elif kind == "generate":
        cfg = DecoderConfig(case["d_model"], case["n_heads"], case["n_kv_heads"], case["d_ff"], case["n_layers"])
        dec = RACDecoder(cfg, inp[0], t_max=case["prompt"] + case["tokens"])
        dec.capture()
        st["dec"], st["inp"] = dec, inp[1:]
    elif kind == "attention":
        st["inp"] = tuple(t.requires_grad_() for t in inp[:3]) + (inp[3],)
    else:
        st["inp"] = inp
    return st


def run(state):
    case, inp = state["case"], state["inp"]
    kind = case["kind"]
    if kind == "linear":
        return ext.fused_linear_forward(inp[0], inp[1], inp[2], case["act"], iters=case["iters"],
                                        mode=MODES[case["mode"]])
    if kind == "train":
        x, w, b, go = inp
        kw = dict(iters=case["iters"], mode=MODES[case["mode"]])
        out, pre = ext.fused_linear_forward(x, w, b, case["act"], return_pre=True, **kw)
        return [out] + ext.fused_linear_backward(go, x, w, b, pre, case["act"], True, **kw)
    if kind == "matmul":
        return ext.matmul_forward(inp[0], inp[1], iters=case["iters"], mode=MODES[case["mode"]])
    if kind == "softmax":
        return ext.softmax(inp[0], iters=case["iters"])
    if kind == "norm_silu":
        return ext.rmsnorm(inp[0], inp[1], 1e-6), ext.silu(inp[2], iters=case["iters"])
    if kind == "rope":
        return ext.rope_apply(inp[0], inp[2], inp[3]), ext.rope_apply(inp[1], inp[2], inp[3])
    if kind == "q8_gemv":
        return ext.q8_gemv(inp[0], inp[1])
    if kind == "attention":
        q, k, v, go = inp
        out = rac_torch.rac_attention(q, k, v, None, case["causal"])
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), go)
    dec = state["dec"]
    prompt, tokens = inp
    dec.reset()
    outs = [dec.forward(prompt)]
    for i in range(tokens.size(0)):
        outs.append(dec.step(tokens[i:i + 1]))
    return [torch.cat(outs)] + dec.k_cache + dec.v_cache


# ── what no implementation can do without ────────────────────────────────

def _mac_flops(case):
    """Operations of one MAC: a FAST MAC is one FMA; a CORDIC MAC the
    rotation path, n (x, y) micro-rotations and the projection (2n + 1 FMAs)."""
    return 2 * (2 * case["iters"] + 1) if case["mode"] == "cordic" else 2


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        e = 2 if case["dtype"] == "bfloat16" else 4
        return {"bytes": e * (m * k + n * k + m * n + (n if case["bias"] else 0)), "flops": _mac_flops(case) * m * n * k}
    if kind == "train":
        m, n, k = case["m"], case["n"], case["k"]
        # reads x, w, b, the gradient; writes out, dx, dw, db
        return {"bytes": 4 * (2 * m * k + 2 * n * k + 2 * n + 2 * m * n), "flops": 3 * _mac_flops(case) * m * n * k}
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": _mac_flops(case) * m * n * k}
    if kind == "softmax":
        e = case["rows"] * case["cols"]
        return {"bytes": 8 * e, "flops": (3 * case["iters"] + 6) * e}
    if kind == "norm_silu":
        r, d, ff = case["rows"], case["d"], case["ff"]
        return {"bytes": 8 * r * (d + ff) + 4 * d, "flops": 4 * r * d + (3 * case["iters"] + 8) * r * ff}
    if kind == "rope":
        e = case["b"] * case["h"] * case["t"] * case["d"]
        return {"bytes": 16 * e + 4 * case["t"] * case["d"], "flops": 2 * 3 * e}
    if kind == "q8_gemv":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k // 32 * 34 + 4 * (m * k + m * n), "flops": 2 * m * n * k}
    if kind == "attention":
        z, t, d = case["b"] * case["h"], case["t"], case["d"]
        pairs = z * t * (t + 1) // 2 if case["causal"] else z * t * t
        # reads q, k, v, the gradient; writes out, dq, dk, dv; two products
        # forward, four backward
        return {"bytes": 8 * 4 * z * t * d, "flops": 6 * 2 * pairs * d}
    d, ff, L = case["d_model"], case["d_ff"], case["n_layers"]
    dh = d // case["n_heads"]
    kvw = case["n_kv_heads"] * dh
    p, n = case["prompt"], case["tokens"]
    w = L * (2 * d * d + 2 * kvw * d + 3 * ff * d)
    # the fp32 weights once for the prompt, the Q8_0 weights once per token,
    # each token's keys and values
    cache = sum(2 * 4 * kvw * (p + i + 1) for i in range(n)) * L + 2 * 4 * kvw * p * L
    att = 4 * d * L * (p * (p + 1) // 2 + sum(p + i + 1 for i in range(n)))
    return {"bytes": 4 * w + n * (w // 32 * 34) + cache + 8 * (p + n) * d, "flops": 2 * w * (p + n) + att}


# ── tolerances ───────────────────────────────────────────────────────────

def tolerance(case):
    kind = case["kind"]
    if kind == "linear" and case["dtype"] == "bfloat16":
        # one bf16 rounding of the output: another order of the fp32 sums
        # moves a value in a few hundred across a rounding boundary
        return {"rel": 5e-4, "max": 2.0 ** -6}
    if kind in ("softmax", "norm_silu"):
        # one ulp of a row's maximum or sum; at 8 and 16 steps the CORDIC exp
        # is a step function of its argument with jumps of 2^-shift
        jump = {8: 8e-3, 16: 6e-5, 24: 2e-6}[case["iters"]]
        return {"rel": 1e-6 + 0.05 * jump, "max": 1e-5 + 8 * jump}
    if kind == "rope":
        return {"rel": 5e-7, "max": 4e-6}
    if kind == "q8_gemv":
        return {"rel": 2e-6, "max": 2e-5}
    if kind in ("linear", "train") and case.get("act") == 3:
        jump = {8: 8e-3, 16: 6e-5, 24: 2e-6}[case["iters"]]
        return {"rel": 1e-5 + 0.05 * jump, "max": 1e-4 + 8 * jump}
    if kind == "generate":
        # sums in another order, through every layer
        return {"rel": 1e-4, "max": 2e-3}
    if kind == "attention":
        return {"rel": 2e-5, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-4}


# ── 64 bits, plain torch ─────────────────────────────────────────────────

_KHAT = {8: 1.64673383, 16: 1.64675049, 24: 1.64675049}    # circular gain, as the format states it
_ATAN = [math.atan(2.0 ** -i) for i in range(24)]


def _rotation_gain(n):
    """The rotate-project factor of one CORDIC MAC: n micro-rotations of
    (1, 0) towards angle 0, divided by the stated gain."""
    x, y, ang = 1.0, 0.0, 0.0
    for i in range(n):
        d = 1.0 if ang >= 0.0 else -1.0
        x, y = x - d * y * 2.0 ** -i, y + d * x * 2.0 ** -i
        ang -= d * _ATAN[i]
    return x / _KHAT[n]


def _gain(case):
    return _rotation_gain(case["iters"]) if case["mode"] == "cordic" else 1.0


def _shifts(n):
    out, s, rep = [], 1, 4
    while len(out) < n:
        out.append(s)
        if s == rep:
            out.append(s)
            rep = 3 * rep + 1
        s += 1
    return out[:n]


def _exp64(x, n):
    """e^x by n Walther steps after the reduction x = k ln2 + r."""
    k = torch.trunc(x / math.log(2.0) + torch.copysign(torch.full_like(x, 0.5), x))
    z = x - k * math.log(2.0)
    p = torch.ones_like(x)
    gain = 1.0
    for s in _shifts(n):
        d = torch.copysign(torch.ones_like(z), z)
        p = p + p * d * 2.0 ** -s
        z = z - d * math.atanh(2.0 ** -s)
        gain *= math.sqrt(1.0 - 4.0 ** -s)
    return p / gain * torch.exp2(k)


def _act64(v, act, n):
    if act == 1:
        return v.clamp_min(0.0)
    if act == 2:
        return 0.5 * v * (1.0 + torch.erf(v * math.sqrt(0.5)))
    if act == 3:
        return v / (1.0 + _exp64(-v, n))
    return v


def _dact64(v, act, n):
    if act == 1:
        return (v > 0).double()
    if act == 2:
        return (0.5 * (1.0 + torch.erf(v * math.sqrt(0.5)))
                + v * torch.exp(-0.5 * v * v) / math.sqrt(2.0 * math.pi))
    if act == 3:
        s = 1.0 / (1.0 + _exp64(-v, n))
        return s * (1.0 + v * (1.0 - s))
    return torch.ones_like(v)


def _q8_values(w):
    """The weights that Q8_0 blocks hold, in 64 bits: 32 int8 and one
    truncated fp16 scale, from fp32 arithmetic as the format states it."""
    blk = w.reshape(-1, 32)
    amax = blk.abs().amax(1, keepdim=True)
    d = amax / torch.full_like(amax, 127.0)                  # a division; by a number torch multiplies
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    q = torch.clamp(torch.round(blk * inv), -127, 127)
    h = d.to(torch.float16)
    over = h.float() > d                                     # truncation, not rounding
    h = torch.where(over, (h.view(torch.int16) - 1).view(torch.float16), h)
    return (q.double() * h.double()).reshape(w.shape)


def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _generate64(case, seed):
    layers, prompt, tokens = _inputs(case, seed)
    nh, nkv = case["n_heads"], case["n_kv_heads"]
    d = case["d_model"]
    dh, kvw, p = d // nh, nkv * (d // nh), case["prompt"]
    x = torch.cat([prompt, tokens]).double()
    t = x.size(0)
    # the causal stack is the same function of each position whether the rows
    # come together or one by one; the prompt runs on the fp32 weights, the
    # tokens on their Q8_0 values
    hidden = torch.ones((t, t), device=DEV, dtype=torch.bool).triu(1)

    def lin(h, w):
        if p > 1:
            return torch.cat([h[:p] @ w.double().t(), h[p:] @ _q8_values(w).t()])
        return h @ _q8_values(w).t()

    ks, vs = [], []
    for lw in layers:
        h = _norm64(x, lw["rms_att"].double(), 1e-5)
        q = lin(h, lw["W_q"]).view(t, nh, dh).transpose(0, 1).contiguous()
        ks.append(lin(h, lw["W_k"]).view(t, nkv, dh).transpose(0, 1))
        vs.append(lin(h, lw["W_v"]).view(t, nkv, dh).transpose(0, 1))
        k, v = (c[-1].repeat_interleave(nh // nkv, 0).contiguous() for c in (ks, vs))
        s = torch.bmm(q, k.transpose(1, 2).contiguous()) * dh ** -0.5
        s.masked_fill_(hidden, float("-inf"))
        s = torch.softmax(s, -1)
        x = x + lin(torch.bmm(s, v).transpose(0, 1).reshape(t, d), lw["W_o"])
        h = _norm64(x, lw["rms_ffn"].double(), 1e-5)
        g = lin(h, lw["W_g"])
        x = x + lin(g * torch.sigmoid(g) * lin(h, lw["W_u"]), lw["W_d"])
    return [x] + ks + vs


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        return _generate64(case, seed)
    inp = _inputs(case, seed)
    if kind == "linear":
        x, w, b = (t.double() for t in inp)
        v = _gain(case) * (x @ w.t())
        return _act64(v + b if case["bias"] else v, case["act"], case["iters"])
    if kind == "train":
        x, w, b, go = (t.double() for t in inp)
        v = x @ w.t() + b
        dv = go * _dact64(v, case["act"], case["iters"])
        return [_act64(v, case["act"], case["iters"]), dv @ w, dv.t() @ x, dv.sum(0)]
    if kind == "matmul":
        return _gain(case) * (inp[0].double() @ inp[1].double())
    if kind == "softmax":
        x = inp[0].double()
        e = _exp64(x - x.amax(-1, keepdim=True), case["iters"])
        return e / e.sum(-1, keepdim=True)
    if kind == "norm_silu":
        return _norm64(inp[0].double(), inp[1].double(), 1e-6), _act64(inp[2].double(), 3, case["iters"])
    if kind == "rope":
        c, s = inp[2].double(), inp[3].double()
        outs = []
        for x in inp[:2]:
            a, b = x[..., 0::2].double(), x[..., 1::2].double()
            outs.append(torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2))
        return tuple(outs)
    if kind == "q8_gemv":
        return inp[0].double() @ _q8_values(inp[1]).t()
    q, k, v, go = (t.double().flatten(0, 1) for t in inp)
    n, scale = 24, case["d"] ** -0.5
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) * scale
    if case["causal"]:
        s.masked_fill_(torch.ones(s.shape[-2:], device=DEV, dtype=torch.bool).triu(1), float("-inf"))
    s = s - s.amax(-1, keepdim=True)
    e = torch.where(s > -700.0, _exp64(s.clamp_min(-700.0), n), torch.zeros_like(s))
    p = e / e.sum(-1, keepdim=True)
    del s, e
    dp = torch.bmm(go, v.transpose(1, 2).contiguous())
    ds = p * (dp - (dp * p).sum(-1, keepdim=True))
    pt, dst = p.transpose(1, 2).contiguous(), ds.transpose(1, 2).contiguous()
    shape = (case["b"], case["h"], case["t"], case["d"])
    return tuple(o.view(shape) for o in (torch.bmm(p, v), scale * torch.bmm(ds, k), scale * torch.bmm(dst, q),
                                         torch.bmm(pt, go)))
