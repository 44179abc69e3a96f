"""The work that programs hand to this library, as cases to be timed.

Three kinds of case, each through a public entry point:

- ``linear``: one quantized projection y = x W^T on device buffers
  (``QLinear.forward_dev``).  One row is a decode step's matvec, a handful of
  rows a batch of sequences or a speculative verify, hundreds of rows a
  prompt.
- ``sample``: one token drawn from a row of logits (``syn_hip_sample``).
- ``lm``: a conversation turn of one of the four decoders at its real layer
  widths and a few layers: a prompt, then decode steps on given tokens; the
  logits of the prompt's end and of every step come back.

The weights, prompts and activations of a case follow from its seed alone.
``exact`` restates each case in plain torch, in float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from synapse_amd import hip

FMT = {"int8": hip.FMT_INT8, "q4_0": hip.FMT_Q4_0, "q8_0": hip.FMT_Q8_0,
       "q4_k": hip.FMT_Q4_K, "q6_k": hip.FMT_Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}

# layer widths of the decoders (Qwen3-0.6B, LLaMA-3.2-3B, LFM2.5-350M,
# Mamba-370M); a case gives the number of layers and the vocabulary
LAYER = {
    "int8": dict(hidden=1024, n_heads=16, n_kv_heads=8, head_dim=128, inter=3072, eps=1e-6,
                 rope_theta=1e6),
    "kquant": dict(hidden=3072, n_heads=24, n_kv_heads=8, head_dim=128, inter=8192, eps=1e-5,
                   rope_theta=5e5),
    "hybrid": dict(hidden=1024, n_heads=16, n_kv_heads=8, head_dim=64, inner=1024, conv_kernel=3,
                   inter=6656, eps=1e-5, rope_theta=1e6),
    "mamba": dict(d_model=1024, d_inner=2048, d_state=16, d_conv=4, dt_rank=64, eps=1e-5),
}
STD = 0.03  # of the decoders' synthetic weights: about 1/sqrt(hidden)


def listed():
    lin = lambda name, fmt, m, k, n: dict(name=name, kind="linear", fmt=fmt, m=m, k=k, n=n)
    return [
        # the smallest matvec of a Qwen3-0.6B decode step (attention q): launch latency
        lin("int8_decode", "int8", 1, 1024, 1024),
        # a 512-token prompt through a Mistral-7B gate projection, W8A8
        lin("int8_prefill", "int8", 512, 4096, 14336),
        # LLaMA-3.2-1B gate/up at batch 1
        lin("q4_0_decode", "q4_0", 1, 2048, 8192),
        # a prompt of no round length through LLaMA-3.2-1B down
        lin("q4_0_prompt", "q4_0", 301, 8192, 2048),
        # 24 sequences decoded together, LLaMA-3.2-3B gate
        lin("q4_k_batch", "q4_k", 24, 3072, 8192),
        # the lm_head of LLaMA-3.2-3B: the largest matvec of a decode step
        lin("q6_k_head", "q6_k", 1, 3072, 128256),
        # a long prompt through a Mistral-7B gate projection
        lin("q8_0_prefill", "q8_0", 2048, 4096, 14336),
        # one sampled token of a chat: the usual settings, Qwen3's vocabulary
        dict(name="sample_chat", kind="sample", vocab=151936, temperature=0.8, top_k=50,
             top_p=0.95, penalty=1.1, history=200),
        # a turn of each decoder: prompt, then 8 decode steps
        dict(name="int8_turn", kind="lm", model="int8", layers=4, vocab=32000, prompt=128, steps=8),
        dict(name="kquant_turn", kind="lm", model="kquant", layers=2, vocab=32000, prompt=256,
             steps=8),
        dict(name="hybrid_turn", kind="lm", model="hybrid", layers=4, vocab=32000, prompt=64,
             steps=8),
        dict(name="mamba_turn", kind="lm", model="mamba", layers=4, vocab=32000, prompt=96,
             steps=8, int8_xdt=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("linear", "sample", "lm"), (7, 1, 4))[0]
    if kind == "linear":
        fmt = rng.choice(sorted(FMT))
        el = 1 if fmt == "int8" else BLOCK[fmt][0]  # int8 takes any row length
        while True:
            m = 1 if rng.random() < 0.3 else _log_int(rng, 2, 2048)
            k = el * max(1, _log_int(rng, 512, 14336) // el)
            n = _log_int(rng, 256, 32768)
            if fmt != "int8":  # the K-split prompt GEMM takes output rows of whole 16 bytes
                n -= n % 4
            if m * k * n <= 2048 * 4096 * 14336:
                return dict(kind="linear", fmt=fmt, m=m, k=k, n=n)
    if kind == "sample":
        top_k = 0 if rng.random() < 0.3 else _log_int(rng, 1, 200)
        return dict(kind="sample", vocab=_log_int(rng, 1000, 151936),
                    temperature=0.0 if rng.random() < 0.1 else round(rng.uniform(0.5, 1.3), 2),
                    top_k=top_k, top_p=1.0 if rng.random() < 0.3 else round(rng.uniform(0.7, 0.99), 2),
                    penalty=1.0 if rng.random() < 0.3 else round(rng.uniform(1.05, 1.3), 2),
                    history=rng.randrange(0, 512))
    model = rng.choice(sorted(LAYER))
    c = dict(kind="lm", model=model, layers=rng.choice((2, 3, 4)), vocab=32000,
             prompt=_log_int(rng, 1, 512), steps=rng.randrange(1, 13))
    if model == "mamba":
        c["int8_xdt"] = rng.random() < 0.5
    return c


# ---------------------------------------------------------------- weights
def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000 + salt)
    return g


def _ints(g, shape, std, centre, lo, hi):
    """rounded normals in [lo, hi]: what a quantizer makes of normal weights"""
    v = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (v * std + centre).round_().clamp_(lo, hi)


def _f16(nb, lo, hi, g):
    """f16 block scales, uniform in [lo, hi)"""
    return (torch.rand(nb, generator=g, device="cuda") * (hi - lo) + lo).half()


def _bytes16(h):
    return h.view(torch.uint8).reshape(h.numel(), 2)


def _nibbles(q):
    """element 2i in the low, 2i+1 in the high nibble of byte i"""
    q = q.to(torch.uint8)
    return q[:, 0::2] | (q[:, 1::2] << 4)


def quantized(fmt, n, k, g, values):
    """A synthetic [n, k] matrix of `fmt`, normal with a standard deviation of
    about 0.03: its stored bytes (int8: the weights and row scales), or, with
    `values`, its values in float64."""
    if fmt == "int8":
        q = _ints(g, (n, k), 36.0, 0.0, -127, 127)
        s = torch.rand(n, generator=g, device="cuda") * 4e-4 + 6e-4
        return q.double() * s.double()[:, None] if values else (q.to(torch.int8), s)
    el, _ = BLOCK[fmt]
    nb = n * (k // el)
    if fmt == "q4_0":
        q = _ints(g, (nb, 32), 2.6, 8.0, 0, 15)
        d = _f16(nb, 0.008, 0.014, g)
        if values:
            return ((q.double() - 8.0) * d.double()[:, None]).reshape(n, k)
        return torch.cat([_bytes16(d), _nibbles(q)], 1)
    if fmt == "q8_0":
        q = _ints(g, (nb, 32), 44.0, 0.0, -127, 127)
        d = _f16(nb, 5e-4, 8e-4, g)
        if values:
            return (q.double() * d.double()[:, None]).reshape(n, k)
        return torch.cat([_bytes16(d), q.to(torch.int8).view(torch.uint8)], 1)
    if fmt == "q4_k":
        q = _ints(g, (nb, 256), 2.6, 7.5, 0, 15)
        sc = torch.randint(8, 16, (nb, 8), generator=g, device="cuda")
        mn = torch.randint(8, 16, (nb, 8), generator=g, device="cuda")
        d, dm = _f16(nb, 7e-4, 1.2e-3, g), _f16(nb, 5e-3, 9e-3, g)
        if values:
            scale = d.double()[:, None] * sc.double()
            low = dm.double()[:, None] * mn.double()
            return (q.double().reshape(nb, 8, 32) * scale[..., None] - low[..., None]).reshape(n, k)
        s8, m8 = sc.to(torch.uint8), mn.to(torch.uint8)  # 4-bit fields: their upper bits are zero
        fields = torch.cat([s8[:, :4], s8[:, 4:] | (m8[:, :4] << 4), m8[:, 4:] << 4], 1)
        return torch.cat([_bytes16(d), _bytes16(dm), fields, _nibbles(q)], 1)
    q = _ints(g, (nb, 256), 10.0, 32.0, 0, 63)  # q6_k
    sc = torch.randint(20, 60, (nb, 16), generator=g, device="cuda")
    d = _f16(nb, 7e-5, 1e-4, g)
    if values:
        scale = d.double()[:, None] * sc.double()
        return ((q.double().reshape(nb, 16, 16) - 32.0) * scale[..., None]).reshape(n, k)
    q = q.to(torch.uint8)
    hi = (q >> 4).reshape(nb, 64, 4)
    qh = hi[..., 0] | (hi[..., 1] << 2) | (hi[..., 2] << 4) | (hi[..., 3] << 6)
    return torch.cat([_nibbles(q & 15), qh, sc.to(torch.uint8), _bytes16(d)], 1)


def _host(t):
    return t.cpu().numpy()


def normal(n, seed, std):
    """The library's synthetic normals (SplitMix64 draws, Box-Muller in
    float64, rounded to float32).  On the CPU, as are the quantizers of the
    decoders' weights below: one level of one weight in ten million that
    another rounding moves would show as 1e-4 in the logits."""
    pairs = (n + 1) // 2
    i = torch.arange(1, 2 * pairs + 1, dtype=torch.int64)
    wrap = lambda v: v - (1 << 64) if v >= 1 << 63 else v
    srl = lambda z, b: (z >> b) & ((1 << (64 - b)) - 1)
    z = i * wrap(0x9E3779B97F4A7C15) + wrap(seed & ((1 << 64) - 1))
    z = (z ^ srl(z, 30)) * wrap(0xBF58476D1CE4E5B9)
    z = (z ^ srl(z, 27)) * wrap(0x94D049BB133111EB)
    z = srl(z ^ srl(z, 31), 11).double().reshape(pairs, 2)
    r = torch.sqrt(-2.0 * torch.log((z[:, 0] + 1.0) / 9007199254740992.0))
    a = 2.0 * math.pi * (z[:, 1] / 9007199254740992.0)
    out = torch.stack([r * torch.cos(a), r * torch.sin(a)], 1).reshape(-1)[:n]
    return (out * float(np.float32(std))).float()  # the library takes std as a float


# ---------------------------------------------------------------- prepare
def _activations(c, seed):
    """normal rows, a few channels ten times larger, as hidden states have them"""
    g = _gen(seed, 1)
    x = torch.randn((c["m"], c["k"]), generator=g, device="cuda")
    big = torch.randint(0, c["k"], (max(1, c["k"] // 500),), generator=g, device="cuda")
    x[:, big] *= 10.0
    return x


def _ids(c, seed):
    return np.random.default_rng(seed).integers(0, c["vocab"], c["prompt"] + c["steps"],
                                                dtype=np.uint32)


def _base(seed):
    return 0x5EED0000 + 100003 * int(seed)


def _kinds(c):
    return [0, 0, 1, 0][:c["layers"]] if c["layers"] > 2 else [0, 1]


PROJ = ("q", "k", "v", "o", "gate", "up", "down")


def _kquant_tensors(c, seed, values):
    """layers of seven projections (Q4_K, the down projection Q6_K), then the lm_head (Q6_K)"""
    w = LAYER["kquant"]
    h, qd, kvd, f = (w["hidden"], w["n_heads"] * w["head_dim"], w["n_kv_heads"] * w["head_dim"],
                     w["inter"])
    shape = dict(q=(qd, h), k=(kvd, h), v=(kvd, h), o=(h, qd), gate=(f, h), up=(f, h), down=(h, f))
    for layer in range(c["layers"]):
        for i, p in enumerate(PROJ):
            fmt = "q6_k" if p == "down" else "q4_k"
            yield layer, p, quantized(fmt, *shape[p], _gen(seed, 10 + 8 * layer + i), values)
    yield -1, "lm_head", quantized("q6_k", c["vocab"], h, _gen(seed, 5), values)


def _embed(c, seed):
    """the K-quant decoder's embedding"""
    shape = (c["vocab"], LAYER["kquant"]["hidden"])
    return torch.randn(shape, generator=_gen(seed, 4), device="cuda") * STD


def _model(c, seed):
    w = LAYER[c["model"]]
    room = c["prompt"] + c["steps"] + 1
    if c["model"] == "mamba":
        m = hip.QuantizedMamba(dict(w, n_layers=c["layers"], vocab=c["vocab"], max_tokens=room),
                               int8_xdt=c["int8_xdt"])
        m.init_synthetic(_base(seed), STD)
    elif c["model"] == "hybrid":
        m = hip.HybridLM(dict(w, n_layers=c["layers"], vocab=c["vocab"], max_seq=room,
                              layer_kinds=_kinds(c)))
        m.init_synthetic(_base(seed), STD)
    elif c["model"] == "int8":
        m = hip.QuantizedCausalLM(dict(w, n_layers=c["layers"], vocab=c["vocab"], max_seq=room))
        m.init_synthetic(_base(seed), STD)
    else:
        m = hip.KQuantCausalLM(dict(w, n_layers=c["layers"], vocab=c["vocab"], max_seq=room))
        m.set_embed(_host(_embed(c, seed)))
        for layer, p, blocks in _kquant_tensors(c, seed, False):
            if layer < 0:
                m.set_lm_head(_host(blocks))
            else:
                m.set_proj(layer, PROJ.index(p), _host(blocks))
        m.finalize()
    return m


def prepare(case, seed):
    hip.init(0)
    c = dict(case)
    if c["kind"] == "linear":
        stored = quantized(c["fmt"], c["n"], c["k"], _gen(seed), False)
        if c["fmt"] == "int8":
            lin = hip.QLinear.int8(_host(stored[0]), _host(stored[1]), hip.LAYOUT_NK)
        elif c["fmt"] == "q4_0":
            lin = hip.QLinear.q4_0(_host(stored), c["n"], c["k"])
        else:
            lin = hip.QLinear.gguf(FMT[c["fmt"]], _host(stored), c["n"], c["k"])
        return dict(c, lin=lin, x=_activations(c, seed),
                    y=torch.zeros((c["m"], c["n"]), device="cuda"))
    if c["kind"] == "sample":
        g = _gen(seed)
        rng = np.random.default_rng(seed)
        logits = torch.randn(c["vocab"], generator=g, device="cuda") * 2.5
        hist = torch.randint(0, c["vocab"], (max(1, c["history"]),), generator=g, device="cuda",
                             dtype=torch.int32)
        return dict(c, logits=logits, hist=hist, u=float(np.float32(rng.random())),
                    token=torch.zeros(1, dtype=torch.int32, device="cuda"),
                    prm=hip.sampler_params(c["temperature"], c["top_k"], c["top_p"], c["penalty"]))
    return dict(c, lm=_model(c, seed), ids=_ids(c, seed))


# ---------------------------------------------------------------- run
def run(state):
    s = state
    if s["kind"] == "linear":
        s["lin"].forward_dev(s["m"], s["x"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    if s["kind"] == "sample":
        hip.check(hip.lib().syn_hip_sample(s["logits"].data_ptr(), s["vocab"], s["hist"].data_ptr(),
                                           s["history"], s["prm"], s["u"], s["token"].data_ptr(),
                                           None, None), "sample")
        return s["token"]
    lm, ids, p = s["lm"], s["ids"], s["prompt"]
    one = lm.decode_one if s["model"] in ("hybrid", "mamba") else lm.forward_one
    if s["model"] == "hybrid":
        lm.reset()
    out = [lm.prefill(ids[:p])]
    for t in ids[p:]:
        out.append(one(int(t)))
    return np.stack(out)


# ---------------------------------------------------------------- work, tolerance
def _weights(c):
    """(weights of the layers, bytes of the layers, bytes of the lm_head)"""
    w, n = LAYER[c["model"]], c["layers"]
    if c["model"] == "mamba":
        dm, di, dr, ds = w["d_model"], w["d_inner"], w["dt_rank"], w["d_state"]
        big, small = 3 * di * dm, (dr + 2 * ds) * di + di * dr
        return (n * (big + small), n * (big + small * (1 if c["int8_xdt"] else 4)),
                c["vocab"] * dm * 4)
    h, f = w["hidden"], w["inter"]
    qd, kvd = w["n_heads"] * w["head_dim"], w["n_kv_heads"] * w["head_dim"]
    attn = 2 * h * qd + 2 * h * kvd
    if c["model"] == "hybrid":
        kinds = _kinds(c)
        total = sum((attn if kind else 4 * w["inner"] * h) + 3 * h * f for kind in kinds)
        return total, total // 32 * 18, c["vocab"] * h * 4
    total = n * (attn + 3 * h * f)
    if c["model"] == "int8":
        return total, total, c["vocab"] * h
    return (total, n * ((attn + 2 * h * f) // 256 * 144 + h * f // 256 * 210),
            c["vocab"] * h // 256 * 210)


def work(case):
    c = case
    if c["kind"] == "linear":
        if c["fmt"] == "int8":
            stored = c["n"] * c["k"] + 4 * c["n"]
        else:
            el, b = BLOCK[c["fmt"]]
            stored = c["n"] * (c["k"] // el) * b
        return {"bytes": stored + 4 * c["m"] * (c["k"] + c["n"]),
                "flops": 2 * c["m"] * c["k"] * c["n"]}
    if c["kind"] == "sample":
        return {"bytes": 4 * (c["vocab"] + c["history"]), "flops": 0}
    # the prompt reads the weights once, each decode step once again
    total, layer_bytes, head = _weights(c)
    head_flops = 2 * c["vocab"] * LAYER[c["model"]].get("hidden", 1024)
    return {"bytes": (1 + c["steps"]) * (layer_bytes + head + 4 * c["vocab"]),
            "flops": 2 * total * (c["prompt"] + c["steps"]) + head_flops * (1 + c["steps"])}


def tolerance(case):
    c = case
    if c["kind"] == "sample":
        return "exact"  # a token
    if c["kind"] == "linear":
        if c["fmt"] == "int8":
            return {"rel": 1e-6}  # exact integer sums, a few 32-bit operations each
        # 32-bit sums for a few rows; for more, activations and weights
        # rounded to 16 bits (2^-12 each at the middle of a binade)
        return {"rel": 1e-5} if c["m"] <= 8 else {"rel": 1.2e-3}
    # the INT8 decoders round activations to 8 bits: a last-bit difference
    # becomes a quantization step in every later layer
    return {"int8": {"rel": 3e-2}, "mamba": {"rel": 3e-2}, "kquant": {"rel": 4e-3},
            "hybrid": {"rel": 2e-5}}[c["model"]]


# ---------------------------------------------------------------- exact
def _q8(x):
    """per-row 8-bit activations: (levels, scale)"""
    m = x.abs().amax(-1, keepdim=True)
    s = torch.where(m > 0, m / 127.0, torch.ones_like(m))
    v = x / s
    return (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp(-127, 127), s


def _w8(w):
    """per-row 8-bit weights of a float32 matrix, rounded as they are stored"""
    m = w.abs().amax(1, keepdim=True)
    s = torch.where(m > 0, m / 127.0, torch.ones_like(m))
    v = w * (1.0 / s)
    q = (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp(-128, 127)
    return q.cuda().double(), s.cuda().double()


def _linear8(x, w):
    q, s = _q8(x)
    return (q @ w[0].T) * s * w[1].T


def _rms(x, g, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g


def _rope(x, theta):
    t, _, hd = x.shape
    i = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    ang = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] / theta ** (2.0 * i / hd)
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attention(q, k, v):
    """causal, q [T, heads, hd], k and v [T, kv heads, hd]"""
    t, nh, hd = q.shape
    rep = nh // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    mask = torch.ones((t, t), device="cuda", dtype=torch.bool).triu(1)
    out = torch.empty_like(q)
    for h in range(nh):
        s = (q[:, h] @ k[:, h].T.contiguous() / math.sqrt(hd)).masked_fill(mask, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ v[:, h].contiguous()
    return out.reshape(t, nh * hd)


def _gqa(x, w, lin, L, qn, kn, eps):
    t, hd = x.shape[0], w["head_dim"]
    q = lin(x, L["q"]).reshape(t, w["n_heads"], hd)
    k = lin(x, L["k"]).reshape(t, w["n_kv_heads"], hd)
    v = lin(x, L["v"]).reshape(t, w["n_kv_heads"], hd)
    if qn is not None:
        q, k = _rms(q, qn, eps), _rms(k, kn, eps)
    return lin(_attention(_rope(q, w["rope_theta"]), _rope(k, w["rope_theta"]), v), L["o"])


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_transformer(c, seed, x):
    """the INT8 and K-quant decoders over all tokens: the last hidden rows and the lm_head"""
    w = LAYER[c["model"]]
    h, qd, kvd, f = (w["hidden"], w["n_heads"] * w["head_dim"], w["n_kv_heads"] * w["head_dim"],
                     w["inter"])
    int8 = c["model"] == "int8"
    lin = _linear8 if int8 else (lambda a, m: a @ m.T)
    layers = [{} for _ in range(c["layers"])]
    if int8:
        shape = dict(q=(qd, h), k=(kvd, h), v=(kvd, h), o=(h, qd), gate=(f, h), up=(f, h),
                     down=(h, f))
        for i, L in enumerate(layers):
            for j, p in enumerate(PROJ):
                n, k = shape[p]
                L[p] = _w8(normal(n * k, _base(seed) + 1 + 8 * i + j, STD).reshape(n, k))
        head = _w8(normal(c["vocab"] * h, _base(seed), STD).reshape(-1, h))
    else:
        for i, p, v in _kquant_tensors(c, seed, True):
            if i < 0:
                head = v
            else:
                layers[i][p] = v
    one = torch.ones((), device="cuda", dtype=torch.float64) if int8 else None
    for L in layers:
        x = x + _gqa(_rms(x, 1.0, w["eps"]), w, lin, L, one, one, w["eps"])
        n = _rms(x, 1.0, w["eps"])
        x = x + lin(_silu(lin(n, L["gate"])) * lin(n, L["up"]), L["down"])
    return lin(_rms(x[c["prompt"] - 1:], 1.0, w["eps"]), head)


def _q4_values(n, k, seed):
    """the Q4_0 values of an [n, k] matrix of synthetic normals: blocks of 32,
    scale max/7 cut to f16, levels round(w * 7 / max) in [-8, 7]"""
    v = normal(n * k, seed, STD).reshape(-1, 32)
    scale = v.abs().amax(1, keepdim=True) / 7.0
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    r = v * inv
    q = (torch.sign(r) * torch.floor(r.abs() + 0.5)).clamp(-8, 7).double()
    bits = scale.view(torch.int32) & ~0x1FFF  # toward zero: the scales are normal f16 values
    return (q.cuda() * bits.view(torch.float32).double().cuda()).reshape(n, k)


def _gain(n, seed):
    return (1.0 + normal(n, seed, 0.1)).double().cuda()


def _exact_hybrid(c, seed, x, embed):
    w = LAYER["hybrid"]
    h, inner, f, hd, ck = w["hidden"], w["inner"], w["inter"], w["head_dim"], w["conv_kernel"]
    qd, kvd = w["n_heads"] * hd, w["n_kv_heads"] * hd
    lin = lambda a, m: a @ m.T
    for i, kind in enumerate(_kinds(c)):
        s = _base(seed) + 1 + 16 * i
        n = _rms(x, _gain(h, s + 8), w["eps"])
        if kind == 0:
            p = n @ _q4_values(3 * inner, h, s).T
            bx = p[:, :inner] * p[:, 2 * inner:]
            taps = normal(inner * ck, s + 1, STD).double().cuda().reshape(inner, ck)
            past = torch.cat([torch.zeros((ck - 1, inner), device="cuda", dtype=torch.float64), bx])
            conv = sum(past[j:j + x.shape[0]] * taps[:, j] for j in range(ck))
            x = x + (p[:, inner:2 * inner] * conv) @ _q4_values(h, inner, s + 2).T
        else:
            L = dict(q=_q4_values(qd, h, s), k=_q4_values(kvd, h, s + 1),
                     v=_q4_values(kvd, h, s + 2), o=_q4_values(h, qd, s + 3))
            x = x + _gqa(n, w, lin, L, _gain(hd, s + 6), _gain(hd, s + 7), w["eps"])
        n = _rms(x, _gain(h, s + 9), w["eps"])
        a = _silu(n @ _q4_values(f, h, s + 10).T) * (n @ _q4_values(f, h, s + 11).T)
        x = x + a @ _q4_values(h, f, s + 12).T
    g = _gain(h, _base(seed) + 1 + 16 * c["layers"])
    return _rms(x[c["prompt"] - 1:], g, w["eps"]) @ embed.T


def _exact_mamba(c, seed, x, embed):
    w = LAYER["mamba"]
    dm, di, ds, dc, dr = w["d_model"], w["d_inner"], w["d_state"], w["d_conv"], w["dt_rank"]
    t = x.shape[0]
    bias = math.log(math.expm1(0.01))
    a = -torch.arange(1, ds + 1, device="cuda", dtype=torch.float64)
    for i in range(c["layers"]):
        s = _base(seed) + 1 + 16 * i
        mat = lambda n, k, j: normal(n * k, s + j, STD).reshape(n, k)
        lin = _linear8 if c["int8_xdt"] else (lambda v, m: v @ m.T)
        rows = _w8 if c["int8_xdt"] else (lambda m: m.double().cuda())
        p = _linear8(_rms(x, 1.0, w["eps"]), _w8(mat(2 * di, dm, 0)))
        taps = mat(di, dc, 1).double().cuda()
        past = torch.cat([torch.zeros((dc - 1, di), device="cuda", dtype=torch.float64), p[:, :di]])
        xc = _silu(sum(past[j:j + t] * taps[:, j] for j in range(dc)))
        xp = lin(xc, rows(mat(dr + 2 * ds, di, 2)))
        delta = torch.nn.functional.softplus(lin(xp[:, :dr], rows(mat(di, dr, 3))) + bias)
        B, C = xp[:, dr:dr + ds], xp[:, dr + ds:]
        state = torch.zeros((di, ds), device="cuda", dtype=torch.float64)
        y = torch.empty((t, di), device="cuda", dtype=torch.float64)
        for j in range(t):
            state = (torch.exp(delta[j][:, None] * a) * state
                     + (delta[j] * xc[j])[:, None] * B[j][None, :])
            y[j] = state @ C[j]
        x = x + _linear8((y + xc) * _silu(p[:, di:]), _w8(mat(dm, di, 4)))
    return _rms(x[c["prompt"] - 1:], 1.0, w["eps"]) @ embed.T


def exact(case, seed):
    c = case
    if c["kind"] == "sample":
        return None  # whole numbers
    if c["kind"] == "linear":
        x = _activations(c, seed)
        if c["fmt"] == "int8":  # the 8-bit levels are part of the function: rounded in 32 bits
            m = x.abs().amax(1, keepdim=True)
            r = x * (127.0 / m)
            q = (torch.sign(r) * torch.floor(r.abs() + 0.5)).clamp(-127, 127)
            x = q.double() * (m / 127.0).double()
        return x.double() @ quantized(c["fmt"], c["n"], c["k"], _gen(seed), True).T
    ids = torch.from_numpy(_ids(c, seed).astype(np.int64)).cuda()
    if c["model"] == "kquant":
        embed = _embed(c, seed)
    else:
        embed = normal(c["vocab"] * 1024, _base(seed), STD).cuda().reshape(c["vocab"], 1024)
    embed = embed.double()
    x = embed[ids]
    if c["model"] == "hybrid":
        out = _exact_hybrid(c, seed, x, embed)
    elif c["model"] == "mamba":
        out = _exact_mamba(c, seed, x, embed)
    else:
        out = _exact_transformer(c, seed, x)
    return out.cpu().numpy()
