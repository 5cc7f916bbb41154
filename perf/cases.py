"""Performance cases of the Q4 matmul library: what a program that decodes and prefills with
quantised weights asks of it, through its public entry points.

A case is a dict of plain values with a ``kind``:

* ``proj``     one decode projection (a GEMV, or a skinny GEMM over a batch of sequences) in
               one of the weight formats a model file holds, with or without the residual
* ``head``     lm_head over the vocabulary and its top-k
* ``ffn``      a decode FFN: RMSNorm, gate and up with SwiGLU, down with the residual
* ``step``     one whole decode step of a dense model, attention left out: logits
* ``prefill``  one prefill projection
* ``layer``    the prefill matmuls and norms of one dense decoder layer, attention left out
* ``moe``      a routed expert block, decode or prefill, with or without a shared expert

Weights are GGUF blocks with the distribution of the benchmark's (random codes, scales and
mins so that a weight is about N(0, 0.01)); activations are N(0, 1).
"""
import importlib
import math

import torch

q4 = importlib.import_module("openflowlm-next_amd")

EPS = 1e-6
DEV = "cuda"

# bytes per weight as the file stores them, and the K multiple of one block
FORMATS = {"q4_1": (20 / 32, 32), "q4_1_fp16": (20 / 32, 32), "q4_0": (18 / 32, 32), "q4_k": (144 / 256, 256),
           "q8_0": (34 / 32, 32)}


def listed():
    return [
        # the smallest call: one attention projection of an 8B model for one token, f32 activations
        dict(name="proj_4096_m1", kind="proj", fmt="q4_1", m=1, n=4096, k=4096, x="f32", residual=False),
        # a full decode batch through an FFN projection, bf16 activations
        dict(name="proj_14336x4096_m16", kind="proj", fmt="q4_1", m=16, n=14336, k=4096, x="bf16", residual=False),
        # a K-quant file, four sequences: the down projection with its residual add
        dict(name="q4k_4096x14336_m4", kind="proj", fmt="q4_k", m=4, n=4096, k=14336, x="bf16", residual=True),
        # the 8-bit lm_head many files carry, with top-40 sampling for a batch of eight
        dict(name="head_q8_m8", kind="head", fmt="q8_0", m=8, n=128256, k=4096, topk=40),
        # an odd decode batch through a whole FFN
        dict(name="ffn_decode_m5", kind="ffn", m=5, h=4096, f=14336),
        # one token through all 32 layers and lm_head of an 8B model
        dict(name="decode_step_8b", kind="step", layers=32, h=4096, f=14336, nq=6144, vocab=128256),
        # a short chat turn: a ragged hundred tokens through one attention projection
        dict(name="prefill_4096_t100", kind="prefill", t=100, n=4096, k=4096, x="bf16", precision="fp16"),
        # a prompt of middling length through one decoder layer's matmuls and norms
        dict(name="prefill_layer_t512", kind="layer", t=512, h=4096, f=14336, nq=6144, precision="fp16"),
        # the largest prompt block through an FFN projection
        dict(name="prefill_14336x4096_t2048", kind="prefill", t=2048, n=14336, k=4096, x="bf16", precision="fp16"),
        # a decode batch of 16 through a 128-expert block, shared expert and residual included
        dict(name="moe_decode_t16", kind="moe", t=16, e=128, topk=8, h=2048, f=768, fs=768),
        # a short prompt through the same experts
        dict(name="moe_t300", kind="moe", t=300, e=128, topk=8, h=2048, f=768, fs=0),
        # a long prompt through the same experts
        dict(name="moe_t2048", kind="moe", t=2048, e=128, topk=8, h=2048, f=768, fs=0),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return min(hi // step * step, max(-(-lo // step) * step, int(v / step + 0.5) * step))


def draw(rng):
    kind = rng.choice(("proj", "proj", "proj", "head", "ffn", "step", "prefill", "prefill", "prefill", "layer", "moe",
                       "moe", "moe"))
    if kind == "proj":
        fmt = rng.choice(("q4_1", "q4_1", "q4_1", "q4_1_fp16", "q4_0", "q4_k", "q8_0"))
        m = _log(rng, 1, 24 if fmt == "q4_1" else 16)
        return dict(kind=kind, fmt=fmt, m=m, n=_log(rng, 512, 28672, 64),
                    k=_log(rng, 1024, 14336, 256 if fmt == "q4_k" else 32), x=rng.choice(("bf16", "bf16", "f32")),
                    residual=rng.random() < 0.4)
    if kind == "head":
        return dict(kind=kind, fmt=rng.choice(("q4_1", "q4_1", "q8_0")), m=_log(rng, 1, 16),
                    n=_log(rng, 32000, 128256, 64), k=_log(rng, 1024, 4096, 32), topk=rng.choice((1, 8, 40, 64)))
    if kind == "ffn":
        return dict(kind=kind, m=_log(rng, 1, 16), h=_log(rng, 1024, 8192, 64), f=_log(rng, 2048, 14336, 64))
    if kind == "step":
        h = _log(rng, 1024, 4096, 64)
        return dict(kind=kind, layers=_log(rng, 8, 32), h=h, f=_log(rng, 2 * h, 7 * h // 2, 64),
                    nq=rng.choice((h + h // 2, 2 * h, 3 * h)) // 64 * 64, vocab=_log(rng, 32000, 128256, 64))
    if kind == "prefill":
        n, k = _log(rng, 512, 28672, 64), _log(rng, 1024, 14336, rng.choice((64, 64, 64, 32)))
        t = _log(rng, 25, max(32, min(4096, 2048 * 14336 * 4096 // (n * k))))
        return dict(kind=kind, t=t, n=n, k=k, x=rng.choice(("bf16", "bf16", "bf16", "f32")) if t <= 1024 else "bf16",
                    precision=rng.choice(("fp16", "fp16", "fp16", "bf16")))
    if kind == "layer":
        h = _log(rng, 1024, 4096, 128)
        f = _log(rng, 2 * h, 7 * h // 2, 128)
        return dict(kind=kind, t=_log(rng, 25, min(1024, 512 * 4096 * 16896 // (h * (f + h)))), h=h, f=f,
                    nq=rng.choice((h + h // 2, 2 * h, 3 * h)) // 64 * 64, precision=rng.choice(("fp16", "fp16", "bf16")))
    topk = rng.choice((2, 4, 8))
    t = _log(rng, 1, 2048)
    shared = t * topk <= 4096 and rng.random() < 0.4    # the block's shared expert rides the decode path
    return dict(kind=kind, t=t, e=rng.choice((16, 32, 64, 128)), topk=topk, h=_log(rng, 1024, 2048, 256),
                f=_log(rng, 384, 1408, 128), fs=_log(rng, 384, 1408, 128) if shared else 0)


# ---------------------------------------------------------------------------
# inputs: every tensor from (seed, index) alone, on the GPU
# ---------------------------------------------------------------------------

def _gen(seed, index):
    return torch.Generator(DEV).manual_seed((int(seed) * 1000003 + index * 7919) % (1 << 62))


def _bytes16(t):
    return t.to(torch.float16).contiguous().unsqueeze(-1).view(torch.uint8)


def _blocks(fmt, n, k, seed, index):
    """GGUF blocks uint8[n, k / block, bytes] of one matrix."""
    g = _gen(seed, index)
    rand = lambda *s: torch.rand(s, generator=g, device=DEV)
    if fmt == "q4_k":
        b = torch.randint(0, 256, (n, k // 256, 144), generator=g, device=DEV, dtype=torch.uint8)
        d = (torch.randn((n, k // 256), generator=g, device=DEV).abs() * 6e-5 + 3e-6).to(torch.float16)
        b[..., 0:2] = _bytes16(d)
        b[..., 2:4] = _bytes16(7.5 * d.float() * (0.9 + 0.2 * rand(n, k // 256)))
        return b
    nb = k // 32
    d = (torch.randn((n, nb), generator=g, device=DEV).abs() * 0.002 + 1e-4).to(torch.float16)
    if fmt == "q8_0":
        b = torch.randint(0, 256, (n, nb, 34), generator=g, device=DEV, dtype=torch.uint8)
        b[..., 0:2] = _bytes16(d.float() / 16)
        return b
    w = 18 if fmt == "q4_0" else 20
    b = torch.randint(0, 256, (n, nb, w), generator=g, device=DEV, dtype=torch.uint8)
    b[..., 0:2] = _bytes16(d)
    if w == 20:
        b[..., 2:4] = _bytes16(-8 * d.float() * (0.9 + 0.2 * rand(n, nb)))
    return b


def _f16(b):
    return b.contiguous().view(torch.float16).squeeze(-1)


def _bf16(t):
    return t.float().to(torch.bfloat16).double()


def _nibbles(c):
    return torch.cat((c & 15, c >> 4), -1).double()


def _weights(fmt, b):
    """The blocks' weights in 64 bits. Scales are those the packed format documents: narrowed to
    bf16, except the fp16-scale and Q4_K forms, which keep the file's."""
    n = b.shape[0]
    if fmt == "q4_k":
        d, dmin = _f16(b[..., 0:2]).double(), _f16(b[..., 2:4]).double()
        s = b[..., 4:16].to(torch.int32)
        sc = torch.cat((s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)), -1).double()
        mn = torch.cat((s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)), -1).double()
        q = _nibbles(b[..., 16:].reshape(n, -1, 4, 32)).reshape(n, -1, 8, 32)
        return (q * (d[..., None] * sc)[..., None] - (dmin[..., None] * mn)[..., None]).reshape(n, -1)
    d = _f16(b[..., 0:2])
    if fmt == "q8_0":
        return (b[..., 2:].contiguous().view(torch.int8).double() * _bf16(d)[..., None]).reshape(n, -1)
    if fmt == "q4_0":
        return ((_nibbles(b[..., 2:]) - 8) * _bf16(d)[..., None]).reshape(n, -1)
    m = _f16(b[..., 2:4])
    d, m = (d.double(), m.double()) if fmt == "q4_1_fp16" else (_bf16(d), _bf16(m))
    return (_nibbles(b[..., 4:]) * d[..., None] + m[..., None]).reshape(n, -1)


def _pack(fmt, n, k, seed, index):
    b = _blocks(fmt, n, k, seed, index)
    if fmt == "q4_k":
        return q4.pack_q4_k_native(b)
    if fmt == "q8_0":
        return q4.pack_q8_native(b, n, k, "q8_0")
    if fmt == "q4_0":
        return q4.pack_q4_0_native(b, n, k)
    return q4.pack_q4_1(b, scales="fp16" if fmt == "q4_1_fp16" else "bf16")


def _exact_w(fmt, n, k, seed, index):
    return _weights(fmt, _blocks(fmt, n, k, seed, index))


def _randn(shape, seed, index, dtype=torch.float32):
    return torch.randn(shape, generator=_gen(seed, index), device=DEV).to(dtype)


def _norm_weight(h, seed, index):
    return (1 + 0.1 * _randn((h,), seed, index)).to(torch.bfloat16)


_DTYPE = {"bf16": torch.bfloat16, "f32": torch.float32}
_GEMM = {"q4_1": "gemm_q4", "q4_1_fp16": "gemm_q4", "q4_0": "gemm_q4_0_native", "q4_k": "gemm_q4k",
         "q8_0": "gemm_q8_native"}


def _interleaved(n_half, parts):
    """Gate and up blocks in alternating 64-row groups, as the packed expert layout wants them."""
    g, u = (p.view(n_half // 64, 64, *p.shape[1:]) for p in parts)
    return torch.stack((g, u), 1).reshape(2 * n_half, *parts[0].shape[1:])


def _routes(c, seed):
    p = torch.softmax(_randn((c["t"], c["e"]), seed, 90), -1)
    w, ids = torch.topk(p, c["topk"], -1)
    return ids.to(torch.int32), (w / w.sum(-1, keepdim=True)).contiguous()


# index of each tensor: 0..9 activations and norms (step: 10 per layer from 1000), 10.. weights
def prepare(case, seed):
    c = case
    kind = c["kind"]
    s = dict(kind=kind, case=c)
    if kind == "proj":
        s["w"] = _pack(c["fmt"], c["n"], c["k"], seed, 10)
        s["x"] = _randn((c["m"], c["k"]), seed, 0, _DTYPE[c["x"]])
        s["residual"] = _randn((c["m"], c["n"]), seed, 1) if c["residual"] else None
        s["gemm"] = getattr(q4, _GEMM[c["fmt"]])
    elif kind == "head":
        s["w"] = _pack(c["fmt"], c["n"], c["k"], seed, 10)
        s["x"] = _randn((c["m"], c["k"]), seed, 0, torch.bfloat16)
    elif kind == "ffn":
        s["gate"], s["up"] = (_pack("q4_1", c["f"], c["h"], seed, i) for i in (10, 11))
        s["down"] = _pack("q4_1", c["h"], c["f"], seed, 12)
        s["x"], s["nw"] = _randn((c["m"], c["h"]), seed, 0), _norm_weight(c["h"], seed, 1)
    elif kind == "step":
        h, f, nq, n = c["h"], c["f"], c["nq"], c["layers"]
        pk = lambda rows, k, i: _pack("q4_1", rows, k, seed, i)
        s["layers"] = [dict(qkv=pk(nq, h, b), o=pk(h, h, b + 1), gate=pk(f, h, b + 2), up=pk(f, h, b + 3),
                            down=pk(h, f, b + 4), attn=_randn((h,), seed, b + 5, torch.bfloat16),
                            nw1=_norm_weight(h, seed, b + 6), nw2=_norm_weight(h, seed, b + 7))
                       for b in range(1000, 1000 + 10 * n, 10)]
        s["head"], s["nw"] = pk(c["vocab"], h, 10), _norm_weight(h, seed, 1)
        s["x"] = _randn((1, h), seed, 0)
        # the buffers a decode loop keeps
        _, sd, sq = q4.decode_segment_splits(h, f, nq)
        e = lambda *shape: torch.empty(shape, device=DEV)
        s.update(x_mid=e(1, h), x_next=e(1, h), x_out=e(1, h), down_planes=e(sd, 1, h), qkv_planes=e(n - 1, sq, 1, nq),
                 qkv0=e(1, nq), logits=e(1, c["vocab"]), workspace=q4.decode_segment_workspace(h, f, nq))
    elif kind == "prefill":
        s["w"] = _pack("q4_1", c["n"], c["k"], seed, 10)
        s["x"] = _randn((c["t"], c["k"]), seed, 0, _DTYPE[c["x"]])
        if c["precision"] == "fp16":
            q4.prefill_scales(s["w"])
    elif kind == "layer":
        h, f = c["h"], c["f"]
        s["qkv"], s["o"] = _pack("q4_1", c["nq"], h, seed, 10), _pack("q4_1", h, h, seed, 11)
        s["gate_up"] = q4.pack_q4_1(_interleaved(f, [_blocks("q4_1", f, h, seed, i) for i in (12, 13)]))
        s["down"] = _pack("q4_1", h, f, seed, 14)
        s["x"], s["attn"] = _randn((c["t"], h), seed, 0), _randn((c["t"], h), seed, 1, torch.bfloat16)
        s["nw"] = [_norm_weight(h, seed, i) for i in (2, 3, 4)]
        if c["precision"] == "fp16":
            for w in ("qkv", "o", "gate_up", "down"):
                q4.prefill_scales(s[w])
    else:
        e, h, f = c["e"], c["h"], c["f"]
        gu = torch.cat([_interleaved(f, [_blocks("q4_1", f, h, seed, 1000 + 10 * i + j) for j in (0, 1)])
                        for i in range(e)])
        s["gate_up"] = q4.PackedExperts(q4.pack_q4_1(gu).data, e, 2 * f, h)
        dn = torch.cat([_blocks("q4_1", h, f, seed, 1000 + 10 * i + 2) for i in range(e)])
        s["down"] = q4.PackedExperts(q4.pack_q4_1(dn).data, e, h, f)
        s["x"] = _randn((c["t"], h), seed, 0, torch.bfloat16)
        s["ids"], s["wts"] = _routes(c, seed)
        s["more"] = {}
        if c["fs"]:
            sgu = q4.pack_q4_1(_interleaved(c["fs"], [_blocks("q4_1", c["fs"], h, seed, i) for i in (10, 11)]))
            s["more"] = dict(shared_expert=(sgu, _pack("q4_1", h, c["fs"], seed, 12)), residual=_randn((c["t"], h), seed, 1),
                             shared_gate_w=_randn((h,), seed, 2, torch.bfloat16) / 16)
        if c["t"] * c["topk"] > q4.MOE_DECODE_MAX_PAIRS:
            q4.prefill_scales(s["gate_up"]), q4.prefill_scales(s["down"])
    return s


def run(state):
    s = state
    kind = s["kind"]
    if kind == "proj":
        return s["gemm"](s["w"], s["x"], residual=s["residual"])
    if kind == "head":
        c = s["case"]
        if c["fmt"] == "q4_1":
            ids, vals, logits = q4.lm_head_topk(s["w"], s["x"], k=c["topk"])
        else:
            logits = q4.gemm_q8_native(s["w"], s["x"])
            ids, vals = q4.logits_topk(logits, k=c["topk"])
        return dict(ids=ids, vals=vals, logits=logits)
    if kind == "ffn":
        h = q4.swiglu_q4(s["gate"], s["up"], s["x"], out_dtype=torch.bfloat16, norm_w=s["nw"], eps=EPS)
        return dict(h=h, y=q4.gemm_q4(s["down"], h, residual=s["x"]))
    if kind == "step":
        ls = s["layers"]
        q4.gemm_q4_rmsnorm(ls[0]["qkv"], s["x"], ls[0]["nw1"], EPS, y=s["qkv0"])
        x = s["x"]
        for i, p in enumerate(ls):
            if i + 1 < len(ls):
                q4.decode_segment(p["o"], p["gate"], p["up"], p["down"], ls[i + 1]["qkv"], p["attn"], x, p["nw2"],
                                  ls[i + 1]["nw1"], EPS, x_mid=s["x_mid"], x_next=s["x_next"],
                                  down_planes=s["down_planes"], qkv_planes=s["qkv_planes"][i], workspace=s["workspace"])
                x = s["x_next"]
            else:
                q4.decode_segment(p["o"], p["gate"], p["up"], p["down"], None, p["attn"], x, p["nw2"], eps=EPS,
                                  x_mid=s["x_mid"], down_planes=s["down_planes"], workspace=s["workspace"])
        q4.gemm_q4_rmsnorm_acc(s["head"], s["x_mid"], s["down_planes"], s["nw"], EPS, x_out=s["x_out"], y=s["logits"])
        return dict(logits=s["logits"], x=s["x_out"], qkv0=s["qkv0"], qkv=s["qkv_planes"].sum(1))
    if kind == "prefill":
        return q4.gemm_q4_prefill(s["w"], s["x"], precision=s["case"]["precision"])
    if kind == "layer":
        prec = s["case"]["precision"]
        _, xn = q4.rmsnorm_prepare(s["x"], s["nw"][0], eps=EPS, precision=prec)
        qkv = q4.gemm_q4_prefill(s["qkv"], xn)
        part = q4.gemm_q4_prefill_partials(s["o"], q4.prefill_prepare(s["attn"], prec))
        x_mid, xn = q4.rmsnorm_prepare(s["x"], s["nw"][1], add=part, eps=EPS, precision=prec)
        h = q4.gemm_q4_prefill_swiglu(s["gate_up"], xn)
        part = q4.gemm_q4_prefill_partials(s["down"], q4.prefill_prepare(h, prec))
        x_next, xn = q4.rmsnorm_prepare(x_mid, s["nw"][2], add=part, eps=EPS, precision=prec)   # xn: the next layer's
        return dict(qkv=qkv, x_mid=x_mid, h=h, x_next=x_next)
    return q4.moe_batch(s["gate_up"], s["down"], s["x"], s["ids"], s["wts"], **s["more"])


def work(case):
    c = case
    kind = c["kind"]
    q = FORMATS["q4_1"][0]
    if kind in ("proj", "prefill", "head"):
        m, n, k = c.get("m", c.get("t")), c["n"], c["k"]
        xb = 4 if c.get("x") == "f32" else 2
        bytes_ = n * k * FORMATS[c.get("fmt", "q4_1")][0] + m * k * xb + m * n * (8 if c.get("residual") else 4)
        return dict(bytes=bytes_ + (8 * m * c["topk"] if kind == "head" else 0), flops=2 * m * n * k)
    if kind == "ffn":
        m, h, f = c["m"], c["h"], c["f"]
        return dict(bytes=3 * h * f * q + m * (8 * h + 2 * f) + 2 * h, flops=6 * m * h * f)
    if kind == "step":
        h, f, nq = c["h"], c["f"], c["nq"]
        weights = c["layers"] * (h * h + 3 * h * f + nq * h) + c["vocab"] * h
        return dict(bytes=weights * q + c["layers"] * (6 * h + 4 * nq) + 10 * h + 4 * c["vocab"], flops=2 * weights)
    if kind == "layer":
        t, h, f, nq = c["t"], c["h"], c["f"], c["nq"]
        weights = h * h + 3 * h * f + nq * h
        return dict(bytes=weights * q + t * (4 * h + 2 * h + 4 * nq + 4 * h + 2 * f + 4 * h) + 6 * h, flops=2 * t * weights)
    t, h, f, fs = c["t"], c["h"], c["f"], c["fs"]
    hit = c["e"] * (1 - (1 - c["topk"] / c["e"]) ** t)      # experts a batch reaches
    bytes_ = (hit * 3 * h * f + 3 * h * fs) * q + t * (2 * h + 4 * h + 8 * c["topk"]) + (t * 4 * h + 2 * h if fs else 0)
    return dict(bytes=bytes_, flops=6 * t * h * (c["topk"] * f + fs))


def tolerance(case):
    """About four times the largest error against 64 bits seen over the ranges of draw()."""
    c = case
    if c["kind"] in ("ffn", "layer", "step"):       # bf16 between the matmuls, as their interfaces have it
        return {"rel": 1.5e-2 if c.get("precision") == "bf16" else 1.2e-2}
    if c["kind"] == "moe":                          # f32 throughout up to 4096 pairs, then h in bf16
        return {"rel": 1.4e-5 if c["t"] * c["topk"] <= q4.MOE_DECODE_MAX_PAIRS else 6.5e-3}
    if c.get("precision") == "bf16":                # weights rounded to bf16
        return {"rel": 9e-3}
    if c["kind"] == "head":                         # a near tie may change places
        return {"rel": 3e-6, "differ": 0.01}
    return {"rel": 3e-6 if c["x"] == "bf16" or c["kind"] == "prefill" else 1.3e-5}   # 32-bit sums; f32 x as two bf16


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------

def _rms(x, nw):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * nw.double()


def _swiglu(g, u):
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    c = case
    kind = c["kind"]
    w = lambda n, k, i, fmt="q4_1": _exact_w(fmt, n, k, seed, i)
    if kind in ("proj", "prefill", "head"):
        m = c.get("m", c.get("t"))
        x = _randn((m, c["k"]), seed, 0, _DTYPE[c.get("x", "bf16")]).double()
        y = x @ w(c["n"], c["k"], 10, c.get("fmt", "q4_1")).T
        if kind == "head":
            return dict(ids=None, vals=None, logits=y)       # which of two near-equal logits leads is not a number
        return y + _randn((m, c["n"]), seed, 1).double() if c.get("residual") else y
    if kind == "ffn":
        x = _randn((c["m"], c["h"]), seed, 0).double()
        xn = _rms(x, _norm_weight(c["h"], seed, 1))
        h = _swiglu(xn @ w(c["f"], c["h"], 10).T, xn @ w(c["f"], c["h"], 11).T)
        return dict(h=h, y=x + h @ w(c["h"], c["f"], 12).T)
    if kind == "step":
        h, f, nq = c["h"], c["f"], c["nq"]
        x, qkv = _randn((1, h), seed, 0).double(), []
        for b in range(1000, 1000 + 10 * c["layers"], 10):
            qkv.append(_rms(x, _norm_weight(h, seed, b + 6)) @ w(nq, h, b).T)
            x = x + _randn((h,), seed, b + 5, torch.bfloat16).double() @ w(h, h, b + 1).T
            xn = _rms(x, _norm_weight(h, seed, b + 7))
            x = x + _swiglu(xn @ w(f, h, b + 2).T, xn @ w(f, h, b + 3).T) @ w(h, f, b + 4).T
        logits = _rms(x, _norm_weight(h, seed, 1)) @ w(c["vocab"], h, 10).T
        return dict(logits=logits, x=x, qkv0=qkv[0], qkv=torch.stack(qkv[1:]))
    if kind == "layer":
        h, f = c["h"], c["f"]
        x = _randn((c["t"], h), seed, 0).double()
        nw = [_norm_weight(h, seed, i) for i in (2, 3)]
        qkv = _rms(x, nw[0]) @ w(c["nq"], h, 10).T
        x_mid = x + _randn((c["t"], h), seed, 1, torch.bfloat16).double() @ w(h, h, 11).T
        xn = _rms(x_mid, nw[1])
        a = _swiglu(xn @ w(f, h, 12).T, xn @ w(f, h, 13).T)
        return dict(qkv=qkv, x_mid=x_mid, h=a, x_next=x_mid + a @ w(h, f, 14).T)
    t, h, f = c["t"], c["h"], c["f"]
    x = _randn((t, h), seed, 0, torch.bfloat16).double()
    ids, wts = _routes(c, seed)
    out = torch.zeros((t, h), dtype=torch.float64, device=DEV)
    for i in range(c["e"]):
        at, slot = (ids == i).nonzero(as_tuple=True)
        if at.numel():
            a = _swiglu(*(x[at] @ w(f, h, 1000 + 10 * i + j).T for j in (0, 1)))
            out.index_add_(0, at, (a @ w(h, f, 1000 + 10 * i + 2).T) * wts[at, slot].double()[:, None])
    if c["fs"]:
        a = _swiglu(*(x @ w(c["fs"], h, j).T for j in (10, 11)))
        sg = torch.sigmoid(x @ (_randn((h,), seed, 2, torch.bfloat16) / 16).double())
        out = _randn((t, h), seed, 1).double() + out + sg[:, None] * (a @ w(h, c["fs"], 12).T)
    return out
