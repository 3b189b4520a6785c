"""The performance cases of this library: the calls a program makes on one MI355X, at the sizes it makes them.

``listed()`` holds the fixed cases, ``draw(rng)`` more of the same kinds over the whole range of sizes.
A case is a dict of plain values; ``prepare`` makes its inputs on the GPU from a seed, ``run`` makes one
pass through the public entry points (``brimkern_amd.Context``), ``exact`` computes the same outputs in
64 bits with plain torch. Weights are drawn normal and encoded into the ``.brik`` planes, activations
are normal with a gain per channel, as the layers meet them. Kinds:

``gemv``     one quantized matrix times one row: a single projection while decoding
``layer``    the matmul side of one decoder layer while decoding: four fused plans
``head``     the LM head of one row, then softcap, repetition penalty and top-k on its logits
``matmul``   2 rows and more, q8 / q4 / q3 or f16 weights: batched decoding, then prefill
``moe``      the three expert-grouped projections of a mixture-of-experts layer
``conv``     a convolution with a quantized weight, as an image model runs it
``convert``  a tensor from one quantized format to another, as the model converter does
"""
import math

import numpy as np
import torch

from brimkern_amd import Context

DEV = "cuda:0"
LEVELS = {"q8": 127, "q4": 15, "q3": 7}
LARGEST = 4096 * 9728 * 2560          # multiply-adds of the largest listed case

_context = None


def context():
    """The one library context of the process (a program keeps it for its lifetime)."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def listed():
    return [
        # the smallest: one decoder layer of a 0.5B model per token, four launches of little work each
        {"name": "decode_layer_q8_small", "kind": "layer", "fmt": "q8", "d": 896, "qd": 896, "kvd": 128, "ffn": 4864,
         "gelu": False},
        # one Qwen3-4B decoder layer per token
        {"name": "decode_layer_q4", "kind": "layer", "fmt": "q4", "d": 2560, "qd": 4096, "kvd": 1024, "ffn": 9728,
         "gelu": False},
        # its LM head and sampling pre-work, once per token
        {"name": "decode_head_q3", "kind": "head", "fmt": "q3", "K": 2560, "N": 151936, "recent": 64,
         "penalty": 1.1, "softcap": 30.0, "k": 64},
        # eight sequences decoded together, or a speculative draft of eight tokens
        {"name": "batch_q4_8x2560x9728", "kind": "matmul", "fmt": "q4", "M": 8, "K": 2560, "N": 9728},
        # a batch of 33 sequences through a q8 down projection
        {"name": "batch_q8_33x9728x2560", "kind": "matmul", "fmt": "q8", "M": 33, "K": 9728, "N": 2560},
        # a 512-token prompt through gate / up
        {"name": "prefill_q4_512x2560x9728", "kind": "matmul", "fmt": "q4", "M": 512, "K": 2560, "N": 9728},
        # an odd prompt length through a q3 query projection
        {"name": "prefill_q3_777x2560x4096", "kind": "matmul", "fmt": "q3", "M": 777, "K": 2560, "N": 4096},
        # a prompt of 4096 tokens through the down projection: the largest
        {"name": "prefill_q4_4096x9728x2560", "kind": "matmul", "fmt": "q4", "M": 4096, "K": 9728, "N": 2560},
        # the same kind of projection with its weight kept in f16
        {"name": "prefill_f16_512x2560x9728", "kind": "matmul", "fmt": "f16", "M": 512, "K": 2560, "N": 9728},
        # a mixture-of-experts layer: 256 tokens, 8 of 64 experts each
        {"name": "moe_q4_256x64e", "kind": "moe", "fmt": "q4", "tokens": 256, "experts": 64, "topk": 8, "H": 2048,
         "F": 768},
        # a 3x3 convolution of a diffusion UNet block
        {"name": "conv_q4_320x64x64_k3", "kind": "conv", "fmt": "q4", "Cin": 320, "H": 64, "W": 64, "Cout": 320,
         "ks": 3, "stride": 1, "pad": 1, "bias": True},
        # one tensor of a q8 model converted to q4
        {"name": "convert_q8_q4_9728x2560", "kind": "convert", "fmt": "q8", "to": "q4", "N": 9728, "K": 2560},
    ]


def _log(rng, lo, hi, unit=1):
    """A whole multiple of ``unit`` in [lo, hi], even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v))) // unit * unit


def draw(rng):
    kind = rng.choice(["gemv", "layer", "head", "matmul", "matmul", "matmul", "matmul", "moe", "conv", "convert"])
    fmt = rng.choice(["q8", "q4", "q4", "q3"])
    if kind == "gemv":
        return {"kind": kind, "fmt": fmt, "K": _log(rng, 256, 9728, 32), "N": _log(rng, 256, 24000)}
    if kind == "layer":
        return {"kind": kind, "fmt": fmt, "d": _log(rng, 512, 4096, 32), "qd": _log(rng, 512, 4096, 32),
                "kvd": _log(rng, 128, 1024), "ffn": _log(rng, 1024, 12288, 32), "gelu": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "fmt": fmt, "K": _log(rng, 512, 2560, 32), "N": _log(rng, 24000, 151936),
                "recent": rng.randint(0, 256), "penalty": rng.choice([1.0, 1.1, 1.3]),
                "softcap": rng.choice([0.0, 30.0]), "k": rng.randint(1, 64)}
    if kind == "matmul":
        fmt = rng.choice(["q8", "q4", "q4", "q3", "f16"])
        K, N = _log(rng, 256, 9728, 8 if fmt == "f16" and rng.random() < 0.25 else 32), _log(rng, 256, 16384)
        return {"kind": kind, "fmt": fmt, "M": min(_log(rng, 2, 4096), LARGEST // (K * N)), "K": K, "N": N}
    if kind == "moe":
        E = rng.choice([8, 16, 32, 64])
        return {"kind": kind, "fmt": "q4", "tokens": _log(rng, 4, 1024), "experts": E, "topk": rng.randint(1, 8),
                "H": _log(rng, 256, 2048, 32), "F": _log(rng, 256, 2048, 32)}
    if kind == "conv":
        ks = rng.choice([1, 3, 3, 5])
        return {"kind": kind, "fmt": rng.choice(["q8", "q4"]), "Cin": _log(rng, 32, 640, 32),
                "H": _log(rng, 8, 96), "W": _log(rng, 8, 96), "Cout": _log(rng, 16, 640), "ks": ks,
                "stride": rng.choice([1, 1, 2]), "pad": ks // 2, "bias": rng.random() < 0.5}
    return {"kind": kind, "fmt": fmt, "to": rng.choice([f for f in ("q8", "q4", "q3") if f != fmt]),
            "N": _log(rng, 256, 16384), "K": _log(rng, 256, 9728, 32)}


# ---- inputs --------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rows(g, M, K):
    """Activations [M, K]: normal, with a log-normal gain per channel."""
    gain = torch.exp(0.4 * torch.randn(K, generator=g, device=DEV))
    return torch.randn(M, K, generator=g, device=DEV) * gain


def _halves(v):
    return v.to(torch.float16)


def encode(fmt, w):
    """Planes of a flat f32 tensor (whole groups of 32): q8 (codes, sc), q4 (nib, sc, mn), q3 (lo, hi,
    sc, mn); f16 just the halves."""
    if fmt == "f16":
        return (_halves(w),)
    gr = w.view(-1, 32)
    if fmt == "q8":
        sc = _halves(gr.abs().amax(1) / 127).clamp_min(6.2e-5)
        return torch.round(gr / sc.float()[:, None]).clamp_(-127, 127).to(torch.int8).view(-1), sc
    L = LEVELS[fmt]
    mn = _halves(gr.amin(1))
    sc = _halves((gr.amax(1) - gr.amin(1)) / L).clamp_min(6.2e-5)
    q = torch.round((gr - mn.float()[:, None]) / sc.float()[:, None]).clamp_(0, L).to(torch.uint8).view(-1)
    if fmt == "q4":
        q = q.view(-1, 2)
        return q[:, 0] | (q[:, 1] << 4), sc, mn

    def fields(v, count, bits):          # `count` fields of `bits` bits per 32-bit word, the first lowest
        per = 8 // bits
        v = v.view(-1, per)
        byte = v[:, 0].clone()
        for j in range(1, per):
            byte |= v[:, j] << (bits * j)
        assert count == 4 * per
        return byte.view(torch.int32)
    return fields(q & 3, 16, 2), fields(q >> 2, 32, 1), sc, mn


def decode(fmt, planes):
    """The f64 values of the planes of :func:`encode`, flat."""
    if fmt == "f16":
        return planes[0].double().view(-1)
    if fmt == "q8":
        codes, sc = planes
        return (codes.view(-1, 32).double() * sc.double()[:, None]).view(-1)
    if fmt == "q4":
        nib, sc, mn = planes
        q = torch.stack((nib & 15, nib >> 4), 1)
    else:
        lo, hi, sc, mn = planes
        q = torch.stack([(lo.view(torch.uint8) >> (2 * j)) & 3 for j in range(4)], 1).view(-1)
        q = q | (torch.stack([(hi.view(torch.uint8) >> j) & 1 for j in range(8)], 1).view(-1) << 2)
    return (q.view(-1, 32).double() * sc.double()[:, None] + mn.double()[:, None]).view(-1)


def _weight(g, fmt, N, K):
    return encode(fmt, (torch.randn(N * K, generator=g, device=DEV) * (1.0 / math.sqrt(K))))


def _out(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _route(g, tokens, experts, topk):
    """The rows of every expert, tokens in order within one, and the experts' offsets."""
    top = torch.randn(tokens, experts, generator=g, device=DEV).topk(topk, 1).indices.view(-1)
    order = torch.sort(top, stable=True).indices
    off = torch.zeros(experts + 1, dtype=torch.int32, device=DEV)
    off[1:] = torch.bincount(top, minlength=experts).cumsum(0)
    return order // topk, off


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, c, kind, fmt = _gen(seed), case, case["kind"], case["fmt"]
    if kind in ("gemv", "head", "matmul"):
        s = {"x": _rows(g, c.get("M", 1), c["K"]), "w": _weight(g, fmt, c["N"], c["K"])}
        if kind == "head":
            s["recent"] = torch.randperm(c["N"], generator=g, device=DEV)[:c["recent"]].to(torch.int32)
        return s
    if kind == "layer":
        d, qd, kvd, ffn = c["d"], c["qd"], c["kvd"], c["ffn"]
        s = {"x": _rows(g, 1, d), "attn": _rows(g, 1, qd)}
        for n in ("an", "fn"):
            s[n] = 1 + 0.1 * torch.randn(d, generator=g, device=DEV)
        for n, N, K in (("q", qd, d), ("k", kvd, d), ("v", kvd, d), ("o", d, qd), ("gate", ffn, d), ("up", ffn, d),
                        ("down", d, ffn)):
            s["w" + n] = _weight(g, fmt, N, K)
        return s
    if kind == "moe":
        rows, off = _route(g, c["tokens"], c["experts"], min(c["topk"], c["experts"]))
        H, F, E = c["H"], c["F"], c["experts"]
        s = {"off": off, "x": _rows(g, c["tokens"], H)[rows].contiguous(), "a": _rows(g, rows.numel(), F)}
        for n, N, K in (("gate", F, H), ("up", F, H), ("down", H, F)):
            s["w" + n] = _weight(g, fmt, E * N, K)
        return s
    if kind == "conv":
        s = {"x": torch.randn(c["Cin"], c["H"], c["W"], generator=g, device=DEV),
             "w": _weight(g, fmt, c["Cout"], c["Cin"] * c["ks"] ** 2)}
        s["b"] = torch.randn(c["Cout"], generator=g, device=DEV) if c["bias"] else None
        return s
    return {"w": _weight(g, fmt, c["N"], c["K"])}


def _at(t):
    return t.data_ptr() if t is not None and t.numel() else None


class State(dict):
    """What a program holds for its calls: buffers, and the plans it made of them."""

    def __del__(self):
        for p in self.get("plans", ()):
            p.destroy()


def prepare(case, seed):
    ctx, c, kind, fmt = context(), case, case["kind"], case["fmt"]
    s = State(_inputs(case, seed), case=dict(case))
    if kind in ("gemv", "head", "matmul"):
        s["y"] = _out(c.get("M", 1), c["N"])
        s["p"] = [_at(p) for p in s["w"]]
        if kind == "head":
            s["ids"], s["vals"] = _out(c["k"], dtype=torch.int32), _out(c["k"])
    elif kind == "layer":
        d, qd, kvd, ffn = c["d"], c["qd"], c["kvd"], c["ffn"]
        for n, size in (("q", qd), ("k", kvd), ("v", kvd), ("h", d), ("gate", ffn), ("up", ffn), ("y", d)):
            s["y" + n] = _out(size)

        def job(n, x, y, K, **fused):
            p = [_at(t) for t in s["w" + n]]
            planes = {"q8": ("p0", "sc"), "q4": ("p0", "sc", "mn"), "q3": ("p0", "p1", "sc", "mn")}[fmt]
            return dict(zip(planes, p), x=_at(x), y=_at(y), K=K, N=y.numel(), **fused)
        norm, ffn_norm = dict(norm_w=_at(s["an"]), eps=1e-6), dict(norm_w=_at(s["fn"]), eps=1e-6)
        s["plans"] = [
            ctx.gemv_plan(fmt, [job(n, s["x"], s["y" + n], d, **norm) for n in ("q", "k", "v")]),
            ctx.gemv_plan(fmt, [job("o", s["attn"], s["yh"], qd, res=_at(s["x"]))]),
            *ctx.gemv_plan_glu(fmt, job("gate", s["yh"], s["ygate"], d, **ffn_norm),
                               job("up", s["yh"], s["yup"], d, **ffn_norm),
                               job("down", s["yup"], s["yy"], ffn, gate=_at(s["ygate"]), res=_at(s["yh"]),
                                   gelu=c["gelu"]))]
    elif kind == "moe":
        R = s["x"].shape[0]
        s["yg"], s["yu"], s["yd"] = _out(R, c["F"]), _out(R, c["F"]), _out(R, c["H"])
        for n in ("gate", "up", "down"):
            s["p" + n] = [_at(p) for p in s["w" + n]]
    elif kind == "conv":
        oh, ow = _conv_out(c)
        s["y"], s["p"] = _out(c["Cout"], oh, ow), [_at(p) for p in s["w"]]
    else:
        n = c["N"] * c["K"]
        s["f32"] = _out(n)
        s["to"] = _planes(c["to"], n)
        s["p"], s["q"] = [_at(p) for p in s["w"]], [_at(p) for p in s["to"]]
    return s


def _planes(fmt, n):
    half = [_out(n // 32, dtype=torch.int16) for _ in range(1 if fmt == "q8" else 2)]
    if fmt == "q8":
        return [_out(n, dtype=torch.int8), *half]
    if fmt == "q4":
        return [_out(n // 2, dtype=torch.uint8), *half]
    return [_out(n // 16, dtype=torch.int32), _out(n // 32, dtype=torch.int32), *half]


def _conv_out(c):
    return tuple((c[a] + 2 * c["pad"] - c["ks"]) // c["stride"] + 1 for a in ("H", "W"))


# ---- one pass ------------------------------------------------------------------------------------


def run(s):
    ctx, c = context(), s["case"]
    kind, fmt = c["kind"], c["fmt"]
    if kind == "gemv" or kind == "matmul":
        name = "matmul_t_f16w" if fmt == "f16" else "matmul_t_" + fmt
        getattr(ctx, name)(_at(s["x"]), *s["p"], _at(s["y"]), c.get("M", 1), c["K"], c["N"])
        return s["y"]
    if kind == "layer":
        for p in s["plans"]:
            p.run()
        return {n: s["y" + n] for n in ("q", "k", "v", "h", "gate", "up", "y")}
    if kind == "head":
        getattr(ctx, "matmul_t_" + fmt)(_at(s["x"]), *s["p"], _at(s["y"]), 1, c["K"], c["N"])
        ctx.logits_topk(_at(s["y"]), c["N"], _at(s["recent"]), c["recent"], c["penalty"], c["softcap"], c["k"],
                        _at(s["ids"]), _at(s["vals"]))
        return {"logits": s["y"], "ids": s["ids"], "vals": s["vals"]}
    if kind == "moe":
        E, R, H, F = c["experts"], s["x"].shape[0], c["H"], c["F"]
        ctx.moe_matmul_t_q4_x2(_at(s["x"]), _at(s["off"]), s["pgate"], _at(s["yg"]), s["pup"], _at(s["yu"]), E, R, H, F)
        ctx.moe_matmul_t_q4(_at(s["a"]), _at(s["off"]), *s["pdown"], _at(s["yd"]), E, R, F, H)
        return {"gate": s["yg"], "up": s["yu"], "down": s["yd"]}
    if kind == "conv":
        ctx.conv2d(fmt, _at(s["x"]), s["p"], _at(s["b"]), _at(s["y"]), c["Cin"], c["H"], c["W"], c["Cout"], c["ks"],
                   c["ks"], c["stride"], c["pad"])
        return s["y"]
    n = c["N"] * c["K"]
    getattr(ctx, "dequant_" + fmt)(*s["p"], _at(s["f32"]), n)
    ctx.quantize(c["to"], _at(s["f32"]), s["q"], n)
    return {"f32": s["f32"], "planes": list(s["to"])}


# ---- what a pass cannot do without ---------------------------------------------------------------


def _wbytes(fmt, n):
    return {"q8": n + n // 16, "q4": n // 2 + n // 8, "q3": n * 3 // 8 + n // 8, "f16": 2 * n}[fmt]


def work(case):
    c, kind, fmt = case, case["kind"], case["fmt"]
    if kind in ("gemv", "head", "matmul"):
        M, K, N = c.get("M", 1), c["K"], c["N"]
        return {"bytes": _wbytes(fmt, N * K) + 4 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "layer":
        d, qd, kvd, ffn = c["d"], c["qd"], c["kvd"], c["ffn"]
        n = d * (2 * qd + 2 * kvd + 3 * ffn)
        return {"bytes": _wbytes(fmt, n) + 4 * (6 * d + 2 * qd + 2 * kvd + 2 * ffn), "flops": 2 * n}
    if kind == "moe":
        R, E, H, F = c["tokens"] * min(c["topk"], c["experts"]), c["experts"], c["H"], c["F"]
        used = min(E, R) * 3 * H * F                   # experts that no row is routed to are not read
        return {"bytes": _wbytes(fmt, used) + 4 * R * (2 * H + 3 * F), "flops": 6 * R * H * F}
    if kind == "conv":
        oh, ow = _conv_out(c)
        n = c["Cout"] * c["Cin"] * c["ks"] ** 2
        return {"bytes": _wbytes(fmt, n) + 4 * (c["Cin"] * c["H"] * c["W"] + c["Cout"] * (oh * ow + 1)),
                "flops": 2 * n * oh * ow}
    n = c["N"] * c["K"]
    return {"bytes": _wbytes(fmt, n) + 4 * n + _wbytes(c["to"], n), "flops": 4 * n}


def tolerance(case):
    """One row: x in 24-bit block floating point and f32 sums, up to 1.0e-6 off 64 bits. More rows, experts
    and convolutions: f16 operands with f32 sums (11-bit significands on both sides), up to 2.9e-4 off.
    Conversions are exact."""
    if case["kind"] == "convert":
        return "exact"
    if case["kind"] in ("gemv", "layer", "head"):
        return {"rel": 4e-6}
    return {"rel": 1.2e-3, "max": 0.01}


def exact(case, seed):
    c, kind, fmt = case, case["kind"], case["fmt"]
    s = _inputs(case, seed)

    def mm(x, w, N, K):
        return x.double() @ decode(fmt, w).view(N, K).t()
    if kind in ("gemv", "matmul"):
        return mm(s["x"], s["w"], c["N"], c["K"])
    if kind == "head":
        y = mm(s["x"], s["w"], c["N"], c["K"])
        if c["softcap"] > 0:
            y = c["softcap"] * torch.tanh(y / c["softcap"])
        if c["penalty"] != 1 and c["recent"]:
            at = s["recent"].long()
            y[0, at] = torch.where(y[0, at] > 0, y[0, at] / c["penalty"], y[0, at] * c["penalty"])
        return {"logits": y, "ids": None, "vals": y[0].topk(c["k"]).values}
    if kind == "layer":
        d, qd, kvd, ffn = c["d"], c["qd"], c["kvd"], c["ffn"]

        def norm(v, w):
            return v / torch.sqrt((v * v).mean() + float(np.float32(1e-6))) * w.double()
        x = s["x"].double()
        n = norm(x, s["an"])
        r = {k: mm(n, s["w" + k], N, d).view(-1) for k, N in (("q", qd), ("k", kvd), ("v", kvd))}
        h = x + mm(s["attn"], s["wo"], d, qd)
        m = norm(h, s["fn"])
        gate, up = mm(m, s["wgate"], ffn, d), mm(m, s["wup"], ffn, d)
        act = torch.nn.functional.gelu(gate, approximate="tanh") if c["gelu"] else torch.nn.functional.silu(gate)
        y = h + mm(act * up, s["wdown"], d, ffn)
        return dict(r, h=h.view(-1), gate=gate.view(-1), up=up.view(-1), y=y.view(-1))
    if kind == "moe":
        off, E, H, F = s["off"].tolist(), c["experts"], c["H"], c["F"]

        def grouped(x, w, N, K):
            w = decode(fmt, w).view(E, N, K)
            return torch.cat([x[off[e]:off[e + 1]].double() @ w[e].t() for e in range(E)])
        return {"gate": grouped(s["x"], s["wgate"], F, H), "up": grouped(s["x"], s["wup"], F, H),
                "down": grouped(s["a"], s["wdown"], H, F)}
    if kind == "conv":
        # unfolded to a product: the convolution itself has no 64-bit form on every library build
        w = decode(fmt, s["w"]).view(c["Cout"], -1)
        cols = torch.nn.functional.unfold(s["x"].double()[None], c["ks"], padding=c["pad"], stride=c["stride"])[0]
        y = w @ cols
        if s["b"] is not None:
            y = y + s["b"].double()[:, None]
        return y.view(c["Cout"], *_conv_out(c))
    return {"f32": decode(fmt, s["w"]), "planes": [None] * (4 if c["to"] == "q3" else 3 if c["to"] == "q4" else 2)}
