"""Performance cases of the MoE expert path and the steps around it.

Each case is one pass of work that a program built on the library has it do:
the norm of one token, a matvec, one expert called with host slices, decode
steps of MoE layers, chunks of a prompt, a sequence through an attention
block, a re-quantization.  Sizes are those of the repository's benchmark and
tests (Qwen3-30B-A3B, Mixtral-8x7B and Qwen3-235B-A22B shapes, the 4096 x
4096 kernel benchmark) with token counts and lengths off the tuned ones.

Device buffers are torch tensors; every call goes through the C ABI
(include/hale_moe.h) on one context, whose stream the caller's device-wide
synchronization covers.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hale-token_amd"))

import hale_moe as H  # noqa: E402

BLOCK = {"q8_0": 34, "q4_0": 18}  # bytes per 32 weights
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_CTX = None


def context():
    """The program's one context, made at first use."""
    global _CTX
    if _CTX is None:
        _CTX = H.Context(0)
    return _CTX


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # the residual add and RMSNorm in front of every block of a decode
        # step: the smallest call of a token
        dict(name="norm_1x2048", kind="norm", rows=1, n=2048, delta=True),
        # the reference's own kernel benchmark: WeightMatrix::matvec
        dict(name="matvec_q8_4096", kind="matvec", dtype="q8_0", rows=4096, cols=4096),
        # the vocabulary projection of every generated token
        dict(name="lm_head_bf16", kind="matvec", dtype="bf16", rows=151936, cols=2048),
        # Expert::forward on host slices, as a provider without the fused layer calls it
        dict(name="expert_host_q8", kind="expert", dtype="q8_0", hidden=2048, inter=768),
        # one token through MoE layers (norm and MoE of each), a captured decode step
        dict(name="decode_30b_q4_t1", kind="moe", dtype="q4_0", hidden=2048, inter=768, experts=128, top_k=8,
             tokens=1, layers=8, graph=True, norm=True),
        # the same for few, large experts
        dict(name="decode_mixtral_q4_t1", kind="moe", dtype="q4_0", hidden=4096, inter=14336, experts=8, top_k=2,
             tokens=1, layers=3, graph=True, norm=True),
        # a serving batch: 29 sequences' tokens per step
        dict(name="batch_30b_q4_t29", kind="moe", dtype="q4_0", hidden=2048, inter=768, experts=128, top_k=8,
             tokens=29, layers=4, graph=True, norm=True),
        # a prompt of ordinary length, q8_0
        dict(name="prefill_30b_q8_t500", kind="moe", dtype="q8_0", hidden=2048, inter=768, experts=128, top_k=8,
             tokens=500, layers=1, graph=False, norm=False),
        # the largest: a long prompt's chunk through a large layer
        dict(name="prefill_235b_q4_t2048", kind="moe", dtype="q4_0", hidden=4096, inter=1536, experts=128, top_k=8,
             tokens=2048, layers=1, graph=False, norm=False),
        # a long conversation through one attention block, token after token
        dict(name="attention_30b_bf16_3000", kind="attention", dtype="bf16", hidden=2048, heads=32, kv_heads=4,
             head_dim=128, qk_norm=True, length=3000),
        # a short one through a quantized block without QK-norm
        dict(name="attention_mixtral_q8_190", kind="attention", dtype="q8_0", hidden=4096, heads=32, kv_heads=8,
             head_dim=128, qk_norm=False, length=190),
        # quantizing weights and reading them back
        dict(name="encode_decode_q4", kind="convert", dtype="q4_0", rows=4096, cols=14336),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _mult(rng, lo, hi, step):
    return max(lo, min(hi, int(round(_log(rng, lo, hi) / step)) * step))


def draw(rng):
    """One more case, of the sizes between and around the listed ones."""
    kind = rng.choice(["norm", "matvec", "expert", "moe", "moe", "moe", "moe", "attention", "attention", "convert"])
    if kind == "norm":
        return dict(kind=kind, rows=int(_log(rng, 1, 1500)), n=int(_log(rng, 64, 8192)), delta=rng.random() < 0.5)
    if kind == "matvec":
        dtype = rng.choice(["f32", "f16", "bf16", "q8_0", "q4_0"])
        cols = _mult(rng, 256, 14336, 32)
        if dtype in SIZE:
            cols += rng.choice([0, 0, rng.randrange(1, 32)])  # rows that no vector width divides
        return dict(kind=kind, dtype=dtype, rows=int(_log(rng, 100, min(160000, 3e8 / cols))), cols=cols)
    if kind == "expert":
        return dict(kind=kind, dtype=rng.choice(["q8_0", "q4_0"]), hidden=_mult(rng, 512, 4096, 32),
                    inter=_mult(rng, 256, 8192, 32))
    if kind == "attention":
        hd = rng.choice([64, 80, 128, 128])
        kv = rng.choice([2, 4, 8])
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16", "q8_0", "q4_0"]), hidden=_mult(rng, 1024, 4096, 32),
                    heads=kv * rng.choice([1, 4, 8 if kv <= 4 else 4]), kv_heads=kv, head_dim=hd,
                    qk_norm=rng.random() < 0.5, length=int(_log(rng, 20, 2000)))
    if kind == "convert":
        return dict(kind=kind, dtype=rng.choice(["q8_0", "q4_0", "f16", "bf16"]), rows=int(_log(rng, 100, 4096)),
                    cols=_mult(rng, 512, 14336, 32))
    experts, top_k, h, i = rng.choice([(128, 8, 2048, 768), (64, 6, 2048, 1408), (16, 2, 4096, 6400),
                                       (8, 2, 4096, 14336), (128, 8, 4096, 1536), (60, 4, 2048, 1408)])
    tokens = max(1, int(_log(rng, 1, 1300)))
    small = tokens <= 64
    return dict(kind="moe", dtype=rng.choice(["q8_0", "q4_0"]), hidden=h - 32 * rng.choice([0, 0, 3]),
                inter=i - 32 * rng.choice([0, 0, 5]), experts=experts, top_k=top_k, tokens=tokens,
                layers=2 if small else 1, graph=small, norm=small)


# ---- inputs ----------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * std


def _blocks(g, rows, cols, dtype, std=0.02):
    """Quantized rows in the reference's block layout, as quantizing
    N(0, std^2) weights leaves them: uint8 [rows][cols / 32 * block bytes]."""
    nb = cols // 32
    top = 127.0 if dtype == "q8_0" else 8.0
    amax = torch.rand(rows, nb, device="cuda", generator=g) * 0.8 + 1.8  # of 32 values, in standard deviations
    codes = torch.randn(rows, nb, 32, device="cuda", generator=g)
    codes = (codes * (top / amax)[..., None]).round_()
    out = torch.empty(rows, nb, BLOCK[dtype], dtype=torch.uint8, device="cuda")
    out[..., :2] = (amax * (std / top)).half().view(torch.uint8).view(rows, nb, 2)
    if dtype == "q8_0":
        out[..., 2:] = codes.clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        n = (codes.clamp_(-8, 7) + 8).to(torch.uint8)
        out[..., 2:] = n[..., :16] | (n[..., 16:] << 4)
    return out.view(rows, nb * BLOCK[dtype])


def _weights(g, rows, cols, dtype, std=0.02):
    if dtype in BLOCK:
        return _blocks(g, rows, cols, dtype, std)
    return _normal(g, rows, cols, std=std).to(TORCH[dtype])


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _upload(t, rows, cols, dtype):
    """The device tensor as a resident matrix."""
    ctx, h = context(), C.c_void_p()
    torch.cuda.synchronize()
    ctx.check(H.lib().hale_matrix_upload_device(ctx.handle, H.parse_dtype(dtype), rows, cols, _ptr(t),
                                                t.numel() * t.element_size(), C.byref(h)), "upload")
    ctx.synchronize()
    return H.WeightMatrix(ctx, h, rows, cols, H.parse_dtype(dtype))


def _expert_chunk(case):
    """Experts generated together: at most about 200 M weights of a matrix."""
    return max(1, min(case["experts"], 200_000_000 // (case["hidden"] * case["inter"])))


def _moe_parts(case, seed):
    """Layer by layer: the router, then the chunks' gate, up and down bytes.
    The generator's order is the same for prepare() and exact()."""
    hid, inter, experts = case["hidden"], case["inter"], case["experts"]
    for layer in range(case["layers"]):
        g = _generator(seed * 1009 + layer)
        yield layer, "router", _normal(g, experts, hid, std=0.03)
        step = _expert_chunk(case)
        for e0 in range(0, experts, step):
            n = min(step, experts - e0)
            yield layer, "experts", (e0, n, _blocks(g, n * inter, hid, case["dtype"]),
                                     _blocks(g, n * inter, hid, case["dtype"]),
                                     _blocks(g, n * hid, inter, case["dtype"]))


def _moe_inputs(case, seed):
    """Hidden states [layers][tokens][H] with a component that all share, so
    that some experts are popular as in a trained model, and norm weights."""
    g = _generator(seed * 1009 + 777)
    shared = _normal(g, 1, 1, case["hidden"], std=0.45)
    x = _normal(g, case["layers"], case["tokens"], case["hidden"], std=0.9) + shared
    return x.contiguous(), _normal(g, case["layers"], case["hidden"], std=0.1) + 1.0


def _attention_inputs(case, seed):
    hid, nh, nkv, hd, n = (case[k] for k in ("hidden", "heads", "kv_heads", "head_dim", "length"))
    g = _generator(seed * 1009 + 5)
    std = 0.8 / math.sqrt(hid)
    mats = {"q": (nh * hd, hid), "k": (nkv * hd, hid), "v": (nkv * hd, hid), "o": (hid, nh * hd)}
    mats = {k: (_weights(g, r, c, case["dtype"], std if k != "o" else 0.8 / math.sqrt(nh * hd)), r, c)
            for k, (r, c) in mats.items()}
    x = _normal(g, n, hid)
    qn = kn = None
    if case["qk_norm"]:
        qn, kn = _normal(g, hd, std=0.1) + 1.0, _normal(g, hd, std=0.1) + 1.0
    angle = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * \
        torch.pow(1e6, -torch.arange(hd // 2, dtype=torch.float64, device="cuda") * 2 / hd)[None, :]
    return mats, x, qn, kn, angle.cos().float().contiguous(), angle.sin().float().contiguous()


EPS = 1e-6


def _norm_inputs(case, seed):
    g = _generator(seed)
    x = _normal(g, case["rows"], case["n"])
    return x, _normal(g, case["rows"], case["n"], std=0.05), _normal(g, case["n"], std=0.1) + 1.0


def _matvec_inputs(case, seed):
    g = _generator(seed)
    return _weights(g, case["rows"], case["cols"], case["dtype"]), _normal(g, case["cols"])


def _expert_inputs(case, seed):
    g = _generator(seed)
    hid, inter = case["hidden"], case["inter"]
    mats = [_blocks(g, r, c, case["dtype"]) for r, c in ((inter, hid), (inter, hid), (hid, inter))]
    return mats, _normal(g, hid).cpu().numpy()


def prepare(case, seed):
    ctx, lib, kind = context(), H.lib(), case["kind"]
    s = {"kind": kind, "ctx": ctx}
    if kind == "norm":
        x, delta, w = _norm_inputs(case, seed)
        out = torch.empty_like(x)
        s.update(out=(out, x) if case["delta"] else out, keep=(delta, w, x))
        s["call"] = (lib.hale_rms_norm_device, (ctx.handle, _ptr(x), _ptr(delta) if case["delta"] else None, _ptr(w),
                                                case["rows"], case["n"], EPS, _ptr(out)))
    elif kind == "matvec":
        w, x = _matvec_inputs(case, seed)
        m = _upload(w, case["rows"], case["cols"], case["dtype"])
        out = torch.empty(case["rows"], device="cuda")
        s.update(out=out, keep=(m, x))
        s["call"] = (lib.hale_matvec_device, (ctx.handle, m.handle, _ptr(x), _ptr(out)))
    elif kind == "expert":
        mats, x = _expert_inputs(case, seed)
        hid, inter = case["hidden"], case["inter"]
        s["expert"] = H.Expert(*(_upload(t, r, c, case["dtype"])
                                 for t, (r, c) in zip(mats, ((inter, hid), (inter, hid), (hid, inter)))))
        s.update(x=x, out=np.zeros(hid, dtype=np.float32))
    elif kind == "moe":
        _prepare_moe(s, case, seed)
    elif kind == "attention":
        mats, x, qn, kn, cos, sin = _attention_inputs(case, seed)
        m = [_upload(*mats[k], case["dtype"]) for k in "qkvo"]
        attn = H.Attention(ctx, *m, None if qn is None else qn.cpu().numpy(), None if kn is None else kn.cpu().numpy(),
                           case["heads"], case["kv_heads"], case["head_dim"], EPS, case["length"])
        out = torch.empty_like(x)
        n, hid, half = case["length"], case["hidden"], case["head_dim"] // 2
        s["calls"] = [(attn.handle, C.c_void_p(x.data_ptr() + 4 * hid * t), t, C.c_void_p(cos.data_ptr() + 4 * half * t),
                       C.c_void_p(sin.data_ptr() + 4 * half * t), C.c_void_p(out.data_ptr() + 4 * hid * t))
                      for t in range(n)]
        s.update(attn=attn, out=out, keep=(x, cos, sin))
    else:
        g = _generator(seed)
        rows, cols, dt = case["rows"], case["cols"], H.parse_dtype(case["dtype"])
        v = _normal(g, rows, cols, std=0.02)
        b = torch.empty(rows * H.row_bytes(dt, cols), dtype=torch.uint8, device="cuda")
        back = torch.empty_like(v)
        s.update(out=(b, back), keep=v)
        s["encode"] = (ctx.handle, dt, rows, cols, _ptr(v), _ptr(b))
        s["decode"] = (ctx.handle, dt, rows, cols, _ptr(b), _ptr(back))
    torch.cuda.synchronize()
    return s


def _prepare_moe(s, case, seed):
    ctx, hid, inter, k, n = s["ctx"], case["hidden"], case["inter"], case["top_k"], case["tokens"]
    layers = []
    for layer, what, part in _moe_parts(case, seed):
        if what == "router":
            router = _upload(part, case["experts"], hid, "f32")
            layers.append(H.MoeLayer(ctx, layer, case["experts"], hid, inter, case["dtype"], k, True, router))
        else:
            torch.cuda.synchronize()
            layers[-1].set_experts_device(part[0], part[1], *(t.data_ptr() for t in part[2:]))
            ctx.synchronize()
    x, w = _moe_inputs(case, seed)
    normed = torch.empty_like(x) if case["norm"] else x
    out = torch.empty_like(x)
    index = torch.empty(case["layers"], n, k, dtype=torch.int32, device="cuda")
    weight = torch.empty(case["layers"], n, k, device="cuda")
    lib = H.lib()
    norms = [(ctx.handle, _ptr(x[i]), None, _ptr(w[i]), n, hid, EPS, _ptr(normed[i])) for i in range(len(layers))]
    moes = [(m.handle, n, _ptr(normed[i]), None, _ptr(out[i]), _ptr(index[i]), _ptr(weight[i]))
            for i, m in enumerate(layers)]

    def step():
        for i in range(len(layers)):
            if case["norm"]:
                _ok(lib.hale_rms_norm_device(*norms[i]))
            _ok(lib.hale_moe_forward_device(*moes[i]))

    for m in layers:
        m.reserve(n)
    torch.cuda.synchronize()
    s.update(out=(out, index, weight), keep=(x, w, normed, layers), step=step)
    if case["graph"]:
        step()  # sizes what the layers grow at their first call
        ctx.synchronize()
        s["graph"] = ctx.capture(step)


def _ok(status):
    if status:
        context().check(status)


def run(s):
    kind = s["kind"]
    if kind in ("norm", "matvec"):
        fn, args = s["call"]
        _ok(fn(*args))
    elif kind == "expert":
        return s["expert"].forward(s["x"], s["out"])
    elif kind == "moe":
        if "graph" in s:
            s["graph"].launch()
        else:
            s["step"]()
    elif kind == "attention":
        fn = H.lib().hale_attention_forward_device
        s["attn"].reset()
        for args in s["calls"]:
            _ok(fn(*args))
    else:
        _ok(H.lib().hale_encode_rows_device(*s["encode"]))
        _ok(H.lib().hale_decode_rows_device(*s["decode"]))
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------

def _bytes_of(rows, cols, dtype):
    return rows * (cols // 32 * BLOCK[dtype] if dtype in BLOCK else cols * SIZE[dtype])


def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["rows"] * case["n"]
        return {"bytes": 4 * (n * (4 if case["delta"] else 2) + case["n"]), "flops": 4 * n}
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": _bytes_of(r, c, case["dtype"]) + 4 * (r + c), "flops": 2 * r * c}
    if kind == "expert":
        h, i = case["hidden"], case["inter"]
        return {"bytes": 2 * _bytes_of(i, h, case["dtype"]) + _bytes_of(h, i, case["dtype"]) + 8 * h, "flops": 6 * h * i}
    if kind == "moe":
        h, i, e, k, n = (case[f] for f in ("hidden", "inter", "experts", "top_k", "tokens"))
        touched = min(e, k) if n == 1 else e * (1 - (1 - k / e) ** n)  # experts of n tokens' routes
        expert = 2 * _bytes_of(i, h, case["dtype"]) + _bytes_of(h, i, case["dtype"])
        acts = 4 * n * h * (4 if case["norm"] else 2) + 8 * n * k
        return {"bytes": case["layers"] * (touched * expert + 4 * e * h + acts),
                "flops": case["layers"] * n * (6 * k * h * i + 2 * e * h)}
    if kind == "attention":
        h, q, kv, n = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["length"]
        mats = 2 * _bytes_of(q, h, case["dtype"]) + 2 * _bytes_of(kv, h, case["dtype"])
        return {"bytes": n * (mats + 8 * h) + 4 * kv * n * (n + 1), "flops": n * (4 * h * q + 4 * h * kv) + 2 * n * (n + 1) * q}
    n = case["rows"] * case["cols"]
    return {"bytes": 8 * n + 2 * _bytes_of(case["rows"], case["cols"], case["dtype"]), "flops": 2 * n}


def tolerance(case):
    """About four times the error against 64 bits that the path shows.  Where
    activations are rounded to 8 bits between two products, a value at a
    rounding border moves by a whole code: most of what those cases allow."""
    kind, quantized = case["kind"], case["dtype"] in BLOCK if "dtype" in case else False
    if kind == "convert":
        return "exact"  # codes are whole numbers; decoding is one product
    if kind == "norm":
        return {"rel": 7e-7, "max": 5e-6}
    if kind == "matvec":
        return {"rel": 1.5e-6, "max": 2e-5}
    if kind == "attention":
        return {"rel": 3e-3, "max": 0.05} if quantized else {"rel": 4e-6, "max": 1e-4}
    return {"rel": 1e-3, "max": 0.1, "differ": 5e-4}


# ---- the same in 64 bits -----------------------------------------------------

def _decode64(b, rows, cols, dtype):
    if dtype not in BLOCK:
        return b.double()
    b = b.view(rows, cols // 32, BLOCK[dtype])
    scale = b[..., :2].contiguous().view(torch.float16).double()
    if dtype == "q8_0":
        q = b[..., 2:].contiguous().view(torch.int8).double()
    else:
        q = torch.cat((b[..., 2:] & 15, b[..., 2:] >> 4), dim=-1).double() - 8
    return (q * scale).view(rows, cols)


def _act64(x, dtype):
    """The activation as a quantized matrix's product takes it: 8-bit codes
    per block of 32, the scale of the block's largest value."""
    if dtype not in BLOCK:
        return x
    v = x.reshape(*x.shape[:-1], -1, 32)
    scale = v.abs().amax(-1, keepdim=True) / 127
    t = torch.where(scale > 0, v / scale, torch.zeros_like(v))
    t = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (t.clamp(-128, 127) * scale).reshape(x.shape)


def _product64(b, rows, cols, dtype, x):
    """x [..][cols] times the matrix of the rows `b`, in slices of its rows."""
    x, got, step = _act64(x, dtype), [], max(1, 100_000_000 // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        got.append(x @ _decode64(b[r:r + n], n, cols, dtype).t())
    return torch.cat(got, dim=-1)


def _norm64(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w


def _expert64(gate, up, down, hid, inter, dtype, x):
    g, u = _product64(gate, inter, hid, dtype, x), _product64(up, inter, hid, dtype, x)
    return _product64(down, hid, inter, dtype, g / (1 + (-g).exp()) * u)


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        x, delta, w = _norm_inputs(case, seed)
        x = x.double() + (delta.double() if case["delta"] else 0)
        out = _norm64(x, w.double())
        return (out, x) if case["delta"] else out
    if kind == "matvec":
        w, x = _matvec_inputs(case, seed)
        return _product64(w, case["rows"], case["cols"], case["dtype"], x.double()[None])[0]
    if kind == "expert":
        mats, x = _expert_inputs(case, seed)
        x = torch.from_numpy(x).cuda().double()[None]
        return _expert64(*mats, case["hidden"], case["inter"], case["dtype"], x)[0].cpu().numpy()
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "attention":
        return _exact_attention(case, seed)
    return None  # compared byte for byte


def _exact_moe(case, seed):
    hid, inter, k = case["hidden"], case["inter"], case["top_k"]
    x, w = _moe_inputs(case, seed)
    x = x.double()
    if case["norm"]:
        x = _norm64(x, w.double()[:, None])
    out, weights = torch.zeros_like(x), []
    index = None
    for layer, what, part in _moe_parts(case, seed):
        if what == "router":
            p = (x[layer] @ part.double().t()).softmax(-1)
            top, index = p.topk(k, dim=-1)
            weights.append(top / top.sum(-1, keepdim=True))
            continue
        e0, n, gate, up, down = part
        for e in range(n):
            tok, slot = (index == e0 + e).nonzero(as_tuple=True)
            if tok.numel():
                y = _expert64(gate[e * inter:(e + 1) * inter], up[e * inter:(e + 1) * inter], down[e * hid:(e + 1) * hid],
                              hid, inter, case["dtype"], x[layer][tok])
                out[layer].index_add_(0, tok, y * weights[layer][tok, slot][:, None])
    return out, None, torch.stack(weights)


def _exact_attention(case, seed):
    mats, x, qn, kn, cos, sin = _attention_inputs(case, seed)
    nh, nkv, hd, n = case["heads"], case["kv_heads"], case["head_dim"], case["length"]
    q, k, v = (_product64(*mats[m], case["dtype"], x.double()) for m in "qkv")
    q, k, v = q.view(n, nh, hd), k.view(n, nkv, hd), v.view(n, nkv, hd)
    if qn is not None:
        q, k = _norm64(q, qn.double()), _norm64(k, kn.double())
    c, s = cos.double()[:, None], sin.double()[:, None]

    def turn(t):
        a, b = t[..., :hd // 2], t[..., hd // 2:]
        return torch.cat((a * c - b * s, b * c + a * s), dim=-1)

    q, k = turn(q), turn(k)
    ctx = torch.empty_like(q)
    later = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for h in range(nh):
        kv = h // (nh // nkv)
        score = (q[:, h] @ k[:, kv].t().contiguous() / math.sqrt(hd)).masked_fill(later, -math.inf)
        ctx[:, h] = score.softmax(-1) @ v[:, kv].contiguous()
    return _product64(*mats["o"], case["dtype"], ctx.reshape(n, nh * hd))
