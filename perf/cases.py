"""Workloads of the quantized linear path: what a program serving a GGUF model asks of this library, as measurable cases.

Kinds of case (each a pass through public entry points on device tensors):
  matmul  kungfu_amd.matmul over a stack of `mats` weights of one shape (the same projection in successive decoder
          layers, so that a decode pass finds its weights in HBM and not in a cache)
  group   kungfu_amd.matmul_group: Q/K/V kept as separate tensors sharing one input
  norm    kungfu_amd.rms_norm_matmul: the norm in front of QKV or gate/up
  swiglu  kungfu_amd.gated_act_q8 on the fused gate/up rows, then the down product on the int8 rows
  layers  a token step through the linear layers of a few decoder layers: norm + QKV, O + residual, norm + gate/up,
          gated activation + down + residual
  moe     kungfu_amd.moe_ffn: the routed expert layer
"""
import math

import torch

import kungfu_amd as kf

TYPES = {"q8_0": kf.TYPE_Q8_0, "q4_K": kf.TYPE_Q4_K, "q5_K": kf.TYPE_Q5_K, "q6_K": kf.TYPE_Q6_K}
EPS = 1e-5
LARGEST_WEIGHTS = 8 * 3 * 4096 * 14336  # weights of the largest listed case (the eight experts)
LARGEST_MACS = 2048 * 4096 * 28672      # multiply-adds of the largest listed case (the gate/up prefill)


def listed():
    return [
        # Q/K/V of a small model at one token, biases on, an odd multiple of the block: launch latency and host path
        {"name": "decode_qkv_small_q8_0", "kind": "group", "ty": "q8_0", "rows": 1, "n_in": 1056, "outs": "1056,352,352", "bias": True},
        # one decoded token through three decoder layers of a Q4_K_M file (q6_K down projections)
        {"name": "decode_layers_q4_K_m", "kind": "layers", "ty": "q4_K", "ty_down": "q6_K", "rows": 1, "n_embd": 4096, "n_qkv": 6144, "n_ff": 14336, "layers": 3},
        # the output head of one token: the largest matrix of a model, q6_K in the common files
        {"name": "decode_head_q6_K", "kind": "matmul", "ty": "q6_K", "rows": 1, "n_in": 4096, "n_out": 128256, "mats": 1, "bias": False, "res": False},
        # eight rows: a speculative verification or eight requests decoded together, on the stacked gate/up matrix
        {"name": "batch8_gate_up_q4_K", "kind": "matmul", "ty": "q4_K", "rows": 8, "n_in": 4096, "n_out": 28672, "mats": 3, "bias": False, "res": False},
        # 24 rows, the wide-input projection in q5_K, with the residual added
        {"name": "batch24_down_q5_K", "kind": "matmul", "ty": "q5_K", "rows": 24, "n_in": 14336, "n_out": 4096, "mats": 4, "bias": False, "res": True},
        # 64 requests decoded together in q8_0
        {"name": "batch64_gate_q8_0", "kind": "matmul", "ty": "q8_0", "rows": 64, "n_in": 4096, "n_out": 14336, "mats": 3, "bias": False, "res": False},
        # a prompt of ordinary, ragged length through QKV with biases
        {"name": "prompt300_qkv_q4_K", "kind": "matmul", "ty": "q4_K", "rows": 300, "n_in": 4096, "n_out": 6144, "mats": 4, "bias": True, "res": False},
        # prefill of a long prompt: norm and the stacked gate/up matrix
        {"name": "prefill_norm_gate_up_q4_K", "kind": "norm", "ty": "q4_K", "rows": 2048, "n_in": 4096, "n_out": 28672},
        # prefill of a long prompt: the down projection in q8_0, residual added
        {"name": "prefill_down_q8_0", "kind": "matmul", "ty": "q8_0", "rows": 2048, "n_in": 14336, "n_out": 4096, "mats": 1, "bias": False, "res": True},
        # a ragged prompt through the gated activation and a q6_K down projection
        {"name": "prompt777_swiglu_down_q6_K", "kind": "swiglu", "ty": "q6_K", "rows": 777, "n_in": 14336, "n_out": 4096},
        # sixteen tokens, two of eight experts each
        {"name": "moe_decode16_q4_K", "kind": "moe", "ty": "q4_K", "rows": 16, "n_slots": 8, "n_used": 2, "n_embd": 4096, "n_ff": 14336},
        # a prompt of 512 tokens through the same experts
        {"name": "moe_prompt512_q4_K", "kind": "moe", "ty": "q4_K", "rows": 512, "n_slots": 8, "n_used": 2, "n_embd": 4096, "n_ff": 14336},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, ty, lo, hi):
    """Input columns: a whole number of the type's blocks."""
    block = 32 if ty == "q8_0" else 256
    return block * _log_int(rng, max(1, lo // block), hi // block)


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "matmul", "matmul", "group", "norm", "swiglu", "layers", "moe", "moe"])
    ty = rng.choice(["q4_K", "q4_K", "q8_0", "q5_K", "q6_K"])
    rows = _log_int(rng, 1, 2048)
    if kind == "matmul":
        n_in = _width(rng, ty, 1024, 14336)
        n_out = _log_int(rng, 500, 40000)
        n_out = max(256, min(n_out, LARGEST_MACS // (rows * n_in), LARGEST_WEIGHTS // n_in))
        mats = max(1, min(4, 300_000_000 // (n_in * n_out), LARGEST_MACS // (rows * n_in * n_out)))
        return {"kind": kind, "ty": ty, "rows": rows, "n_in": n_in, "n_out": n_out, "mats": mats, "bias": rng.random() < 0.3, "res": rng.random() < 0.3}
    if kind == "group":
        n_in = _width(rng, ty, 1024, 8192)
        head = 64 * _log_int(rng, 1, 32)
        rows = min(rows, 512)
        return {"kind": kind, "ty": ty, "rows": rows, "n_in": n_in, "outs": "%d,%d,%d" % (64 * _log_int(rng, 8, 128), head, head), "bias": rng.random() < 0.5}
    if kind == "norm":
        n_in = _width(rng, ty, 1024, 8192)
        n_out = min(_log_int(rng, 1000, 28672), LARGEST_MACS // (rows * n_in))
        return {"kind": kind, "ty": ty, "rows": rows, "n_in": n_in, "n_out": n_out}
    if kind == "swiglu":
        n_in = _width(rng, ty, 1024, 14336)
        return {"kind": kind, "ty": ty, "rows": rows, "n_in": n_in, "n_out": 32 * _log_int(rng, 32, 160)}
    if kind == "layers":
        ty = rng.choice(["q4_K", "q8_0", "q5_K"])
        ty_down = rng.choice([ty, "q6_K"])
        n_embd = 256 * _log_int(rng, 4, 20)
        n_ff = 256 * int(n_embd * rng.uniform(2.0, 3.5) / 256)
        return {"kind": kind, "ty": ty, "ty_down": ty_down, "rows": _log_int(rng, 1, 32), "n_embd": n_embd, "n_qkv": n_embd + 2 * 64 * rng.randint(2, 16),
                "n_ff": n_ff, "layers": 3}
    ty = rng.choice(["q4_K", "q4_K", "q8_0"])
    n_slots = rng.choice([4, 8, 16, 32, 64])
    n_used = rng.choice([1, 2, 2, 4])
    n_embd = 256 * _log_int(rng, 4, 16)
    n_ff = 256 * _log_int(rng, 2, 32)
    while n_slots * 3 * n_embd * n_ff > LARGEST_WEIGHTS:
        n_slots //= 2
    rows = max(1, min(_log_int(rng, 1, 512), LARGEST_MACS // (n_used * 3 * n_embd * n_ff)))
    return {"kind": "moe", "ty": ty, "rows": rows, "n_slots": n_slots, "n_used": min(n_used, n_slots), "n_embd": n_embd, "n_ff": n_ff}


# ------------------------------------------------------------------------------------------------ weights
# Valid block bytes of N(0, 0.02) weights, encoded on the device, and the values the blocks stand for in 64 bits.

def _f16_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).view(*v.shape, 2)


def _pack_scales(sc, mn):
    """The twelve bytes of eight 6-bit scales and mins (q4_K / q5_K)."""
    a = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    b = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    c = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return torch.cat([a, b, c], 1)


def _encode(ty, v):
    """v [blocks][block] f32 -> [blocks][bytes] uint8."""
    nb = v.shape[0]
    if ty == "q8_0":
        d = v.abs().amax(1, keepdim=True) / 127.0
        q = torch.round(v / d).to(torch.int8)
        return torch.cat([_f16_bytes(d).view(nb, 2), q.view(torch.uint8)], 1)
    if ty == "q6_K":
        g = v.view(nb, 16, 16)
        gs = g.abs().amax(2) / 31.0
        d = (gs.amax(1, keepdim=True) / 127.0).to(torch.float16).float()
        sc = torch.round(gs / d).clamp(1, 127)
        q = (torch.round(g / (d * sc).unsqueeze(2)).clamp(-32, 31) + 32).to(torch.uint8).view(nb, 2, 4, 32)
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2).view(nb, 128)
        qh = ((q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)).view(nb, 64)
        return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16_bytes(d).view(nb, 2)], 1)
    steps = 15 if ty == "q4_K" else 31
    g = v.view(nb, 8, 32)
    lo = g.amin(2).clamp(max=0.0)
    scale = (g.amax(2) - lo) / steps
    d = (scale.amax(1, keepdim=True) / 63.0).to(torch.float16).float()
    dmin = ((-lo).amax(1, keepdim=True) / 63.0).to(torch.float16).float()
    sc = torch.round(scale / d).clamp(1, 63)
    mn = torch.round(-lo / dmin).clamp(0, 63)
    q = torch.round((g + (dmin * mn).unsqueeze(2)) / (d * sc).unsqueeze(2)).clamp(0, steps).to(torch.uint8)
    head = torch.cat([_f16_bytes(d).view(nb, 2), _f16_bytes(dmin).view(nb, 2), _pack_scales(sc.to(torch.uint8), mn.to(torch.uint8))], 1)
    low = q & 15
    nib = (low[:, 0::2] | (low[:, 1::2] << 4)).reshape(nb, 128)
    if ty == "q4_K":
        return torch.cat([head, nib], 1)
    qh = torch.zeros(nb, 32, dtype=torch.uint8, device=v.device)
    for s in range(8):
        qh |= (q[:, s] >> 4) << s
    return torch.cat([head, qh, nib], 1)


def _f16_at(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _decode(ty, b):
    """b [blocks][bytes] uint8 -> [blocks][block] f64."""
    nb = b.shape[0]
    if ty == "q8_0":
        return b[:, 2:].contiguous().view(torch.int8).double() * _f16_at(b, 0)
    if ty == "q6_K":
        ql, qh = b[:, :128].view(nb, 2, 64), b[:, 128:192].reshape(nb, 2, 32)
        runs = []
        for k in range(4):
            low = (ql[:, :, 32 * (k & 1):32 * (k & 1) + 32] >> (4 * (k >> 1))) & 15
            runs.append(low | (((qh >> (2 * k)) & 3) << 4))
        q = torch.stack(runs, 2).reshape(nb, 16, 16).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (q * (sc * _f16_at(b, 208)).unsqueeze(2)).view(nb, 256)
    s = b[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double() * _f16_at(b, 0)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * _f16_at(b, 2)
    nib = b[:, -128:].reshape(nb, 4, 1, 32)
    q = torch.cat([nib & 15, nib >> 4], 2).reshape(nb, 8, 32)
    if ty == "q5_K":
        qh = b[:, 16:48].view(nb, 1, 32)
        q = q | (((qh >> torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)) & 1) << 4)
    return (q.double() * sc.unsqueeze(2) - mn.unsqueeze(2)).view(nb, 256)


CHUNK = 1 << 25  # weights handled at a time


def _block(ty):
    return kf.BLOCK[TYPES[ty]]


def _weights(gen, ty, n_out, n_in):
    block, size = _block(ty)
    out = torch.empty(n_out, n_in // block * size, dtype=torch.uint8, device="cuda")
    step = max(1, CHUNK // n_in)
    for at in range(0, n_out, step):
        r = min(step, n_out - at)
        v = torch.randn(r * n_in // block, block, device="cuda", generator=gen) * 0.02
        out[at:at + r] = _encode(ty, v).view(r, -1)
    return out


def _product64(ty, w, xq, n_in):
    """xq [rows][n_in] f64 (the rounded activations) times the decoded weights, in 64 bits."""
    block, size = _block(ty)
    n_out = w.shape[0]
    y = torch.empty(xq.shape[0], n_out, dtype=torch.float64, device="cuda")
    step = max(1, CHUNK // n_in)
    for at in range(0, n_out, step):
        r = min(step, n_out - at)
        d = _decode(ty, w[at:at + r].reshape(r * n_in // block, size)).view(r, n_in)
        y[:, at:at + r] = xq @ d.t()
    return y


# ------------------------------------------------------------------------------------------------ activations

def _rows(gen, rows, n):
    """Activation rows: normal values whose channels differ in size, as a decoder's residual stream has them."""
    ch = torch.exp(0.5 * torch.randn(n, device="cuda", generator=gen))
    return torch.randn(rows, n, device="cuda", generator=gen) * ch


def _rounded(ty, x):
    """The int8 rounding of f32 rows that the path is defined on (Q8_0 or Q8K activations), as f64 values."""
    x = x.float()
    rows, n = x.shape
    if ty == "q8_0":
        v = x.view(rows, n // 32, 32)
        d = v.abs().amax(2, keepdim=True) / torch.full((), 127.0, device=x.device)
        p = v * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
        q = torch.sign(p) * torch.floor(p.abs().double() + 0.5)
        return (q * d.to(torch.float16).double()).view(rows, n)
    v = x.view(rows, n // 256, 256)
    mx = v.gather(2, v.abs().argmax(2, keepdim=True))
    isc = torch.full((), -127.0, device=x.device) / mx
    q = torch.round(isc * v).clamp(max=127.0)
    q = torch.where(mx != 0, q, torch.zeros_like(q))
    d = torch.where(mx != 0, 1.0 / isc, torch.zeros_like(mx))
    return (q.double() * d.double()).view(rows, n)


def _norm64(x, w):
    """rms_norm of f32 rows: squares and sums in 64 bits, the stored values in 32, as the entry point states."""
    x = x.float()
    ss = ((x * x).double().sum(1, keepdim=True) / x.shape[1]).float()
    inv = (1.0 / (ss + torch.full((), EPS, device=x.device)).double().sqrt().float().double()).float()
    return (x * inv) * w


def _silu_mul(g, u):
    """silu(g) * u on f32 values: exp in 64 bits, the stored values in 32."""
    g, u = g.float(), u.float()
    e = torch.exp(-g.double()).float()
    return (g.double() / (1.0 + e).double()).float() * u


# ------------------------------------------------------------------------------------------------ the cases

def _split(case):
    return [int(v) for v in case["outs"].split(",")]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, ty, rows = case["kind"], case["ty"], case["rows"]
    s = {"case": dict(case), "ty": TYPES[ty]}

    def vec(n, scale=0.1):
        return torch.randn(n, device="cuda", generator=gen) * scale

    def buf(*shape):
        return torch.empty(*shape, device="cuda")

    if kind == "matmul":
        n_in, n_out = case["n_in"], case["n_out"]
        s["act"] = kf.alloc_act(rows, n_in)
        s["mats"] = [{"w": _weights(gen, ty, n_out, n_in), "x": _rows(gen, rows, n_in), "bias": vec(n_out) if case["bias"] else None,
                      "res": _rows(gen, rows, n_out) if case["res"] else None, "y": buf(rows, n_out)} for _ in range(case["mats"])]
    elif kind == "group":
        n_in, outs = case["n_in"], _split(case)
        s["act"], s["x"] = kf.alloc_act(rows, n_in), _rows(gen, rows, n_in)
        s["members"] = [(_weights(gen, ty, o, n_in), buf(rows, o), vec(o) if case["bias"] else None, None) for o in outs]
    elif kind == "norm":
        n_in, n_out = case["n_in"], case["n_out"]
        s.update(act=kf.alloc_act(rows, n_in), x=_rows(gen, rows, n_in), nw=1.0 + vec(n_in), w=_weights(gen, ty, n_out, n_in), y=buf(rows, n_out))
    elif kind == "swiglu":
        n_in, n_out = case["n_in"], case["n_out"]
        s.update(act=kf.alloc_act(rows, n_in), gu=_rows(gen, rows, 2 * n_in), w=_weights(gen, ty, n_out, n_in), res=_rows(gen, rows, n_out), y=buf(rows, n_out))
    elif kind == "layers":
        e, q, f = case["n_embd"], case["n_qkv"], case["n_ff"]
        s.update(act=kf.alloc_act(rows, e), fact=kf.alloc_act(rows, f), x=_rows(gen, rows, e))
        s["layers"] = [{"n1": 1.0 + vec(e), "n2": 1.0 + vec(e), "qkv": _weights(gen, ty, q, e), "o": _weights(gen, ty, e, e),
                        "gate_up": _weights(gen, ty, 2 * f, e), "down": _weights(gen, case["ty_down"], e, f), "y_qkv": buf(rows, q), "attn": buf(rows, e),
                        "h": buf(rows, e), "gu": buf(rows, 2 * f), "out": buf(rows, e)} for _ in range(case["layers"])]
    else:
        n, e, f, used = case["n_slots"], case["n_embd"], case["n_ff"], case["n_used"]
        sel = torch.rand(rows, n, device="cuda", generator=gen).argsort(1)[:, :used].to(torch.int32).contiguous()
        wts = torch.softmax(torch.randn(rows, used, device="cuda", generator=gen), 1)
        s.update(gate=_weights(gen, ty, n * f, e), up=_weights(gen, ty, n * f, e), down=_weights(gen, ty, n * e, f), x=_rows(gen, rows, e), sel=sel, wts=wts,
                 out=buf(rows, e), scratch=torch.empty(kf.moe_scratch_bytes(rows, used, e, f, n), dtype=torch.uint8, device="cuda"))
    return s


def _down(ty, w, act, y, rows, n, n_out, res):
    """The product on rows a producer has already quantized: the few-row product, past 64 rows the tile GEMM where the
    type takes the width."""
    fits = {"q8_0": n % 128 == 0, "q6_K": n % 2048 == 0}.get(ty, True)
    if rows > 64 and fits:
        kf.gemm_i8(TYPES[ty], w, act, y, rows, n, n_out, res=res)
    else:
        kf.gemv(TYPES[ty], w, act, y, rows, n, n_out, res=res)


def run(s):
    case, ty = s["case"], s["ty"]
    kind, rows = case["kind"], case["rows"]
    if kind == "matmul":
        for m in s["mats"]:
            kf.matmul(ty, m["w"], m["x"], s["act"], m["y"], case["n_out"], bias=m["bias"], res=m["res"])
        return [m["y"] for m in s["mats"]]
    if kind == "group":
        kf.matmul_group(ty, s["members"], s["x"], s["act"])
        return [m[1] for m in s["members"]]
    if kind == "norm":
        kf.rms_norm_matmul(ty, s["w"], s["x"], s["act"], s["y"], case["n_out"], norm_w=s["nw"], eps=EPS)
        return s["y"]
    if kind == "swiglu":
        n = case["n_in"]
        kf.gated_act_q8(s["gu"], s["gu"][:, n:], s["act"], kf.act_kind(ty), rows, n, 2 * n)
        _down(case["ty"], s["w"], s["act"], s["y"], rows, n, case["n_out"], s["res"])
        return s["y"]
    if kind == "layers":
        e, f, tyd = case["n_embd"], case["n_ff"], case["ty_down"]
        x, got = s["x"], []
        for L in s["layers"]:
            kf.rms_norm_matmul(ty, L["qkv"], x, s["act"], L["y_qkv"], case["n_qkv"], norm_w=L["n1"], eps=EPS)
            # the attention's place: the query columns go on to the output projection
            attn = L["y_qkv"] if case["n_qkv"] == e else L["attn"].copy_(L["y_qkv"][:, :e])
            kf.matmul(ty, L["o"], attn, s["act"], L["h"], e, res=x)
            kf.rms_norm_matmul(ty, L["gate_up"], L["h"], s["act"], L["gu"], 2 * f, norm_w=L["n2"], eps=EPS)
            kf.gated_act_q8(L["gu"], L["gu"][:, f:], s["fact"], kf.act_kind(TYPES[tyd]), rows, f, 2 * f)
            _down(tyd, L["down"], s["fact"], L["out"], rows, f, e, L["h"])
            x = L["out"]
            got += [L["y_qkv"], L["h"], L["gu"], x]
        return got
    kf.moe_ffn(ty, s["gate"], s["up"], s["down"], case["n_slots"], case["n_embd"], case["n_ff"], s["x"], s["sel"], s["wts"], s["out"], s["scratch"])
    return s["out"]


def exact(case, seed):
    s = prepare(case, seed)
    kind, ty, rows = case["kind"], case["ty"], case["rows"]

    def plus(y, bias, res):
        if bias is not None:
            y += bias.double()
        if res is not None:
            y += res.double()
        return y

    if kind == "matmul":
        return [plus(_product64(ty, m["w"], _rounded(ty, m["x"]), case["n_in"]), m["bias"], m["res"]) for m in s["mats"]]
    if kind == "group":
        xq = _rounded(ty, s["x"])
        return [plus(_product64(ty, m[0], xq, case["n_in"]), m[2], None) for m in s["members"]]
    if kind == "norm":
        return _product64(ty, s["w"], _rounded(ty, _norm64(s["x"], s["nw"])), case["n_in"])
    if kind == "swiglu":
        n = case["n_in"]
        return plus(_product64(ty, s["w"], _rounded(ty, _silu_mul(s["gu"][:, :n], s["gu"][:, n:])), n), None, s["res"])
    if kind == "layers":
        e, f, tyd = case["n_embd"], case["n_ff"], case["ty_down"]
        x, got = s["x"].double(), []
        for L in s["layers"]:
            qkv = _product64(ty, L["qkv"], _rounded(ty, _norm64(x, L["n1"])), e)
            h = _product64(ty, L["o"], _rounded(ty, qkv[:, :e].contiguous()), e) + x
            gu = _product64(ty, L["gate_up"], _rounded(ty, _norm64(h, L["n2"])), e)
            x = _product64(tyd, L["down"], _rounded(tyd, _silu_mul(gu[:, :f], gu[:, f:])), f) + h
            got += [qkv, h, gu, x]
        return got
    n, e, f = case["n_slots"], case["n_embd"], case["n_ff"]
    xq, sel, wts = _rounded(ty, s["x"]), s["sel"].long(), s["wts"].double()
    out = torch.zeros(rows, e, dtype=torch.float64, device="cuda")
    for k in range(n):
        r, j = (sel == k).nonzero(as_tuple=True)
        if r.numel() == 0:
            continue
        g = _product64(ty, s["gate"][k * f:(k + 1) * f], xq[r], e)
        u = _product64(ty, s["up"][k * f:(k + 1) * f], xq[r], e)
        y = _product64(ty, s["down"][k * e:(k + 1) * e], _rounded(ty, _silu_mul(g, u)), f)
        out.index_put_((r,), y * wts[r, j].unsqueeze(1), accumulate=True)
    return out


def work(case):
    kind, ty, rows = case["kind"], case["ty"], case["rows"]

    def mat(t, n_out, n_in):
        block, size = _block(t)
        return n_out * (n_in // block) * size

    def io(*cols):
        return 4 * rows * sum(cols)

    if kind == "matmul":
        n_in, n_out, mats = case["n_in"], case["n_out"], case["mats"]
        b = mat(ty, n_out, n_in) + io(n_in, n_out) + (4 * n_out if case["bias"] else 0) + (io(n_out) if case["res"] else 0)
        return {"bytes": mats * b, "flops": mats * 2 * rows * n_in * n_out}
    if kind == "group":
        n_out = sum(_split(case))
        return {"bytes": mat(ty, n_out, case["n_in"]) + io(case["n_in"], n_out) + (4 * n_out if case["bias"] else 0), "flops": 2 * rows * case["n_in"] * n_out}
    if kind == "norm":
        n_in, n_out = case["n_in"], case["n_out"]
        return {"bytes": mat(ty, n_out, n_in) + io(n_in, n_out) + 4 * n_in, "flops": 2 * rows * n_in * n_out}
    if kind == "swiglu":
        n_in, n_out = case["n_in"], case["n_out"]
        return {"bytes": mat(ty, n_out, n_in) + io(2 * n_in, n_out, n_out), "flops": 2 * rows * n_in * n_out}
    if kind == "layers":
        e, q, f = case["n_embd"], case["n_qkv"], case["n_ff"]
        w = mat(ty, q + e + 2 * f, e) + mat(case["ty_down"], e, f)
        return {"bytes": case["layers"] * (w + io(q, e, 2 * f, e) + 8 * e) + io(e), "flops": case["layers"] * 2 * rows * (e * (q + e + 2 * f) + e * f)}
    n, e, f, used = case["n_slots"], case["n_embd"], case["n_ff"], case["n_used"]
    touched = n * (1.0 - (1.0 - used / n) ** rows)  # experts that some token is routed to, on average
    return {"bytes": touched * (mat(ty, 2 * f, e) + mat(ty, e, f)) + io(e, e, 2 * used), "flops": 2 * rows * used * 3 * e * f}


def tolerance(case):
    # The integers are the same for every correct implementation; the 32-bit sums over a row's blocks are not: 5e-8 to
    # 3.5e-7 from the 64-bit result over the listed and drawn shapes.
    # Where a product's result is rounded to int8 again (the chained layers, the hidden rows of the experts), a last-bit
    # difference can move a value across a rounding step: one such step in a row of a few thousand columns is 5e-4 of
    # it, 6e-5 over 512 tokens.
    if case["kind"] in ("layers", "moe"):
        return {"rel": 2e-3}
    return {"rel": 2e-6}
