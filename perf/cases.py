"""Timed cases of the quantized linear-layer path: what a program that runs a GGUF model on this
library has it do, through the entry points of ``apeiron_amd.chart``.

Sizes are the projection shapes of the two model classes the benchmark uses (hidden 896 / FFN 4864
and hidden 1536 / FFN 8960, vocabulary 151936), from one token (decode) over short batches to long
prompts, every weight family, odd widths and token counts, f32 and pre-quantized inputs.

Weights are random block payloads whose projections of a unit-variance input have about unit
variance (block scales spread by a factor of about 1.6, the K-quants' mins placed so that weights
average zero, as trained ones do); activations are normal with a spread of channel scales.
"""
from __future__ import annotations

import math

import torch

from apeiron_amd import chart

Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q6_K = 6, 8, 10, 11, 12, 14
TYPES = {"Q5_0": Q5_0, "Q8_0": Q8_0, "Q2_K": Q2_K, "Q3_K": Q3_K, "Q4_K": Q4_K, "Q6_K": Q6_K}
BLOCK = {Q5_0: (32, 22), Q8_0: (32, 34), Q2_K: (256, 84), Q3_K: (256, 110), Q4_K: (256, 144), Q6_K: (256, 210)}


def listed():
    return [
        # one projection of a small model's decode step: the shortest call, latency alone
        {"name": "gemv_q8_0", "op": "gemv", "type": "Q8_0", "n_out": 4864, "n_in": 896, "codes": False},
        # every projection of a decode token's layers, launched from the host / as a captured graph
        {"name": "decode_layer_eager", "op": "decode", "hidden": 896, "kv": 128, "ff": 4864, "layers": 1, "graph": False},
        {"name": "decode_layers_graph", "op": "decode", "hidden": 1536, "kv": 256, "ff": 8960, "layers": 8, "graph": True},
        # the vocabulary head: the largest product of a token, streamed from memory
        {"name": "gemv_q6_k_head", "op": "gemv", "type": "Q6_K", "n_out": 151936, "n_in": 1536, "codes": False},
        # the quantizer on its own, as the engine quantizes a prompt's columns once for several uses
        {"name": "quant_2048", "op": "quant", "n_tok": 2048, "n_in": 8960},
        # a few tokens at once (sequences decoded together, a drafted run verified, a one-line prompt): one projection
        # from the engine's own quantized activations at widths off every grid, and a layer's whole FFN
        {"name": "gemm_q5_0_n5_odd", "op": "gemm", "type": "Q5_0", "n_out": 4861, "n_in": 901, "n_tok": 5, "codes": True},
        {"name": "ffn_n8", "op": "ffn", "type": "Q4_K", "down": "Q6_K", "hidden": 1536, "ff": 8960, "n_tok": 8},
        # q/k/v of a short prompt: one input, three projections of two types, a ragged token count
        {"name": "qkv_n137", "op": "qkv", "hidden": 1536, "kv": 256, "n_tok": 137},
        # prefill chunks of 512 and 300 tokens, wide and deep, from f32 and from codes
        {"name": "gemm_q8_0_n512", "op": "gemm", "type": "Q8_0", "n_out": 896, "n_in": 4864, "n_tok": 512, "codes": True},
        {"name": "gemm_q3_k_n300", "op": "gemm", "type": "Q3_K", "n_out": 4864, "n_in": 896, "n_tok": 300, "codes": False},
        # a layer's FFN on a 512-token chunk (gate/up, SwiGLU, hidden quantizer, a Q6_K down)
        {"name": "ffn_n512", "op": "ffn", "type": "Q4_K", "down": "Q6_K", "hidden": 1536, "ff": 8960, "n_tok": 512},
        # the same layer on a long prompt, all Q4_K: the largest pass
        {"name": "ffn_n2048", "op": "ffn", "type": "Q4_K", "down": "Q4_K", "hidden": 1536, "ff": 8960, "n_tok": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A projection width: mostly multiples of 128 as models have them, otherwise any number."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.35 else max(128, n // 128 * 128)


def draw(rng):
    op = rng.choice(["gemv", "gemv", "gemm", "gemm", "gemm", "qkv", "ffn", "ffn", "decode", "quant"])
    kind = rng.choice(sorted(TYPES))
    if op == "gemv":
        wide = rng.random() < 0.25
        return {"op": op, "type": kind, "n_out": _log_int(rng, 30000, 151936) if wide else _width(rng, 128, 18000),
                "n_in": rng.choice([896, 1536]) if wide else _width(rng, 512, 8960), "codes": rng.random() < 0.4}
    if op == "gemm":
        n_out, n_in = _width(rng, 128, 9000), _width(rng, 256, 8960)
        return {"op": op, "type": kind, "n_out": n_out, "n_in": n_in,
                "n_tok": min(_log_int(rng, 2, 2048), 80_000_000_000 // (n_out * n_in)), "codes": rng.random() < 0.4}
    if op == "qkv":
        return {"op": op, "hidden": rng.choice([896, 1536, _width(rng, 256, 2048)]), "kv": rng.choice([128, 256, 512]),
                "n_tok": _log_int(rng, 2, 1024)}
    if op == "ffn":
        k = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q3_K", "Q2_K", "Q6_K", "Q5_0"])
        return {"op": op, "type": k, "down": rng.choice([k, "Q6_K"]), "hidden": rng.choice([896, 1536, _width(rng, 256, 1536)]),
                "ff": _width(rng, 512, 8960), "n_tok": _log_int(rng, 2, 1500)}
    if op == "decode":
        return {"op": op, "hidden": rng.choice([896, 1536, _width(rng, 256, 1536)]), "kv": rng.choice([128, 256]),
                "ff": _width(rng, 512, 8960), "layers": rng.choice([1, 2, 4, 8]), "graph": rng.random() < 0.6}
    return {"op": op, "n_tok": _log_int(rng, 1, 2048), "n_in": _width(rng, 128, 8960)}


# ---- inputs --------------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _f16_words(v):
    b = v.to(torch.float16).view(torch.int16).to(torch.int32) & 0xFFFF
    return (b & 0xFF).to(torch.uint8), (b >> 8).to(torch.uint8)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _payload(kind, n_out, n_in, g):
    """GGUF block bytes [n_out][blocks][block bytes] on the GPU."""
    qk, bb = BLOCK[kind]
    nb = -(-n_in // qk)
    raw = _bytes(g, n_out, nb, bb)
    spread = torch.exp(0.25 * torch.randn(n_out, nb, generator=g, device="cuda"))
    unit = 1.0 / math.sqrt(n_in)

    def put(at, v):
        raw[..., at], raw[..., at + 1] = _f16_words(v)

    if kind == Q8_0:
        raw[..., 2:] = torch.where(raw[..., 2:] == 128, torch.zeros_like(raw[..., 2:]), raw[..., 2:])  # codes -127..127
        put(0, spread * unit / 73.0)
    elif kind == Q5_0:
        put(0, spread * unit / 9.2)
    elif kind == Q6_K:
        raw[..., 192:208] = torch.randint(20, 128, (n_out, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
        put(208, spread * unit / (18.5 * 80.0))
    elif kind == Q3_K:
        put(108, spread * unit / (2.3 * 18.5))
    elif kind == Q2_K:
        sc = torch.randint(2, 11, (n_out, nb, 16), generator=g, device="cuda")
        raw[..., :16] = (sc | (((3 * sc + 1) // 2) << 4)).to(torch.uint8)  # m = 1.5 sc
        put(80, spread * unit / (1.1 * 6.5))
        raw[..., 82:84] = raw[..., 80:82]
    else:  # Q4_K: sc in 1..8, m = 7.5 sc, dmin = d; 6-bit pairs packed as the format has them
        sc = torch.randint(1, 9, (n_out, nb, 8), generator=g, device="cuda")
        m = (15 * sc + 1) // 2
        raw[..., 4:8] = (sc[..., :4] | ((sc[..., 4:] >> 4) << 6)).to(torch.uint8)
        raw[..., 8:12] = (m[..., :4] | ((m[..., 4:] >> 4) << 6)).to(torch.uint8)
        raw[..., 12:16] = ((sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)).to(torch.uint8)
        put(0, spread * unit / (4.6 * 5.0))
        raw[..., 2:4] = raw[..., 0:2]
    return raw


def _acts(n_tok, n_in, g):
    channel = torch.exp(0.5 * torch.randn(n_in, generator=g, device="cuda"))
    return torch.randn(n_tok, n_in, generator=g, device="cuda") * channel


def _weights(case):
    """(name, type, n_out, n_in) of a case's projections, layer by layer for a decode token."""
    op = case["op"]
    if op in ("gemv", "gemm"):
        return [("w", TYPES[case["type"]], case["n_out"], case["n_in"])]
    if op == "qkv":
        h, kv = case["hidden"], case["kv"]
        return [("q", Q4_K, h, h), ("k", Q4_K, kv, h), ("v", Q6_K, kv, h)]
    if op == "ffn":
        h, ff = case["hidden"], case["ff"]
        return [("gate", TYPES[case["type"]], ff, h), ("up", TYPES[case["type"]], ff, h), ("down", TYPES[case["down"]], h, ff)]
    if op == "decode":
        h, kv, ff = case["hidden"], case["kv"], case["ff"]
        return [w for l in range(case["layers"])
                for w in (("q", Q4_K, h, h), ("k", Q4_K, kv, h), ("v", Q6_K, kv, h), ("o", Q4_K, h, h), ("gate", Q4_K, ff, h),
                          ("up", Q4_K, ff, h), ("down", Q4_K if l % 2 else Q6_K, h, ff))]
    return []


def _inputs(case):
    """[n_tok][n_in] of each input vector of a case."""
    op = case["op"]
    if op == "decode":
        return [(1, case["hidden"])] * (3 * case["layers"])
    if op == "gemv":
        return [(1, case["n_in"])]
    return [(case["n_tok"], case["hidden"] if op in ("qkv", "ffn") else case["n_in"])]


def _data(case, seed):
    g = _gen(seed)
    raws = [(kind, n_out, n_in, _payload(kind, n_out, n_in, g)) for _, kind, n_out, n_in in _weights(case)]
    return raws, [_acts(t, k, g) for t, k in _inputs(case)]


def _empty(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    dev = chart.device()
    raws, xs = _data(case, seed)
    W = [dev.upload(kind, raw.reshape(-1).cpu().numpy(), n_out, n_in) for kind, n_out, n_in, raw in raws]
    op = case["op"]
    s = {"case": case, "dev": dev, "W": W, "x": xs}
    if op == "quant":
        s["out"] = [_empty(case["n_tok"], case["n_in"], dtype=torch.int8),
                    _empty(case["n_tok"], -(-case["n_in"] // 32), dtype=torch.int64)]
    elif op in ("gemv", "gemm"):
        n_tok = case.get("n_tok", 1)
        s["out"] = [_empty(n_tok, case["n_out"])]
        if case["codes"]:
            codes, scales = _empty(n_tok, case["n_in"], dtype=torch.int8), _empty(n_tok, -(-case["n_in"] // 32), dtype=torch.int64)
            dev.quant_act_f32_dev(xs[0].data_ptr(), n_tok, case["n_in"], codes.data_ptr(), scales.data_ptr(), _stream())
            s["q"] = (codes, scales)
    elif op == "qkv":
        s["out"] = [_empty(case["n_tok"], w.n_out) for w in W]
    elif op == "ffn":
        n, ff = case["n_tok"], case["ff"]
        s["out"] = [_empty(n, case["hidden"]), _empty(n, ff, dtype=torch.int8), _empty(n, -(-ff // 32), dtype=torch.int64)]
    else:
        L, h, kv, ff = case["layers"], case["hidden"], case["kv"], case["ff"]
        s["out"] = [_empty(L, h), _empty(L, kv), _empty(L, kv), _empty(L, h), _empty(L, h),
                    _empty(L, -(-ff // 16) * 16, dtype=torch.int8), _empty(L, -(-ff // 32), dtype=torch.int64)]
        s["plans"] = [chart.GemvPlan(dev, W[7 * l:7 * l + 3], [xs[3 * l].data_ptr()] * 3, [s["out"][k][l].data_ptr() for k in range(3)])
                      for l in range(L)]
        if case["graph"]:
            _decode(s, _stream())
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"], stream=torch.cuda.Stream()):
                _decode(s, _stream())
    return s


# ---- the passes ----------------------------------------------------------------------------------


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _decode(s, stream):
    W, x, out = s["W"], s["x"], s["out"]
    for l, plan in enumerate(s["plans"]):
        o, gate, up, down = W[7 * l + 3:7 * l + 7]
        plan.run(stream)
        o.gemv_f32_dev(x[3 * l + 1].data_ptr(), out[3][l].data_ptr(), stream)
        chart.ffn_dev(s["dev"], gate, up, down, x[3 * l + 2].data_ptr(), out[4][l].data_ptr(), out[5][l].data_ptr(),
                      out[6][l].data_ptr(), stream)


def run(s):
    case, dev, W, x, out = s["case"], s["dev"], s["W"], s["x"], s["out"]
    op, stream = case["op"], _stream()
    if op == "decode":
        if case["graph"]:
            s["graph"].replay()
        else:
            _decode(s, stream)
    elif op == "quant":
        dev.quant_act_f32_dev(x[0].data_ptr(), case["n_tok"], case["n_in"], out[0].data_ptr(), out[1].data_ptr(), stream)
    elif op == "gemv":
        if case["codes"]:
            W[0].gemv_q8_dev(s["q"][0].data_ptr(), s["q"][1].data_ptr(), out[0].data_ptr(), stream)
        else:
            W[0].gemv_f32_dev(x[0].data_ptr(), out[0].data_ptr(), stream)
    elif op == "gemm":
        if case["codes"]:
            W[0].gemm_q8_dev(s["q"][0].data_ptr(), s["q"][1].data_ptr(), case["n_tok"], out[0].data_ptr(), stream)
        else:
            W[0].gemm_f32_dev(x[0].data_ptr(), case["n_tok"], out[0].data_ptr(), stream)
    elif op == "qkv":
        chart.gemm_group_f32_dev(dev, W, x[0].data_ptr(), case["n_tok"], [y.data_ptr() for y in out], stream)
    else:
        chart.ffn_prefill_dev(dev, W[0], W[1], W[2], x[0].data_ptr(), case["n_tok"], out[0].data_ptr(), out[1].data_ptr(),
                              out[2].data_ptr(), stream)
    return out


def _read_bytes(kind, n_in):
    """Bytes of one weight row that a product has to read (a ragged last super-block in part)."""
    qk, bb = BLOCK[kind]
    full, rem = divmod(n_in, qk)
    if rem == 0 or qk == 32:
        return bb * (-(-n_in // qk))
    half = -(-rem // 128)
    tail = {Q4_K: 16 + 32 * (-(-rem // 64)), Q2_K: 20 + 32 * half, Q3_K: 46 + 32 * half, Q6_K: 2 + 104 * half}[kind]
    return bb * full + tail


def work(case):
    op = case["op"]
    n_tok = case.get("n_tok", 1)
    if op == "quant":
        n = n_tok * case["n_in"]
        return {"bytes": 5 * n + 8 * n_tok * -(-case["n_in"] // 32), "flops": 4 * n}
    size = flops = 0
    for name, kind, n_out, n_in in _weights(case):
        size += n_out * _read_bytes(kind, n_in)
        flops += 2 * n_tok * n_out * n_in
        if name not in ("gate", "up"):
            size += 4 * n_tok * n_out  # the outputs
        elif name == "gate":
            size += n_tok * (n_out + 8 * -(-n_out // 32))  # the hidden codes and scales
    for t, k in _inputs(case):
        size += t * (k + 8 * -(-k // 32) if case.get("codes") else 4 * k)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Relative errors between correct implementations, about four times what was measured."""
    if case["op"] == "quant":
        return "exact"
    if case["op"] in ("ffn", "decode"):
        # a last-bit difference of a gate or up value moves a few hidden codes by one, and so the down projection
        return {"rel": 1e-3, "max": 2e-2, "differ": 2e-3}
    return {"rel": 1e-6, "max": 1e-5}


# ---- 64-bit reference ----------------------------------------------------------------------------


def _dequant(kind, raw, n_in):
    """f64 weights [n_out][n_in] of a payload [n_out][blocks][bytes]."""
    n_out, nb, _ = raw.shape
    b = raw.to(torch.int32)

    def half(at):
        return (b[..., at] | (b[..., at + 1] << 8)).to(torch.int16).view(torch.float16).double()

    if kind == Q8_0:
        w = half(0)[..., None] * raw[..., 2:].view(torch.int8).double()
    elif kind == Q5_0:
        qh = b[..., 2].long() | (b[..., 3].long() << 8) | (b[..., 4].long() << 16) | (b[..., 5].long() << 24)
        bits = (qh[..., None] >> torch.arange(32, device=raw.device)) & 1
        q = torch.cat([b[..., 6:22] & 15, b[..., 6:22] >> 4], -1) | (bits << 4)
        w = half(0)[..., None] * (q - 16).double()
    elif kind == Q4_K:
        s = b[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:12] & 15) | ((s[..., :4] >> 6) << 4)], -1)
        m = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
        q = b[..., 16:].reshape(n_out, nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).reshape(n_out, nb, 8, 32)
        w = half(0)[..., None, None] * sc[..., None].double() * q.double() - (half(2)[..., None] * m.double())[..., None]
    elif kind == Q6_K:
        ql, qh = b[..., :128].reshape(n_out, nb, 2, 2, 32), b[..., 128:192].reshape(n_out, nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 3)  # [half][4][32]
        hi = torch.cat([(qh >> (2 * t)) & 3 for t in range(4)], 3)
        q = ((lo | (hi << 4)) - 32).reshape(n_out, nb, 16, 16)
        w = half(208)[..., None, None] * raw[..., 192:208].view(torch.int8).double()[..., None] * q.double()
    else:
        qs = b[..., (32 if kind == Q3_K else 16):][..., :64].reshape(n_out, nb, 2, 1, 32)
        q = torch.cat([(qs >> (2 * r)) & 3 for r in range(4)], 3)  # [half][pair][32]
        if kind == Q2_K:
            q = q.reshape(n_out, nb, 16, 16)
            sc, m = b[..., :16] & 15, b[..., :16] >> 4
            w = half(80)[..., None, None] * (sc[..., None] * q).double() - (half(82)[..., None] * m.double())[..., None]
        else:
            hm = b[..., :32].reshape(n_out, nb, 1, 1, 32)
            hb = torch.cat([torch.cat([(hm >> (4 * n + r)) & 1 for r in range(4)], 3) for n in range(2)], 2)
            q = ((q | (hb << 2)) - 4).reshape(n_out, nb, 16, 16)
            s = b[..., 96:108]
            low = torch.cat([s[..., :8] & 15, s[..., :8] >> 4], -1)
            high = torch.cat([(s[..., 8:12] >> (2 * i)) & 3 for i in range(4)], -1)
            w = half(108)[..., None, None] * ((low | (high << 4)) - 32).double()[..., None] * q.double()
    return w.reshape(n_out, -1)[:, :n_in]


def _quant(x):
    """The power-of-two int8 quantizer on real f64 rows: codes and scales, as integers."""
    t, k = x.shape
    nb = -(-k // 32)
    v = x * 4294967296.0
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    q = torch.nn.functional.pad(q, (0, 32 * nb - k)).to(torch.int64).reshape(t, nb, 32)
    top = q.abs().amax(-1)
    _, length = torch.frexp(top.double())  # bit length (0 for 0)
    e = torch.clamp(length.to(torch.int64) - 7, min=0)
    e = e + (top > (127 << e)).to(torch.int64)
    m = q.abs()
    c = (m >> e[..., None]) + torch.where(e[..., None] > 0, (m >> torch.clamp(e[..., None] - 1, min=0)) & 1, torch.zeros_like(m))
    scales = torch.where(top > 0, torch.ones_like(e) << e, torch.zeros_like(e))
    return (torch.sign(q) * c).reshape(t, -1)[:, :k], scales


def _real(codes, scales):
    k = codes.shape[1]
    return codes.double() * (scales.double() / 4294967296.0).repeat_interleave(32, 1)[:, :k]


def exact(case, seed):
    if case["op"] == "quant":
        return None
    raws, xs = _data(case, seed)
    xq = [_real(*_quant(x.double())) for x in xs]

    def prod(i, x):
        kind, n_out, n_in, raw = raws[i]
        step = max(1, (1 << 28) // n_in)
        return torch.cat([x @ _dequant(kind, raw[r:r + step], n_in).T for r in range(0, n_out, step)], 1)

    def ffn(i, x):
        gate, up = prod(i, x), prod(i + 1, x)
        codes, scales = _quant(gate / (1.0 + torch.exp(-gate)) * up)
        return prod(i + 2, _real(codes, scales)), codes, scales

    if case["op"] in ("gemv", "gemm"):
        return [prod(0, xq[0])]
    if case["op"] == "qkv":
        return [prod(i, xq[0]) for i in range(3)]
    if case["op"] == "ffn":
        return [ffn(0, xq[0])[0], None, None]
    rows = []
    for l in range(case["layers"]):
        a, o, f = xq[3 * l:3 * l + 3]
        rows.append([prod(7 * l, a), prod(7 * l + 1, a), prod(7 * l + 2, a), prod(7 * l + 3, o), ffn(7 * l + 4, f)[0]])
    return [torch.cat([r[k] for r in rows]) for k in range(5)] + [None, None]
