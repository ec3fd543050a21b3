"""The work whose speed is measured: quantized linears as a program that runs a model on this
framework calls them, from one decoded token to a prompt of thousands.

A case is one call such a program makes: a decoder layer's linears over M rows (`mxu.dot`), one
linear, the LM head with its greedy or sampled pick, a chained decode step (`chain.DecodeChain`),
a weight matrix packed at load time (`quant.quantize_mxu`).  The shapes are Qwen3-0.6B's and
Qwen3-1.7B's linears, the prefill GEMM and the LM heads of bench.py.

`run` is the path; `exact` is the same in plain torch in 64 bits: the quantizer's literal fp32
steps (amax * f32(1/127), 127 * recip(amax), rint) on the activations, the packed weights'
values in float64 and their float64 product."""
import math

import numpy as np
import torch

DEV = "cuda"
QWEN3_06B = {"hidden": 1024, "q_dim": 2048, "kv_dim": 1024, "F": 3072}
QWEN3_17B = {"hidden": 2048, "q_dim": 2048, "kv_dim": 1024, "F": 6144}


def listed():
    return [
        # one token through a layer's linears: launches and latency
        {"name": "decode1_int4", "kind": "layer", "fmt": "int4", "M": 1, "graph": True, **QWEN3_06B},
        # a few sequences decoded together (or a draft of a few tokens verified)
        {"name": "decode6_int8", "kind": "layer", "fmt": "int8", "M": 6, "graph": True, **QWEN3_06B},
        # a serving batch in 4 bits
        {"name": "decode16_int4", "kind": "layer", "fmt": "int4", "M": 16, "graph": True, **QWEN3_17B},
        # a larger, ragged batch, or a short prompt's rows beside a decode batch
        {"name": "batch50_fp4", "kind": "layer", "fmt": "fp4", "M": 50, "graph": True, **QWEN3_17B},
        # the 512-token prompt of the published prefill figures, int8 and 4-bit
        {"name": "prefill512_int8", "kind": "layer", "fmt": "int8", "M": 512, "graph": False, **QWEN3_06B},
        {"name": "prefill512_int4", "kind": "layer", "fmt": "int4", "M": 512, "graph": False, **QWEN3_06B},
        # a long prompt of no round length
        {"name": "prefill1999_nvfp4", "kind": "layer", "fmt": "nvfp4", "M": 1999, "graph": False, **QWEN3_17B},
        # the prefill GEMM of bench.py (per-row weight scales, one activation scale a row) over a
        # long prompt
        {"name": "gemm4096_rsc_row", "kind": "linear", "fmt": "rsc", "M": 4096, "K": 2048, "N": 8192, "row": True},
        # the LM head with the greedy pick, and a larger one with the sampler after it
        {"name": "head_greedy", "kind": "head", "fmt": "int8", "V": 151936, "K": 1024, "sample": False},
        {"name": "head_sample", "kind": "head", "fmt": "rsc", "V": 262144, "K": 2560, "sample": True},
        # a decode step through a stack of layers as one persistent launch
        {"name": "chain_int4", "kind": "chain", "fmt": "int4", "layers": 8, **QWEN3_17B},
        # a checkpoint's matrix packed while a model loads
        {"name": "pack_int4", "kind": "pack", "fmt": "int4", "N": 6144, "K": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "linear", "linear", "head", "chain", "pack"])
    fmt = rng.choice(["int8", "rsc", "int4", "fp4", "nvfp4"])
    if kind == "layer":
        hidden = 256 * rng.randint(2, 8)
        M = _log(rng, 1, 1500)
        return {"kind": kind, "fmt": fmt, "M": M, "graph": M <= 64, "hidden": hidden,
                "q_dim": 256 * rng.randint(2, 8), "kv_dim": 128 * rng.randint(1, 8), "F": 256 * rng.randint(4, 24)}
    if kind == "linear":
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 1, 3000), "K": 256 * rng.randint(1, 16),
                "N": _log(rng, 100, 6000), "row": rng.random() < 0.3}
    if kind == "head":
        return {"kind": kind, "fmt": rng.choice(["int8", "rsc", "int4"]), "V": _log(rng, 30000, 262000),
                "K": 256 * rng.randint(2, 10), "sample": rng.random() < 0.5}
    if kind == "chain":
        s = rng.choice([QWEN3_06B, QWEN3_17B, {"hidden": 256 * rng.randint(2, 8), "q_dim": 256 * rng.randint(4, 8),
                                               "kv_dim": 256 * rng.randint(1, 4), "F": 256 * rng.randint(8, 24)}])
        return {"kind": kind, "fmt": rng.choice(["int4", "fp4", "nvfp4"]), "layers": rng.randint(2, 8), **s}
    return {"kind": kind, "fmt": fmt, "N": _log(rng, 500, 8000), "K": 256 * rng.randint(2, 16)}


# ------------------------------------------------------------------------- packed weights
# Rows as a loaded checkpoint holds them (the MXU's formats), from N(0, std) weights with a
# plain packer: each group's ideal scale, no search.  `_pack` returns the bytes and the float64
# values they stand for.

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _offset(top, part):
    """The largest d <= 31 with part * 2^d <= top (fp32 magnitudes; 0 for a zero part)."""
    t, p = top.view(torch.int32), part.view(torch.int32)
    d = (t >> 23) - (p >> 23) - ((p & 0x7FFFFF) > (t & 0x7FFFFF)).int()
    return torch.where(part > 0, d.clamp(0, 31), torch.zeros_like(d))


def _codes(g, fmt):
    """Grid values g -> 4-bit codes and their values (int4, or E2M1 sign and magnitude)."""
    if fmt == "int4":
        v = g.round().clamp(-7, 7)
        return v.to(torch.int32) & 15, v.double()
    mid = torch.tensor([(a + b) / 2 for a, b in zip(_E2M1, _E2M1[1:])], device=g.device)
    mag = torch.bucketize(g.abs().contiguous(), mid)
    neg = (g < 0) & (mag > 0)
    v = torch.tensor(_E2M1, dtype=torch.float64, device=g.device)[mag]
    return mag.int() | (neg.int() << 3), torch.where(neg, -v, v)


def _pack(W, fmt, values):
    """(element rows, scale rows, float64 values or None) of W [N, K]."""
    N, K = W.shape
    KB = K // 128
    top = W.abs().amax(1)
    val = None
    if fmt in ("int8", "rsc"):
        S = top * np.float32(1 / 127)
        d = torch.zeros((N, KB), dtype=torch.int32, device=W.device)
        if fmt == "int8":
            d = _offset(top[:, None].expand(N, KB).contiguous(), W.view(N, KB, 128).abs().amax(2))
        sc = torch.ldexp(1 / S[:, None], d)
        q = (W.view(N, KB, 128) * sc[..., None]).round().clamp(-127, 127)
        rows = q.to(torch.int8).view(N, K).view(torch.uint8)
        srows = torch.zeros((N, 4 if fmt == "rsc" else 4 + 4 * -(-KB // 4)), dtype=torch.uint8, device=W.device)
        srows[:, :4] = S.view(torch.uint8).view(N, 4)
        if fmt == "int8":
            srows[:, 4:4 + KB] = d.to(torch.uint8)
        if values:
            val = (q.double() * torch.exp2(-d.double())[..., None]).view(N, K) * S.double()[:, None]
        return rows, srows, val
    if fmt == "nvfp4":
        ts = top / np.float32(448 * 6)
        x = W.view(N, K // 16, 16) / ts[:, None, None]
        e4 = (x.abs().amax(2) / 6).to(torch.float8_e4m3fn)
        s = e4.float()
        g = x / torch.where(s > 0, s, torch.ones_like(s))[..., None]
        Sw = ts * 16
        srows = torch.zeros((N, 16 + 16 * -(-KB // 2)), dtype=torch.uint8, device=W.device)
        srows[:, 16:16 + 8 * KB] = e4.view(torch.uint8)
        code, v = _codes(g, fmt)
        if values:
            val = (v * s.double()[..., None]).view(N, K) * ts.double()[:, None]
    else:
        qmax = 7.0 if fmt == "int4" else 6.0
        sb = W.view(N, KB, 4, 32).abs().amax(3) / qmax
        Sw = sb.amax((1, 2)) / 63
        d = torch.floor(torch.log2(63 * Sw[:, None] / sb.amax(2))).clamp(0, 255).int()
        unit = torch.ldexp(Sw[:, None].expand(N, KB), -d)
        m = (sb / unit[..., None]).round().clamp(1, 63)
        s = unit[..., None] * m
        code, v = _codes(W.view(N, KB, 4, 32) / s[..., None], fmt)
        word = d.long()
        for b in range(4):
            word |= m[:, :, b].long() << (8 + 6 * b)
        srows = torch.zeros((N, 8 + 8 * -(-KB // 2)), dtype=torch.uint8, device=W.device)
        srows[:, 8:8 + 4 * KB] = word.to(torch.int32).view(torch.uint8).view(N, 4 * KB)
        if values:
            val = (v * (m.double() * torch.exp2(-d.double())[..., None])[..., None]).view(N, K) * Sw.double()[:, None]
        if fmt == "fp4":
            Sw = Sw * 0.5                              # (the elements count twice the E2M1 value)
    srows[:, :4] = Sw.contiguous().view(torch.uint8).view(N, 4)
    c = code.reshape(N, K // 2, 2)
    rows = torch.zeros((N, -(-K // 256) * 128), dtype=torch.uint8, device=W.device)
    rows[:, :K // 2] = (c[..., 0] | (c[..., 1] << 4)).to(torch.uint8)
    return rows, srows, val


def _weight(g, N, K, fmt, std=0.02, values=False):
    W = torch.randn((N, K), generator=g, device=DEV)
    return _pack(W * std, fmt, values)


# ---------------------------------------------------------------------------- the inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _hidden(g, M, K):
    """Normed hidden rows: N(0, 1) with channels of unequal size, as a norm's gains leave them."""
    x = torch.randn((M, K), generator=g, device=DEV)
    return x * torch.exp(0.5 * torch.randn((K,), generator=g, device=DEV))


def _gated(g, M, K):
    """A down projection's input: silu(g) * u."""
    a = torch.randn((M, K), generator=g, device=DEV)
    return torch.nn.functional.silu(a) * torch.randn((M, K), generator=g, device=DEV)


def _chunk(F, fmt):
    """The columns each of a down projection's quantizer ranges covers: about an eighth of F, in
    blocks of 128 (int8) or 256 (4-bit), at least 256."""
    q = 128 if fmt in ("int8", "rsc") else 256
    lo = min(F, 256)
    c = max(lo, F // 8 // q * q)
    while F % c and c > lo:
        c -= q
    while F % c:
        c += q
    return c


def _linears(case):
    """(N, K, input, ranges) of each linear of a layer."""
    h, F = case["hidden"], case["F"]
    c = _chunk(F, case["fmt"])
    return [(case["q_dim"] + 2 * case["kv_dim"], h, _hidden, None), (h, case["q_dim"], None, None),
            (2 * F, h, _hidden, None), (h, F, _gated, [c] * (F // c))]


def _layer_inputs(case, g):
    for N, K, make, ranges in _linears(case):
        yield N, K, (make or _plain)(g, case["M"], K), ranges


def _plain(g, M, K):
    return torch.randn((M, K), generator=g, device=DEV)


def _kind(fmt):
    return "int8" if fmt == "rsc" else fmt


def prepare(case, seed):
    from opentpu_amd import chain, mxu, sampler
    g = _gen(seed)
    kind, fmt = case["kind"], case["fmt"]

    def weight(N, K):
        rows, srows, _ = _weight(g, N, K, fmt)
        return mxu.QWeight.from_packed(rows, srows, _kind(fmt), K, fmt == "rsc")

    if kind == "layer":
        calls = []
        for N, K, x, ranges in _layer_inputs(case, g):
            calls.append((x, weight(N, K), ranges))
        state = {"calls": calls}
        if case["graph"]:                              # a decode loop replays its captured step
            _layer(state)
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["out"] = _layer(state)
        return state
    if kind == "linear":
        x = _hidden(g, case["M"], case["K"])
        return {"x": x, "w": weight(case["N"], case["K"]), "row": case["row"]}
    if kind == "head":
        state = {"x": _hidden(g, 1, case["K"]), "w": weight(case["V"], case["K"])}
        if case["sample"]:
            context = torch.randint(0, case["V"], (200,), generator=g, device=DEV).tolist()
            state["sampler"] = sampler.Sampler(case["V"], sampler.Sampling(0.8, 50, 0.9, 1.1), context)
            state["u"] = torch.rand((1,), generator=g, device=DEV)
        return state
    if kind == "chain":
        s = chain.Shape(case["hidden"], case["q_dim"], case["kv_dim"], case["F"], case["layers"])
        x = _plain(g, 1, case["hidden"])
        layers = [{n: _weight(g, N, K, fmt, K ** -0.5)[:2] for n, N, K in s.weight_shapes()}
                  for _ in range(case["layers"])]
        c = chain.DecodeChain.from_packed(layers, s, fmt)
        c.step(x)                                      # (builds its plan)
        return {"chain": c, "x": x}
    return {"W": torch.randn((case["N"], case["K"]), generator=g, device=DEV) * 0.02, "fmt": fmt}


def _layer(state):
    from opentpu_amd import mxu
    return [mxu.dot(x, w, ranges=ranges) for x, w, ranges in state["calls"]]


def run(state):
    from opentpu_amd import fp32, mxu, quant
    if "calls" in state:
        if "graph" not in state:
            return _layer(state)
        state["graph"].replay()
        return state["out"]
    if "row" in state:
        return mxu.dot(state["x"], state["w"], row_mode=state["row"])
    if "chain" in state:
        return state["chain"].step(state["x"], check=False)
    if "W" in state:
        fmt = state["fmt"]
        return quant.quantize_mxu(state["W"], _kind(fmt), rsc=fmt == "rsc")
    w = state["w"]
    q, Sa, da = fp32.quantize_mx(state["x"], 32)
    tok, logits, _ = mxu.lm_head_argmax(q, Sa, da, w.rows, w.srows, w.fmt, w.K, rsc=w.rsc)
    if "sampler" not in state:
        return tok, logits
    return state["sampler"].pick_device(logits, state["u"]), logits


# ------------------------------------------------------------------- what the path has to do

def _row_bytes(K, fmt):
    KB = K // 128
    if fmt == "rsc":
        return K + 4
    if fmt == "int8":
        return K + 4 + KB
    return K // 2 + (16 + 8 * KB if fmt == "nvfp4" else 8 + 4 * KB)


def _linear_work(M, N, K, fmt):
    return N * _row_bytes(K, fmt) + 4 * M * K + 4 * M * N, 2 * M * N * K


def work(case):
    kind, fmt = case["kind"], case["fmt"]
    if kind == "pack":
        N, K = case["N"], case["K"]
        return {"bytes": 4 * N * K + N * _row_bytes(K, fmt), "flops": 0}
    if kind == "linear":
        b, f = _linear_work(case["M"], case["N"], case["K"], fmt)
    elif kind == "head":
        b, f = _linear_work(1, case["V"], case["K"], fmt)
        if case["sample"]:
            b += 2 * 4 * case["V"]                     # the penalty's factors (the logits stay on chip)
    else:
        each = [_linear_work(case.get("M", 1), N, K, fmt) for N, K, _, _ in _linears(case)]
        n = case.get("layers", 1)
        b, f = n * sum(e[0] for e in each), n * sum(e[1] for e in each)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # sums are exact integers and every fp32 step is given: another correct implementation
    # gives the same bits
    return "exact"


# ----------------------------------------------------------------------- the path in 64 bits

def _recip(x):
    """The quantizer's fp32 reciprocal of positive normal x: a linear seed on the significand, two
    Newton steps, a correction step."""
    b = x.view(torch.int32)
    a = ((b & 0x7FFFFF) | 0x3F800000).view(torch.float32)
    y = (0x7EF311C3 - a.view(torch.int32)).view(torch.float32)
    y = y * (2 - a * y)
    y = y * (2 - a * y)
    y = y * (1 - a * y) + y
    return (y.view(torch.int32) + (127 - (b >> 23)) * (1 << 23)).view(torch.float32)


def _quantized(x, row=False):
    """The float64 values of the rows of x (fp32) as int8 rows with a scale a row and an offset a
    group of 32."""
    M, K = x.shape
    top = x.abs().amax(1)
    ok = top > 0
    safe = torch.where(ok, top, torch.ones_like(top))
    S = torch.where(ok, top * torch.tensor(0x3C010204, dtype=torch.int32, device=x.device).view(torch.float32),
                    torch.zeros_like(top))
    inv = torch.where(ok, 127 * _recip(safe), torch.zeros_like(top))
    xg = x.view(M, K // 32, 32)
    d = _offset(top[:, None].expand(M, K // 32).contiguous(), xg.abs().amax(2))
    if row:
        d = torch.zeros_like(d)
    q = (xg * torch.ldexp(inv[:, None].expand_as(d), d)[..., None]).round().clamp(-127, 127)
    return (q.double() * torch.exp2(-d.double())[..., None]).view(M, K) * S.double()[:, None]


def _dot64(x, val, ranges=None, row=False):
    y, c = 0, 0
    for w in ranges or [x.shape[1]]:
        y = y + _quantized(x[:, c:c + w].contiguous(), row) @ val[:, c:c + w].T
        c += w
    return y


def exact(case, seed):
    g = _gen(seed)
    kind, fmt = case["kind"], case["fmt"]
    if kind == "pack":
        return None                                    # (bytes)
    if kind == "layer":
        out = []
        for N, K, x, ranges in _layer_inputs(case, g):
            out.append(_dot64(x, _weight(g, N, K, fmt, values=True)[2], ranges))
        return out
    if kind == "linear":
        x = _hidden(g, case["M"], case["K"])
        return _dot64(x, _weight(g, case["N"], case["K"], fmt, values=True)[2], row=case["row"])
    if kind == "head":
        x = _hidden(g, 1, case["K"])
        return None, _dot64(x, _weight(g, case["V"], case["K"], fmt, values=True)[2])[0]
    h, q_dim, F = case["hidden"], case["q_dim"], case["F"]
    c = _chunk(F, fmt)
    x = _plain(g, 1, h)
    for _ in range(case["layers"]):
        qkv, o, gu, down = [_weight(g, N, K, fmt, K ** -0.5, True)[2] for N, K, _, _ in _linears(case)]
        y = _dot64(_dot64(x, qkv).float()[:, :q_dim].contiguous(), o).float()
        gate = _dot64(y, gu).float()
        y = _dot64(gate[:, :F] * gate[:, F:], down, [c] * (F // c))
        x = y.float()
    return y
