"""Performance cases of the quantized-weight matrix path.

The work a language model's host program gives this library: the steps of one
decoded token (matrix-vector products, the feed-forward pair behind its norm,
the lm_head with greedy selection, routed expert layers), recorded once into a
graph and replayed per token, and the products and expert layers of a prompt,
called as they come.  A decode case holds the matrices of several layers, as a
model does, so a pass streams its weights instead of finding the last pass's
bytes in a cache; each layer takes its own input rows, because what one layer
hands to the next (attention) is not part of this library.

listed() names the cases, draw() gives further ones of the same ranges.
"""
import functools
import math

import torch

import oco_amd as oco

# GGUF codes of the formats that checkpoints of these models store matrices in
F16, Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, MXFP4 = 1, 2, 8, 12, 13, 14, 39
BLOCKS = {F16: (1, 2), Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210),
          MXFP4: (32, 17)}

# The two expert banks of this repository's benchmark:
# format, hidden, ffn, experts, routes per token
BANKS = {"gpt_oss_20b": (MXFP4, 2880, 2880, 32, 4), "qwen3_30b_a3b": (Q4_K, 2048, 768, 128, 8)}
VOCABULARY = 4096  # rows of the embedding table that residual rows come from
EPSILON = 1e-6


def listed():
    return [
        # Attention projections of gpt-oss-20b around one decoded token: k and v (two 512 x 2880 in one
        # grid), q (4096 x 2880) behind their norm, o (2880 x 4096).  The smallest calls of a token.
        {"name": "decode_attention_q8_0", "kind": "attention", "layers": 12},
        # One MXFP4 matrix per layer with an f32 row: the decode product of the headline benchmark.
        {"name": "decode_mxfp4", "kind": "matvec", "format": MXFP4, "n": 5760, "k": 2880, "layers": 24, "x": "f32"},
        # Feed-forward of a dense 8B model at decode: norm, gate and up in one grid (Q4_K), down (Q6_K).
        {"name": "decode_ffn_q4_k_m", "kind": "ffn", "layers": 4},
        # End of every token: lm_head logits in f32, then the greedy choice.
        {"name": "decode_head_q6_k", "kind": "head", "n": 151936, "k": 4096},
        # Eight sequences decoded together (or eight draft tokens verified): few rows on a large matrix.
        {"name": "rows8_q4_k", "kind": "matmul", "format": Q4_K, "n": 12288, "k": 4096, "m": 8, "layers": 4,
         "y": "bf16"},
        # Routed expert layer of a mixture model, one token and sixteen, and a bank of many small experts.
        {"name": "decode_experts_mxfp4_b1", "kind": "experts", "bank": "gpt_oss_20b", "tokens": 1, "layers": 4},
        {"name": "decode_experts_mxfp4_b16", "kind": "experts", "bank": "gpt_oss_20b", "tokens": 16, "layers": 2},
        {"name": "decode_experts_q4_k_b4", "kind": "experts", "bank": "qwen3_30b_a3b", "tokens": 4, "layers": 4},
        # Prompt chunks: the expert layer, the norm with the product behind it, dense products of an
        # ordinary chunk and of a long ragged one.
        {"name": "prefill_experts_q4_k", "kind": "experts", "bank": "qwen3_30b_a3b", "tokens": 512, "layers": 1},
        {"name": "prefill_norm_mxfp4", "kind": "norm_matmul", "n": 5760, "k": 2880, "m": 512},
        {"name": "prefill_q4_k", "kind": "matmul", "format": Q4_K, "n": 12288, "k": 4096, "m": 512, "layers": 1,
         "y": "bf16"},
        {"name": "prefill_q6_k_ragged", "kind": "matmul", "format": Q6_K, "n": 4096, "k": 12288, "m": 1999, "layers": 1,
         "y": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, fmt, lo, hi):
    unit = max(BLOCKS[fmt][0], 32)
    return max(1, _log(rng, lo, hi) // unit) * unit


def draw(rng):
    """Any of the listed kinds, at any size between a draft model's and the largest listed ones."""
    kind = rng.choice(["matvec", "matvec", "matmul", "matmul", "matmul", "experts", "experts", "norm_matmul", "head"])
    if kind == "matvec":
        fmt = rng.choice([Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, MXFP4])
        return {"kind": kind, "format": fmt, "n": _log(rng, 256, 16384), "k": _width(rng, fmt, 1024, 12288),
                "layers": rng.randint(4, 12), "x": rng.choice(["f32", "bf16"])}
    if kind == "head":
        return {"kind": kind, "n": _log(rng, 30000, 151936), "k": _width(rng, Q6_K, 1024, 4096)}
    if kind == "experts":
        return {"kind": kind, "bank": rng.choice(sorted(BANKS)), "tokens": _log(rng, 1, 512), "layers": 1}
    if kind == "norm_matmul":
        return {"kind": kind, "n": _log(rng, 512, 8192), "k": _width(rng, MXFP4, 1024, 4096), "m": _log(rng, 32, 1024)}
    fmt = rng.choice([F16, Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, MXFP4])
    m, n, k = _log(rng, 2, 2048), _log(rng, 512, 12288), _width(rng, fmt, 1024, 12288)
    n = n if rng.random() < 0.25 else -(-n // 4) * 4  # model widths are whole quads but for an odd head
    while m * n * k > 1999 * 4096 * 12288:
        m = (m + 1) // 2
    return {"kind": kind, "format": fmt, "n": n, "k": k, "m": m, "layers": 1, "y": rng.choice(["f32", "bf16"])}


# ---- weights: normal values with the scales of trained matrices, as the GGUF packers round them -------

def _codes(gen, shape, mean, sd, lo, hi):
    v = torch.randn(shape, generator=gen, device="cuda")
    return v.mul_(sd).add_(mean).round_().clamp_(lo, hi).to(torch.uint8)


def _half(gen, blocks, size):
    """f16 block scales around `size`, as bytes [blocks, 2]."""
    d = (torch.rand((blocks, 1), generator=gen, device="cuda") + 0.5) * size
    return d.to(torch.float16)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _k_scales(gen, nb):
    """The 12 bytes of eight 6-bit (scale, minimum) pairs, and d : dmin such that weights centre on zero."""
    sc = torch.randint(24, 64, (nb, 8), generator=gen, device="cuda", dtype=torch.uint8)
    mn = (sc.to(torch.int16) + torch.randint(-4, 5, (nb, 8), generator=gen, device="cuda", dtype=torch.int16))
    mn = mn.clamp_(0, 63).to(torch.uint8)
    low = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6)], 1)
    return torch.cat([low, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)


def weights(fmt, rows, k, seed):
    """rows x k values of standard deviation about 0.02 in GGUF blocks: uint8 [rows * bytes of a row]."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    unit, size = BLOCKS[fmt]
    if fmt == F16:
        return _bytes((torch.randn((rows, k), generator=gen, device="cuda") * 0.02).to(torch.float16)).view(-1)
    out = torch.empty((rows * (k // unit), size), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 28) // unit)  # blocks at a time: the codes pass through f32
    for at in range(0, out.shape[0], step):
        b = out[at:at + step]
        nb = b.shape[0]
        if fmt == Q8_0:
            b[:, :2] = _bytes(_half(gen, nb, 0.0005))
            b[:, 2:] = (_codes(gen, (nb, 32), 128.0, 40.0, 1, 255).to(torch.int16) - 128).to(torch.int8).view(torch.uint8)
        elif fmt == Q4_0:
            b[:, :2] = _bytes(_half(gen, nb, 0.0075))
            q = _codes(gen, (nb, 2, 16), 8.0, 2.7, 0, 15)
            b[:, 2:] = q[:, 0] | (q[:, 1] << 4)
        elif fmt == MXFP4:
            b[:, 0] = torch.randint(119, 123, (nb,), generator=gen, device="cuda", dtype=torch.uint8)
            v = torch.randn((nb, 32), generator=gen, device="cuda")
            edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
            q = torch.bucketize(v.abs() * 2.0, edges, out_int32=True).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
            b[:, 1:] = q[:, :16] | (q[:, 16:] << 4)
        elif fmt == Q6_K:
            q = _codes(gen, (nb, 2, 2, 2, 32), 32.0, 10.7, 0, 63)  # [half, quarter / 2, quarter % 2, column]
            b[:, :128] = ((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(nb, 128)
            hi = (q >> 4).reshape(nb, 2, 4, 32)
            b[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(nb, 64)
            sc = torch.randint(64, 128, (nb, 16), generator=gen, device="cuda", dtype=torch.int16)
            sign = torch.randint(0, 2, (nb, 16), generator=gen, device="cuda", dtype=torch.int16) * 2 - 1
            b[:, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
            b[:, 208:] = _bytes(_half(gen, nb, 2e-5))
        else:  # Q4_K, Q5_K
            mid, sd = (7.5, 2.7) if fmt == Q4_K else (15.5, 5.4)
            d = _half(gen, nb, 0.02 / sd / 48)
            b[:, :2] = _bytes(d)
            b[:, 2:4] = _bytes((d.float() * mid).to(torch.float16))
            b[:, 4:16] = _k_scales(gen, nb)
            q = _codes(gen, (nb, 4, 2, 32), mid, sd, 0, 15 if fmt == Q4_K else 31)  # [pair, sub-block % 2, column]
            if fmt == Q5_K:
                bits = torch.arange(8, device="cuda", dtype=torch.uint8).view(1, 8, 1)
                b[:, 16:48] = ((q.reshape(nb, 8, 32) >> 4) << bits).sum(1, dtype=torch.uint8)
            b[:, size - 128:] = ((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(nb, 128)
    return out.view(-1)


def _scale(b, at):
    return _bytes(b[:, at:at + 2]).view(torch.float16).double()


def decoded(fmt, data, rows, k):
    """The weights as f64 [rows, k] (the decode rules of the GGUF formats)."""
    unit, size = BLOCKS[fmt]
    if fmt == F16:
        return data.view(torch.float16).view(rows, k).double()
    b = data.view(-1, size)
    nb = b.shape[0]
    if fmt == Q8_0:
        w = b[:, 2:].view(torch.int8).double() * _scale(b, 0)
    elif fmt == Q4_0:
        w = (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0) * _scale(b, 0)
    elif fmt == MXFP4:
        table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=b.device)
        table = torch.cat([table, -table])
        w = table[torch.cat([b[:, 1:] & 15, b[:, 1:] >> 4], 1).long()]
        w = torch.ldexp(w, (b[:, :1].to(torch.int32) - 127))
    elif fmt == Q6_K:
        ql, qh = b[:, :128].view(nb, 2, 2, 32), b[:, 128:192].view(nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)).double().sub_(32.0).view(nb, 16, 16)
        w = q * b[:, 192:208].view(torch.int8).double().unsqueeze(2) * _scale(b, 208).unsqueeze(2)
    else:  # Q4_K, Q5_K
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, size - 128:].view(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if fmt == Q5_K:
            bits = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (((b[:, 16:48].unsqueeze(1) >> bits) & 1) << 4)
        w = q.double() * (sc * _scale(b, 0)).unsqueeze(2) - (mn * _scale(b, 2)).unsqueeze(2)
    return w.reshape(rows, k)


def _rows(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


# ---- preparation --------------------------------------------------------------------------------------

@functools.lru_cache(None)
def _stream():
    return oco.Stream()


def _recorded(state, launch):
    """The launches of one token, recorded once and replayed (state keeps the graph)."""
    torch.cuda.synchronize()
    state["graph"] = oco.Graph(_stream(), launch)
    return state


def _norm_weight(gen, k):
    return 1.0 + 0.1 * torch.randn(k, generator=gen, device="cuda")


def _matrix(k, n, m=1, bias=0):
    return oco.Matrix(k, n, m, 0, 1, 1, bias)


def _inputs(case, seed):
    """Weights and activations of a case, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 8191 + 17)
    kind, s = case["kind"], {}
    if kind == "attention":
        s["layers"] = []
        for i in range(case["layers"]):
            at = seed * 1009 + 8 * i
            s["layers"].append({"q": weights(Q8_0, 4096, 2880, at), "k": weights(Q8_0, 512, 2880, at + 1),
                                "v": weights(Q8_0, 512, 2880, at + 2), "o": weights(Q8_0, 2880, 4096, at + 3),
                                "norm": _norm_weight(gen, 2880), "bias": 0.1 * _rows(gen, 8000, dtype=torch.float32)})
        s["x"], s["mixed"] = _rows(gen, case["layers"], 2880), _rows(gen, case["layers"], 4096)
    elif kind == "ffn":
        s["layers"] = []
        for i in range(case["layers"]):
            at = seed * 1009 + 8 * i
            s["layers"].append({"gate": weights(Q4_K, 12288, 4096, at), "up": weights(Q4_K, 12288, 4096, at + 1),
                                "down": weights(Q6_K, 4096, 12288, at + 2), "norm": _norm_weight(gen, 4096)})
        s["x"], s["act"] = _rows(gen, case["layers"], 4096), _rows(gen, case["layers"], 12288, dtype=torch.float32)
    elif kind == "experts":
        fmt, hidden, ffn, experts, _ = BANKS[case["bank"]]
        biased, t = case["bank"] == "gpt_oss_20b", case["tokens"]
        s["layers"] = []
        for i in range(case["layers"]):
            at = seed * 1009 + 8 * i
            s["layers"].append({
                "gate": weights(fmt, experts * ffn, hidden, at), "up": weights(fmt, experts * ffn, hidden, at + 1),
                "down": weights(fmt, experts * hidden, ffn, at + 2), "norm": _norm_weight(gen, hidden),
                "router": _rows(gen, experts, hidden, dtype=torch.float32) / math.sqrt(hidden),
                "router_bias": 0.1 * _rows(gen, experts, dtype=torch.float32) if biased else None,
                "biases": [0.1 * _rows(gen, experts * r, dtype=torch.float32) for r in (ffn, ffn, hidden)]
                if biased else [None] * 3})
        s["table"] = _rows(gen, VOCABULARY, hidden)
        s["tokens"] = torch.randint(0, VOCABULARY, (case["layers"] * t,), generator=gen, device="cuda", dtype=torch.int32)
    else:
        layers, fmt = case.get("layers", 1), Q6_K if kind == "head" else MXFP4 if kind == "norm_matmul" else case["format"]
        s["w"] = [weights(fmt, case["n"], case["k"], seed * 1009 + i) for i in range(layers)]
        s["x"] = _rows(gen, layers, case.get("m", 1), case["k"],
                       dtype=torch.float32 if case.get("x") == "f32" or kind == "head" else torch.bfloat16)
        if kind == "norm_matmul":
            s["norm"] = _norm_weight(gen, case["k"])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], kind = case, case["kind"]
    D, empty = oco.DType, functools.partial(torch.empty, device="cuda")
    if kind == "attention":
        L = case["layers"]
        s["out"] = {"k": empty((L, 512)), "v": empty((L, 512)), "q": empty((L, 4096)), "o": empty((L, 2880))}

        def launch():
            out = s["out"]
            for i, w in enumerate(s["layers"]):
                x, b = s["x"][i].data_ptr(), w["bias"].data_ptr()
                oco.matvec_group(Q8_0, [w["k"].data_ptr(), w["v"].data_ptr()], x,
                                 [out["k"][i].data_ptr(), out["v"][i].data_ptr()], _matrix(2880, 512, bias=1), D.BF16, D.F32,
                                 w["norm"].data_ptr(), EPSILON, True, [b, b + 4 * 512], stream=_stream())
                oco.matvec_norm(Q8_0, w["q"].data_ptr(), x, w["norm"].data_ptr(), EPSILON, out["q"][i].data_ptr(),
                                _matrix(2880, 4096, bias=1), True, D.F32, b + 4 * 1024, stream=_stream())
                oco.matvec(Q8_0, w["o"].data_ptr(), s["mixed"][i].data_ptr(), out["o"][i].data_ptr(),
                           _matrix(4096, 2880, bias=1), D.BF16, D.F32, b + 4 * 5120, stream=_stream())
        return _recorded(s, launch)
    if kind == "ffn":
        L = case["layers"]
        s["out"] = {"gate": empty((L, 12288)), "up": empty((L, 12288)), "down": empty((L, 4096))}

        def launch():
            out = s["out"]
            for i, w in enumerate(s["layers"]):
                oco.matvec_group(Q4_K, [w["gate"].data_ptr(), w["up"].data_ptr()], s["x"][i].data_ptr(),
                                 [out["gate"][i].data_ptr(), out["up"][i].data_ptr()], _matrix(4096, 12288), D.BF16, D.F32,
                                 w["norm"].data_ptr(), EPSILON, True, stream=_stream())
                oco.matvec(Q6_K, w["down"].data_ptr(), s["act"][i].data_ptr(), out["down"][i].data_ptr(),
                           _matrix(12288, 4096), stream=_stream())
        return _recorded(s, launch)
    if kind == "matvec":
        s["out"] = empty((case["layers"], case["n"]))
        dt = D.F32 if case["x"] == "f32" else D.BF16

        def launch():
            for i, w in enumerate(s["w"]):
                oco.matvec(case["format"], w.data_ptr(), s["x"][i].data_ptr(), s["out"][i].data_ptr(),
                           _matrix(case["k"], case["n"]), dt, D.F32, stream=_stream())
        return _recorded(s, launch)
    if kind == "head":
        n = case["n"]
        s["out"] = {"logits": empty(n), "token": empty(1, dtype=torch.int32)}
        need = oco.argmax_workspace(n)
        s["workspace"] = empty(max(need, 4), dtype=torch.uint8)

        def launch():
            logits = s["out"]["logits"].data_ptr()
            oco.matvec(Q6_K, s["w"][0].data_ptr(), s["x"].data_ptr(), logits, _matrix(case["k"], n), stream=_stream())
            oco.argmax(logits, n, s["out"]["token"].data_ptr(), _stream(), s["workspace"].data_ptr(), need)
        return _recorded(s, launch)
    if kind == "experts":
        fmt, hidden, ffn, experts, k = BANKS[case["bank"]]
        L, t, biased = case["layers"], case["tokens"], case["bank"] == "gpt_oss_20b"
        for w in s["layers"]:
            w["bank"] = oco.ExpertBank(
                fmt, hidden, ffn, experts, k, *[w[p].data_ptr() for p in ("gate", "up", "down")],
                *[b if b is None else b.data_ptr() for b in w["biases"]],
                activation=oco.Activation.SWIGLU_CLIPPED if biased else oco.Activation.SWIGLU, up_bias_one=biased)
        s["workspace"] = oco.DeviceBuffer(s["layers"][0]["bank"].workspace_bytes(t))
        s["normed"] = empty((t, hidden), dtype=torch.bfloat16)
        s["out"] = {"rows": empty((L, t, hidden), dtype=torch.bfloat16), "ids": empty((L, t, k), dtype=torch.int32),
                    "probs": empty((L, t, k))}
        return _recorded(s, functools.partial(_experts, s, _stream())) if t <= 16 else s
    # products of several rows: decode batches are replayed as the matvecs are, prompts called as they come
    n, k, m = case["n"], case["k"], case["m"]
    if kind == "norm_matmul":
        s["bytes"] = oco.matmul_workspace(MXFP4, _matrix(k, n, m))
        s["out"] = empty((m, n), dtype=torch.bfloat16)
    else:
        s["bytes"] = oco.matmul_workspace(case["format"], _matrix(k, n, m))
        s["out"] = empty((case["layers"], m, n), dtype=torch.bfloat16 if case["y"] == "bf16" else torch.float32)
    s["workspace"] = empty(max(s["bytes"], 256), dtype=torch.uint8)
    return _recorded(s, functools.partial(_matmul, s, _stream())) if m <= 16 else s


def _experts(s, stream):
    """Residual rows of the tokens, then per layer: norm, router, experts, added to the residual."""
    case, out = s["case"], s["out"]
    _, hidden, _, _, _ = BANKS[case["bank"]]
    t = case["tokens"]
    oco.embed(oco.WeightFormat.Bf16, s["table"].data_ptr(), hidden, VOCABULARY, s["tokens"].data_ptr(),
              case["layers"] * t, out["rows"].data_ptr(), stream=stream)
    for i, w in enumerate(s["layers"]):
        rows = out["rows"][i].data_ptr()
        oco.norm(rows, w["norm"].data_ptr(), s["normed"].data_ptr(), t, hidden, EPSILON, True, stream=stream)
        w["bank"].forward(w["router"].data_ptr(), w["router_bias"].data_ptr() if w["router_bias"] is not None else None,
                          s["normed"].data_ptr(), oco.DType.BF16, t, rows, out["ids"][i].data_ptr(),
                          out["probs"][i].data_ptr(), workspace=s["workspace"], stream=stream)


def _matmul(s, stream):
    case = s["case"]
    p, dt = _matrix(case["k"], case["n"], case["m"]), oco.DType.BF16 if case["y"] == "bf16" else oco.DType.F32
    for i, w in enumerate(s["w"]):
        oco.matmul(case["format"], w.data_ptr(), s["x"][i].data_ptr(), s["out"][i].data_ptr(), p, oco.DType.BF16, dt,
                   stream=stream, workspace=s["workspace"].data_ptr(), workspace_bytes=s["bytes"])


def run(s):
    case = s["case"]
    if "graph" in s:
        s["graph"].launch()
    elif case["kind"] == "experts":
        _experts(s, None)
    elif case["kind"] == "matmul":
        _matmul(s, None)
    else:
        n, k, m = case["n"], case["k"], case["m"]
        split = s["workspace"].data_ptr()
        oco.norm_mx_split(s["x"].data_ptr(), s["norm"].data_ptr(), None, m, k, EPSILON, True, split, s["bytes"])
        oco.matmul_mx_split(s["w"][0].data_ptr(), split, s["bytes"], s["out"].data_ptr(), _matrix(k, n, m),
                            oco.DType.BF16)
    return s["out"]


# ---- what a pass has to do, and how exact its results are ---------------------------------------------

def _weight_bytes(fmt, n, k):
    unit, size = BLOCKS[fmt]
    return n * (k // unit) * size


def work(case):
    kind, L = case["kind"], case.get("layers", 1)
    if kind == "attention":
        shapes = [(4096, 2880), (512, 2880), (512, 2880), (2880, 4096)]
        byte = sum(_weight_bytes(Q8_0, n, k) + 8 * n for n, k in shapes) + 2 * (2880 + 4096) + 4 * 2880
        return {"bytes": L * byte, "flops": L * sum(2 * n * k for n, k in shapes)}
    if kind == "ffn":
        byte = 2 * _weight_bytes(Q4_K, 12288, 4096) + _weight_bytes(Q6_K, 4096, 12288) + 6 * 4096 + 12 * 12288 + 4 * 4096
        return {"bytes": L * byte, "flops": L * 6 * 12288 * 4096}
    if kind == "experts":
        fmt, hidden, ffn, experts, k = BANKS[case["bank"]]
        t = case["tokens"]
        hit = experts * (1.0 - (1.0 - k / experts) ** t)  # distinct experts expected under even routing
        byte = hit * 3 * _weight_bytes(fmt, ffn, hidden) + 4 * hidden * (experts + 1) + t * (4 * hidden + 8 * k)
        return {"bytes": L * byte, "flops": L * 2 * t * (3 * k * hidden * ffn + experts * hidden)}
    fmt = Q6_K if kind == "head" else MXFP4 if kind == "norm_matmul" else case["format"]
    n, k, m = case["n"], case["k"], case.get("m", 1)
    x = 4 if case.get("x") == "f32" or kind == "head" else 2
    y = 4 if kind in ("matvec", "head") or case.get("y") == "f32" else 2
    byte = _weight_bytes(fmt, n, k) + x * m * k + y * m * n + (4 * k if kind == "norm_matmul" else 0)
    return {"bytes": L * byte, "flops": L * 2 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matvec", "head"):  # 32-bit sums of exact weights: up to 4.6e-7 from exact()
        return {"rel": 2e-6}
    if kind in ("attention", "ffn"):  # the same behind a bf16 norm, whose rounding may fall the other way in a few places
        return {"rel": 1e-4}
    if kind == "experts":  # bf16 residual rows (2.9e-3); ids may differ where two logits tie to 32-bit sums
        return {"rel": 1e-2, "differ": 0.002}
    if kind == "norm_matmul" or case["y"] == "bf16":  # bf16 results: 1.7e-3
        return {"rel": 7e-3}
    return {"rel": 2e-3 if case["format"] == MXFP4 else 1e-3}  # split (4e-4) or half (2.1e-4) activations, f32 results


def _normed(x, w):
    """RMS norm rows as the library stores them: bf16."""
    v = x.double()
    v = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPSILON) * w.double()
    return v.to(torch.bfloat16).double()


def _bf16(v):
    return v.to(torch.bfloat16).double()


def _expert_rows(case, w, resid):
    fmt, hidden, ffn, experts, k = BANKS[case["bank"]]
    x = _normed(resid, w["norm"])
    logits = x @ _bf16(w["router"]).T + (0.0 if w["router_bias"] is None else _bf16(w["router_bias"]))
    ids = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :k]
    probs = _bf16(torch.softmax(_bf16(logits.gather(1, ids)), 1))
    biases = [torch.zeros(experts * r, dtype=torch.float64, device="cuda") if b is None else b.double()
              for b, r in zip(w["biases"], (ffn, ffn, hidden))]
    out = resid.double().clone()
    for e in range(experts):
        token, slot = torch.nonzero(ids == e, as_tuple=True)
        if not len(token):
            continue
        part = {}
        for p, r, c in (("gate", ffn, hidden), ("up", ffn, hidden), ("down", hidden, ffn)):
            size = w[p].numel() // experts
            part[p] = decoded(fmt, w[p][e * size:(e + 1) * size], r, c)
        g = x[token] @ part["gate"].T + _bf16(biases[0][e * ffn:(e + 1) * ffn])
        if case["bank"] == "gpt_oss_20b":  # clipped SwiGLU, up + 1
            g = g.clamp(max=7.0)
            u = (x[token] @ part["up"].T + _bf16(biases[1][e * ffn:(e + 1) * ffn] + 1.0)).clamp(-6.0, 8.0)
            act = torch.sigmoid(1.702 * g) * g * u
        else:
            act = torch.sigmoid(g) * g * (x[token] @ part["up"].T)
        down = act @ part["down"].T + _bf16(biases[2][e * hidden:(e + 1) * hidden])
        out.index_add_(0, token, down * probs[token, slot].unsqueeze(1))
    return out, ids, probs


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "attention":
        out = {p: [] for p in ("k", "v", "q", "o")}
        for i, w in enumerate(s["layers"]):
            x, b, at = _normed(s["x"][i], w["norm"]), _bf16(w["bias"]), 0
            for p, n, k in (("k", 512, 2880), ("v", 512, 2880), ("q", 4096, 2880), ("o", 2880, 4096)):
                row = s["mixed"][i].double() if p == "o" else x
                out[p].append(decoded(Q8_0, w[p], n, k) @ row + b[at:at + n])
                at += n
        return {p: torch.stack(v) for p, v in out.items()}
    if kind == "ffn":
        out = {"gate": [], "up": [], "down": []}
        for i, w in enumerate(s["layers"]):
            x = _normed(s["x"][i], w["norm"])
            out["gate"].append(decoded(Q4_K, w["gate"], 12288, 4096) @ x)
            out["up"].append(decoded(Q4_K, w["up"], 12288, 4096) @ x)
            out["down"].append(decoded(Q6_K, w["down"], 4096, 12288) @ s["act"][i].double())
        return {p: torch.stack(v) for p, v in out.items()}
    if kind == "experts":
        t, hidden = case["tokens"], BANKS[case["bank"]][1]
        rows = s["table"][s["tokens"].long()].view(case["layers"], t, hidden)
        got = [_expert_rows(case, w, rows[i]) for i, w in enumerate(s["layers"])]
        return {"rows": torch.stack([g[0] for g in got]), "ids": torch.stack([g[1] for g in got]).int(),
                "probs": torch.stack([g[2] for g in got])}
    n, k = case["n"], case["k"]
    fmt = Q6_K if kind == "head" else MXFP4 if kind == "norm_matmul" else case["format"]
    got = []
    for i, w in enumerate(s["w"]):
        x = _normed(s["x"][i], s["norm"]) if kind == "norm_matmul" else s["x"][i].double()
        got.append(x @ decoded(fmt, w, n, k).T)
    if kind == "head":
        return {"logits": got[0][0], "token": torch.argmax(got[0][0]).int().view(1)}
    if kind == "norm_matmul":
        return got[0]
    return torch.stack([g[0] for g in got]) if kind == "matvec" else torch.stack(got)
