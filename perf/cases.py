"""The work that is timed: quantized linear layers and MoE experts as a serving program calls them.

A case is one call (or the calls of one step) of the public entry points on
inputs made from a seed.  `listed()` holds the fixed cases, `draw(rng)` more of
the same ranges:

- linear: one projection of a decode step (1-16 rows), a short or ragged
  prompt, or a prefill chunk of up to 2048 rows; bfloat16 or float16; affine
  codes of 2, 3, 4, 5, 6 or 8 bits or mxfp4; with and without a layer bias;
  rarely the untransposed product.
- multi: q/k/v or gate/up of one activation in one call.
- gather: the experts of a routed MoE layer, from one token (unsorted) to a
  prefill chunk (rows sorted by expert).
- moe: the fused single-token expert block.
- convert: quantize one matrix and dequantize another, as a loader does.
"""
import math

import torch

import mlxcel_amd as mq

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


# ---- cases -------------------------------------------------------------------


def _linear(name, M, N, K, bits=4, gs=64, mode="affine", dtype="bf16", bias=False, transpose=True):
    return {"name": name, "kind": "linear", "M": M, "N": N, "K": K, "bits": bits, "gs": gs, "mode": mode,
            "dtype": dtype, "bias": bias, "transpose": transpose}


def listed():
    return [
        # one token through an attention output projection: the smallest call, latency
        _linear("decode_o_1", 1, 4096, 4096),
        # one token through the vocabulary head: the largest decode read
        _linear("decode_head_1", 1, 151936, 4096),
        # 8 sequences, q/k/v in one call
        {"name": "decode_qkv_8", "kind": "multi", "M": 8, "Ns": "4096,1024,1024", "K": 4096, "bits": 4, "gs": 64,
         "mode": "affine", "dtype": "bf16"},
        # 16 sequences through an 8-bit MLP down projection
        _linear("decode_down_16_8bit", 16, 4096, 14336, bits=8),
        # 8 sequences through the gate projection of a 3-bit checkpoint
        _linear("decode_gate_8_3bit", 8, 14336, 4096, bits=3),
        # a ragged 333-token prompt, float16, a fused q/k/v projection with a layer bias
        _linear("prefill_qkv_333_f16", 333, 6144, 4096, dtype="f16", bias=True),
        # a 512-token prefill chunk through the gate projection of a 6-bit checkpoint
        _linear("prefill_gate_512_6bit", 512, 14336, 4096, bits=6),
        # a 2048-token prefill chunk through the gate projection
        _linear("prefill_gate_2048", 2048, 14336, 4096),
        # 16 tokens through 32 mxfp4 experts, top 4 (gate and up in one matrix)
        {"name": "experts_mxfp4_16", "kind": "gather", "T": 16, "top": 4, "E": 32, "N": 5760, "K": 2880, "bits": 4,
         "gs": 32, "mode": "mxfp4"},
        # a 512-token chunk through 128 affine 4-bit experts, top 8
        {"name": "experts_affine_512", "kind": "gather", "T": 512, "top": 8, "E": 128, "N": 768, "K": 2048, "bits": 4,
         "gs": 64, "mode": "affine"},
        # one token through the fused expert block
        {"name": "moe_token", "kind": "moe", "E": 128, "din": 2048, "dff": 768, "k": 8, "gu_bits": 4, "d_bits": 4,
         "gs": 64},
        # loading: quantize one MLP matrix, dequantize another
        {"name": "convert_mlp", "kind": "convert", "rows": 14336, "cols": 4096, "bits": 4, "gs": 64,
         "mode": "affine"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _multiple(rng, lo, hi, of):
    return max(of, _log_int(rng, lo, hi) // of * of)


# products of this many multiply-adds cost no more than the listed 512-row one
_MOST = 512 * 14336 * 4096


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "multi", "gather", "gather", "moe", "convert"))
    if kind in ("linear", "multi"):
        M = _log_int(rng, 1, 2048)
        gs = rng.choice((32, 64, 64, 64, 128))
        K = _multiple(rng, 512, 14336, gs)
        dtype = rng.choice(("bf16", "bf16", "f16"))
        if kind == "multi":
            kv = _log_int(rng, 128, 2048)
            Ns = rng.choice(("%d,%d,%d" % (_log_int(rng, 1024, 8192), kv, kv), "%d,%d" % ((_log_int(rng, 1024, 14336),) * 2)))
            M = min(M, max(1, _MOST // (sum(int(n) for n in Ns.split(",")) * K)))
            return {"kind": "multi", "M": M, "Ns": Ns, "K": K, "bits": rng.choice((4, 4, 8)), "gs": gs,
                    "mode": "affine", "dtype": dtype}
        bits = rng.choice((4, 4, 4, 8, 8, 2, 3, 5, 6))
        mode, transpose = "affine", True
        N = _log_int(rng, 256, 16384)
        if rng.random() < 0.1:
            mode, bits, gs = "mxfp4", 4, 32
        elif rng.random() < 0.1:
            transpose, N = False, max(gs, N // gs * gs)
        M = min(M, max(1, _MOST // (N * K)))
        return {"kind": "linear", "M": M, "N": N, "K": K, "bits": bits, "gs": gs, "mode": mode, "dtype": dtype,
                "bias": transpose and rng.random() < 0.25, "transpose": transpose}
    if kind == "gather":
        E = rng.choice((8, 16, 32, 60, 64, 128))
        mode = rng.choice(("affine", "affine", "mxfp4"))
        bits, gs = (4, 32) if mode == "mxfp4" else (rng.choice((4, 4, 8)), rng.choice((32, 64, 64, 128)))
        K = _multiple(rng, 512, 4096, 128)
        N = _log_int(rng, 512, 5760)
        top = rng.choice((1, 2, 4, 6, 8))
        T = _log_int(rng, 1, 1024)
        T = min(T, max(1, _MOST // 8 // (top * N * K)))
        return {"kind": "gather", "T": T, "top": top, "E": E, "N": N, "K": K, "bits": bits, "gs": gs, "mode": mode}
    if kind == "moe":
        return {"kind": "moe", "E": rng.choice((8, 32, 60, 128)), "din": _multiple(rng, 1024, 4096, 128),
                "dff": _multiple(rng, 512, 2048, 128), "k": rng.choice((1, 2, 4, 6, 8)),
                "gu_bits": rng.choice((4, 4, 8)), "d_bits": rng.choice((4, 4, 6, 8)), "gs": rng.choice((32, 64, 128))}
    mode = rng.choice(("affine", "affine", "affine", "mxfp4"))
    bits, gs = (4, 32) if mode == "mxfp4" else (rng.choice((2, 4, 4, 6, 8)), rng.choice((32, 64, 64, 128)))
    return {"kind": "convert", "rows": _log_int(rng, 128, 14336), "cols": _multiple(rng, 512, 4096, 128),
            "bits": bits, "gs": gs, "mode": mode}


# ---- inputs ------------------------------------------------------------------


def _pack(q, bits):
    """Codes [rows, cols] as the little-endian bit stream in uint32 words [rows, cols * bits / 32]."""
    rows, cols = q.shape
    q = q.to(torch.int64).view(rows, cols // 32, 32)
    words = torch.zeros((rows, cols // 32, bits), dtype=torch.int64, device=q.device)
    for i in range(32):
        at, shift = divmod(i * bits, 32)
        words[:, :, at] |= (q[:, :, i] << shift) & 0xFFFFFFFF
        if shift + bits > 32:
            words[:, :, at + 1] |= q[:, :, i] >> (32 - shift)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    return words.view(rows, cols * bits // 32).view(torch.uint32)


def _unpack(w, bits):
    """The codes of `_pack`, as int64."""
    rows = w.shape[0]
    words = (w.view(torch.int32).to(torch.int64) & 0xFFFFFFFF).view(rows, -1, bits)
    out = torch.empty((rows, words.shape[1], 32), dtype=torch.int64, device=w.device)
    for i in range(32):
        at, shift = divmod(i * bits, 32)
        v = words[:, :, at] >> shift
        if shift + bits > 32:
            v = v | (words[:, :, at + 1] << (32 - shift))
        out[:, :, i] = v & ((1 << bits) - 1)
    return out.view(rows, -1)


def _weights(gen, rows, cols, c, bits, dtype):
    """(w, scales, biases) of a matrix ~ N(0, 0.02), grouped along its last dimension."""
    gs, parts = c["gs"], []
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        m = torch.randn((min(step, rows - r), cols), generator=gen, device="cuda") * 0.02
        g = m.view(m.shape[0], cols // gs, gs)
        if c.get("mode", "affine") == "mxfp4":
            e = torch.floor(torch.log2(g.abs().amax(-1).clamp_min(1e-30))) - 2
            level = (g / torch.exp2(e)[..., None]).view(m.shape).clamp(-6, 6)
            edge = torch.tensor([(a + b) / 2 for a, b in zip(_E2M1, _E2M1[1:])], device="cuda")
            q = torch.bucketize(level.abs(), edge) + 8 * (level < 0)
            parts.append((_pack(q, 4), (e + 127).to(torch.uint8), None))
        else:
            lo, hi = g.amin(-1), g.amax(-1)
            s = ((hi - lo) / (2 ** bits - 1)).to(dtype)
            b = lo.to(dtype)
            q = ((g - b.float()[..., None]) / s.float()[..., None]).round().clamp(0, 2 ** bits - 1)
            parts.append((_pack(q.view(m.shape), bits), s, b))
    w, s, b = zip(*parts)
    return torch.cat([v.view(torch.int32) for v in w]).view(torch.uint32), torch.cat(s), None if b[0] is None else torch.cat(b)


def _values(w, s, b, c, bits):
    """The dequantized matrix in 64 bits."""
    q = _unpack(w, bits)
    if c.get("mode", "affine") == "mxfp4":
        table = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device="cuda")
        v, k = table[q], torch.exp2(s.double() - 127)
        return (v.view(*k.shape, c["gs"]) * k[..., None]).view(q.shape)
    g = q.view(q.shape[0], -1, c["gs"]).double()
    return (g * s.double()[..., None] + b.double()[..., None]).view(q.shape)


def _stack(t, *shape):
    return None if t is None else t.view(*shape)


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": c}
    if c["kind"] == "linear":
        dtype = _DTYPES[c["dtype"]]
        s["x"] = torch.randn((c["M"], c["K"]), generator=gen, device="cuda").to(dtype)
        rows, cols = (c["N"], c["K"]) if c["transpose"] else (c["K"], c["N"])
        s["w"] = _weights(gen, rows, cols, c, c["bits"], dtype)
        s["bias"] = torch.randn((c["N"],), generator=gen, device="cuda").to(dtype) if c["bias"] and c["transpose"] else None
    elif c["kind"] == "multi":
        dtype = _DTYPES[c["dtype"]]
        s["x"] = torch.randn((c["M"], c["K"]), generator=gen, device="cuda").to(dtype)
        s["ws"] = [_weights(gen, int(n), c["K"], c, c["bits"], dtype) for n in c["Ns"].split(",")]
    elif c["kind"] == "gather":
        E, T, top = c["E"], c["T"], c["top"]
        w = _weights(gen, E * c["N"], c["K"], c, c["bits"], torch.bfloat16)
        s["w"] = tuple(_stack(t, E, c["N"], -1) for t in w)
        x = torch.randn((T, c["K"]), generator=gen, device="cuda").to(torch.bfloat16)
        ids = torch.rand((T, E), generator=gen, device="cuda").topk(top, dim=-1).indices.to(torch.int32)
        s["sorted"] = T * top >= 64
        if s["sorted"]:  # the caller sorts the rows by expert, as its MoE layer does
            order = torch.sort(ids.view(-1), stable=True)
            s["ids"] = order.values.contiguous()
            s["x"] = x[order.indices // top].view(T * top, 1, c["K"]).contiguous()
        else:
            s["ids"], s["x"] = ids, x.view(T, 1, 1, c["K"])
    elif c["kind"] == "moe":
        E, din, dff, k = c["E"], c["din"], c["dff"], c["k"]
        s["x"] = torch.randn((din,), generator=gen, device="cuda").to(torch.bfloat16)
        s["ids"] = torch.rand((E,), generator=gen, device="cuda").topk(k).indices.to(torch.int32)
        s["scores"] = torch.softmax(torch.randn((k,), generator=gen, device="cuda"), 0)
        for name, rows, cols, bits in (("gate", dff, din, c["gu_bits"]), ("up", dff, din, c["gu_bits"]), ("down", din, dff, c["d_bits"])):
            w = _weights(gen, E * rows, cols, c, bits, torch.bfloat16)
            s[name] = tuple(_stack(t, E, rows, -1) for t in w)
    else:
        s["m"] = (torch.randn((c["rows"], c["cols"]), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
        s["w"] = _weights(gen, c["rows"], c["cols"], c, c["bits"], torch.bfloat16)
    return s


# ---- one pass ------------------------------------------------------------------


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "linear":
        w, sc, b = s["w"]
        if s["bias"] is not None:
            return mq.quantized_linear(s["x"], w, sc, b, s["bias"], c["gs"], c["bits"], c["mode"])
        return mq.quantized_matmul(s["x"], w, sc, b, c["transpose"], c["gs"], c["bits"], c["mode"])
    if c["kind"] == "multi":
        ws, scs, bs = zip(*s["ws"])
        return mq.quantized_matmul_multi(s["x"], ws, scs, bs, c["gs"], c["bits"], c["mode"])
    if c["kind"] == "gather":
        w, sc, b = s["w"]
        return mq.gather_qmm(s["x"], w, sc, b, None, s["ids"], True, c["gs"], c["bits"], c["mode"], s["sorted"])
    if c["kind"] == "moe":
        return mq.fused_moe_expert(s["x"], s["ids"], *s["gate"], *s["up"], *s["down"], s["scores"], c["din"], c["dff"],
                                   c["k"], c["gu_bits"], c["d_bits"], c["gs"])
    w, sc, b = s["w"]
    codes, *scales = mq.quantize(s["m"], c["gs"], c["bits"], c["mode"])
    return {"quantized": [codes.view(torch.int32), *scales],
            "dequantized": mq.dequantize(w, sc, b, c["gs"], c["bits"], c["mode"])}


# ---- what a pass cannot do without ----------------------------------------------


def _matrix_bytes(rows, cols, c, bits):
    return rows * cols * bits // 8 + rows * (cols // c["gs"]) * (1 if c.get("mode") == "mxfp4" else 4)


def work(case):
    c = case
    if c["kind"] == "linear":
        rows, cols = (c["N"], c["K"]) if c["transpose"] else (c["K"], c["N"])
        return {"bytes": _matrix_bytes(rows, cols, c, c["bits"]) + 2 * c["M"] * (c["N"] + c["K"]),
                "flops": 2 * c["M"] * c["N"] * c["K"]}
    if c["kind"] == "multi":
        N = sum(int(n) for n in c["Ns"].split(","))
        return {"bytes": _matrix_bytes(N, c["K"], c, c["bits"]) + 2 * c["M"] * (N + c["K"]), "flops": 2 * c["M"] * N * c["K"]}
    if c["kind"] == "gather":
        B = c["T"] * c["top"]
        touched = c["E"] * (1 - (1 - c["top"] / c["E"]) ** c["T"])
        x_rows = B if B >= 64 else c["T"]
        return {"bytes": touched * _matrix_bytes(c["N"], c["K"], c, c["bits"]) + 2 * (x_rows * c["K"] + B * c["N"]) + 4 * B,
                "flops": 2 * B * c["N"] * c["K"]}
    if c["kind"] == "moe":
        n = c["k"] * (2 * _matrix_bytes(c["dff"], c["din"], c, c["gu_bits"]) + _matrix_bytes(c["din"], c["dff"], c, c["d_bits"]))
        return {"bytes": n + 4 * c["din"] + 8 * c["k"], "flops": 6 * c["k"] * c["din"] * c["dff"]}
    n = c["rows"] * c["cols"]
    return {"bytes": 2 * (2 * n + _matrix_bytes(c["rows"], c["cols"], c, c["bits"])), "flops": 0}


# ---- what the results are compared with -----------------------------------------


def tolerance(case):
    if case["kind"] == "convert":
        return "exact"
    if case.get("dtype") == "f16":
        return {"rel": 0.002}
    return {"rel": 0.01}


def _rounds(n, step):
    return [(r, min(n, r + step)) for r in range(0, n, step)]


def exact(case, seed):
    c, s = case, prepare(case, seed)

    def product(x, w, sc, b, bits):
        # x @ values(w).T, a block of weight rows at a time
        return torch.cat([x @ _values(w[r:e], sc[r:e], None if b is None else b[r:e], c, bits).T
                          for r, e in _rounds(w.shape[0], max(1, (1 << 25) // x.shape[-1]))], -1)

    if c["kind"] == "linear":
        x = s["x"].double()
        y = product(x, *s["w"], c["bits"]) if c["transpose"] else x @ _values(*s["w"], c, c["bits"])
        return y if s["bias"] is None else y + s["bias"].double()
    if c["kind"] == "multi":
        return [product(s["x"].double(), *w, c["bits"]) for w in s["ws"]]
    if c["kind"] == "gather":
        w, sc, b = s["w"]
        ids = s["ids"].view(-1).long()
        x = s["x"].view(-1, c["K"]).double()
        x = x if s["sorted"] else x.repeat_interleave(c["top"], 0)
        y = torch.empty((ids.numel(), c["N"]), dtype=torch.float64, device="cuda")
        for e in ids.unique().tolist():
            at = ids == e
            y[at] = product(x[at], w[e], sc[e], None if b is None else b[e], c["bits"])
        return y.view(-1, 1, c["N"]) if s["sorted"] else y.view(c["T"], c["top"], 1, c["N"])
    if c["kind"] == "moe":
        x, y = s["x"].double(), 0.0
        for j, e in enumerate(s["ids"].tolist()):
            gate, up = (product(x[None], *(t[e] for t in s[n]), c["gu_bits"])[0] for n in ("gate", "up"))
            h = gate / (1 + torch.exp(-gate)) * up
            y = y + s["scores"][j].double() * product(h[None], *(t[e] for t in s["down"]), c["d_bits"])[0]
        return y
    return {"quantized": [None] * (2 if c["mode"] == "mxfp4" else 3), "dequantized": _values(*s["w"], c, c["bits"])}
