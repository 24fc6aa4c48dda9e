"""The work whose speed is watched: decoder blocks of quantized linear layers, as an inference program runs them.

A case is one pass through the layers of a model part: per block RMSNorm, the q / k / v / o projections and the gated
MLP, then the final norm and the LM head (the attention between the projections runs elsewhere: its output is an input
here).  Decode passes have one row (a single sequence) or a few (a batch, a speculative step), prefill passes the rows
of a prompt.  A serving program captures its decode step into a HIP graph once and replays it ("graph"); prompts, whose
length changes from call to call, and small interactive programs call the layers one by one.

Sizes are those of the repository's configurations, tests and benchmark (hidden / intermediate 4096 / 14336, 1024 / 3072,
5120 / 13824, 3584 / 18944; vocabularies of 128256, 151936 and 152064), row counts of a prompt or a batch are any number.
Weights are N(0, 0.02) quantized to their format, activations N(0, 1); trellis words are uniform bits, which decode to
normally distributed weights.
"""
from __future__ import annotations

import torch

from tattletale_amd import QuantGatedMLP, QuantLinear, formats as F
from tattletale_amd.qlinear import rmsnorm

DEVICE = "cuda"
EPS = 1e-5
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FORMATS = {"q8_0": F.Q8_0, "q4_k": F.Q4_K, "q6_k": F.Q6_K, "exl3": F.EXL3}
BYTES_PER_WEIGHT = {"q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}

#: fields of a case:
#: fmt     q8_0 | q4_k | q6_k | exl3, or q4_k_m: Q4_K with v, down and the head in Q6_K, the usual mixture
#: bits    bits per weight of the trellis format
#: hidden, q, kv, ffn, vocab   sizes (vocab 0: no head; a head is Q6_K unless the format is q8_0 or exl3)
#: rows    activation rows (tokens); head_rows of them reach the head: all of a decode pass, the last of a prompt
#: dtype   activation type, bias: biases on q / k / v, blocks: decoder blocks in a pass, graph: replayed as a HIP graph


def _case(name, fmt, hidden, q, kv, ffn, vocab, rows, dtype, blocks, graph, bits=0, bias=False):
    return {"name": name, "fmt": fmt, "bits": bits, "hidden": hidden, "q": q, "kv": kv, "ffn": ffn, "vocab": vocab,
            "rows": rows, "head_rows": rows if rows <= 64 else 1, "dtype": dtype, "bias": bias, "blocks": blocks,
            "graph": graph}


def listed():
    return [
        # a small model called layer by layer: what an interactive program without graphs pays, launches and host time
        _case("decode_1024_eager", "q4_k_m", 1024, 2048, 1024, 3072, 151936, 1, "bf16", 4, False),
        # the same model in its 8-bit form with fp32 activations (the operator's reference precision)
        _case("decode_1024_q8_f32", "q8_0", 1024, 2048, 1024, 3072, 0, 1, "f32", 4, True),
        # the usual single-sequence decode step, head included
        _case("decode_4096", "q4_k_m", 4096, 4096, 1024, 14336, 128256, 1, "bf16", 2, True),
        # a wider model without grouped heads, 6-bit, fp16
        _case("decode_5120_q6_f16", "q6_k", 5120, 5120, 5120, 13824, 32003, 1, "f16", 1, True),
        # 8-bit weights with fp32 activations at full size
        _case("decode_4096_q8_f32", "q8_0", 4096, 4096, 1024, 14336, 0, 1, "f32", 2, True),
        # a small batch of sequences, or a speculative step
        _case("decode_4096_rows8", "q4_k_m", 4096, 4096, 1024, 14336, 128256, 8, "bf16", 2, True),
        # a larger batch, odd row count, biases on q / k / v, long ragged MLP rows, fp16
        _case("decode_3584_rows43_f16", "q4_k", 3584, 3584, 512, 18944, 152064, 43, "f16", 1, True, bias=True),
        # prompts: short and odd, ordinary, long
        _case("prefill_5120_rows333_f16", "q6_k", 5120, 5120, 5120, 13824, 32003, 333, "f16", 1, False),
        _case("prefill_4096_rows512", "q4_k_m", 4096, 4096, 1024, 14336, 128256, 512, "bf16", 1, False),
        _case("prefill_4096_rows4096", "q4_k", 4096, 4096, 1024, 14336, 0, 4096, "bf16", 1, False),
        # trellis-coded weights, decode and prompt
        _case("exl3_decode_4096", "exl3", 4096, 4096, 1024, 14336, 0, 1, "f16", 2, True, bits=3),
        _case("exl3_prefill_4096_rows512", "exl3", 4096, 4096, 1024, 14336, 0, 512, "f16", 1, False, bits=3),
    ]


def _spread(rng, low, high, step):
    """A multiple of `step` from low to high, spread evenly over the logarithm."""
    v = low * (high / low) ** rng.random()
    return min(high, max(low, int(v / step + 0.5) * step))


def draw(rng):
    fmt = rng.choice(["q4_k_m", "q4_k_m", "q4_k", "q6_k", "q8_0", "exl3"])
    bits = rng.choice([2, 3, 4, 5, 6]) if fmt == "exl3" else 0
    dtype = rng.choice(["f16"] if fmt == "exl3" else ["bf16", "bf16", "f16", "f32"])
    hidden = _spread(rng, 768, 8192, 256)
    ffn = _spread(rng, 2 * hidden, 4 * hidden, 256)
    kv = max(256, hidden // rng.choice([1, 2, 4, 8]) // 128 * 128)
    kind = rng.choice(["one", "one", "few", "batch", "prompt", "prompt"])
    rows = {"one": 1, "few": rng.randint(2, 8), "batch": rng.randint(9, 64), "prompt": _spread(rng, 65, 4096, 1)}[kind]
    vocab = _spread(rng, 8001, 152001, 1) | 1 if fmt != "exl3" and rng.random() < 0.5 else 0
    case = _case("", fmt, hidden, hidden, kv, ffn, vocab, rows, dtype, 1, rows <= 64 and rng.random() < 0.75, bits,
                 rng.random() < 0.25)
    del case["name"]
    most = max(work(c)["flops"] for c in listed())
    while case["rows"] > 64 and work(case)["flops"] > most:          # no prompt larger than the largest listed one
        case["rows"] = max(65, case["rows"] // 2)
    return case


# ------------------------------------------------------------------------------------------------- weights
def _u8(t):
    return t.contiguous().view(torch.uint8)


def _pack_q8_0(w):
    d = (w.abs().amax(-1, keepdim=True) / 127).half()
    q = (w / d.float().clamp_min(1e-30)).round().clamp(-127, 127).to(torch.int8)
    return torch.cat([_u8(d), _u8(q)], -1)


def _pack_q4_k(w):
    """w (blocks, 256): 8 sub-blocks of 32 with 6-bit scales and minima, 4-bit quants."""
    s = w.view(-1, 8, 32)
    low = (-s.amin(-1)).clamp_min(0)
    scale = (s.amax(-1) + low) / 15
    d, dmin = (scale.amax(-1, keepdim=True) / 63).half(), (low.amax(-1, keepdim=True) / 63).half()
    df, mf = d.float().clamp_min(1e-30), dmin.float().clamp_min(1e-30)
    sc, mn = (scale / df).round().clamp(1, 63), (low / mf).round().clamp(0, 63)
    q = ((s + (mf * mn)[..., None]) / (df * sc)[..., None]).round().clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4) << 6, mn[:, :4] | (mn[:, 4:] >> 4) << 6,
                        (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], -1)
    q = q.view(-1, 4, 2, 32)
    return torch.cat([_u8(d), _u8(dmin), packed, (q[:, :, 0] | q[:, :, 1] << 4).reshape(-1, 128)], -1)


def _pack_q6_k(w):
    """w (blocks, 256): 16 sub-blocks of 16 with 8-bit scales, 6-bit quants."""
    s = w.view(-1, 16, 16)
    scale = s.abs().amax(-1) / 31
    d = (scale.amax(-1, keepdim=True) / 127).half()
    df = d.float().clamp_min(1e-30)
    sc = (scale / df).round().clamp(1, 127)
    q = ((s / (df * sc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(-1, 2, 4, 32)
    ql = torch.cat([(q[:, :, 0] & 15) | (q[:, :, 2] & 15) << 4, (q[:, :, 1] & 15) | (q[:, :, 3] & 15) << 4], -1)
    qh = q[:, :, 0] >> 4 | (q[:, :, 1] >> 4) << 2 | (q[:, :, 2] >> 4) << 4 | (q[:, :, 3] >> 4) << 6
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), _u8(sc.to(torch.int8)), _u8(d)], -1)


_PACK = {"q8_0": (_pack_q8_0, 32), "q4_k": (_pack_q4_k, 256), "q6_k": (_pack_q6_k, 256)}


def _layer(gen, fmt, bits, n_out, n_in, bias=None):
    if fmt == "exl3":
        trellis = torch.randint(-32768, 32768, (n_in // 16, n_out // 16, 16 * bits), generator=gen, device=DEVICE,
                                dtype=torch.int16)
        sign = [torch.randint(0, 2, (n,), generator=gen, device=DEVICE).half() * 2 - 1 for n in (n_in, n_out)]
        return QuantLinear.init(trellis, F.EXL3, n_in, n_out, bias, sign[0], sign[1] * 0.02, bits)
    pack, block = _PACK[fmt]
    part = max(1, (1 << 26) // n_in)
    rows = [pack((torch.randn(min(part, n_out - r), n_in, generator=gen, device=DEVICE) * 0.02).view(-1, block)).view(-1)
            for r in range(0, n_out, part)]
    return QuantLinear.init(torch.cat(rows), FORMATS[fmt], n_in, n_out, bias)


def _matrices(case):
    """(name, format, n_out, n_in) of the matrices of one block."""
    h, f = case["hidden"], case["fmt"]
    base, fine = ("q4_k", "q6_k") if f == "q4_k_m" else (f, f)
    return [("q", base, case["q"], h), ("k", base, case["kv"], h), ("v", fine, case["kv"], h), ("o", base, h, case["q"]),
            ("gate_up", base, 2 * case["ffn"], h), ("down", fine, h, case["ffn"])]


def _head_format(case):
    return case["fmt"] if case["fmt"] in ("q8_0", "exl3") else "q6_k"


# ------------------------------------------------------------------------------------------------- the pass
_stream = None


def _decode_stream():
    """The stream on which a program captures and replays its decode steps."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=gen, device=DEVICE) * scale + shift).to(dtype)

    h, m = case["hidden"], case["rows"]
    blocks = []
    for _ in range(case["blocks"]):
        layers = {}
        for name, fmt, n_out, n_in in _matrices(case):
            bias = normal(n_out, scale=0.1) if case["bias"] and name in "qkv" else None
            layers[name] = _layer(gen, fmt, case["bits"], n_out, n_in, bias)
        blocks.append({**layers, "mlp": QuantGatedMLP.init(layers["gate_up"], layers["down"]),
                       "norm1": normal(h, scale=0.1, shift=1.0), "norm2": normal(h, scale=0.1, shift=1.0),
                       "attn": normal(m, case["q"])})
    state = {"blocks": blocks, "x": normal(m, h), "norm": normal(h, scale=0.1, shift=1.0), "head": None,
             "head_rows": case["head_rows"], "graph": None}
    if case["vocab"]:
        state["head"] = _layer(gen, _head_format(case), case["bits"], case["vocab"], h)
    if case["graph"]:
        stream = _decode_stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _forward(state)                      # workspaces are made outside of the capture
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                out = _forward(state)
        state["graph"], state["out"] = graph, out
    return state


def _forward(state):
    hidden, residual = state["x"], None
    out = {"q": [], "k": [], "v": []}
    for b in state["blocks"]:
        normed, new = rmsnorm(hidden, b["norm1"], EPS, residual)
        residual = hidden if new is None else new
        for name in "qkv":
            out[name].append(b[name].forward(normed))
        normed, residual = rmsnorm(b["o"].forward(b["attn"]), b["norm2"], EPS, residual)
        hidden = b["mlp"].forward(normed)
    normed, residual = rmsnorm(hidden, state["norm"], EPS, residual)
    out["residual"], out["normed"] = residual, normed
    if state["head"] is not None:
        out["logits"] = state["head"].forward(normed[-state["head_rows"]:], out_dtype=torch.float32)
    return out


def run(state):
    if state["graph"] is None:
        return _forward(state)
    with torch.cuda.stream(_decode_stream()):
        state["graph"].replay()
    return state["out"]


def work(case):
    """Weights once, inputs once, outputs once; two operations per weight and row."""
    size = 4 if case["dtype"] == "f32" else 2
    h, m = case["hidden"], case["rows"]

    def weight(fmt, n_out, n_in):
        return n_out * n_in * (case["bits"] / 8 if fmt == "exl3" else BYTES_PER_WEIGHT[fmt])

    total = flops = 0.0
    for _, fmt, n_out, n_in in _matrices(case):
        total += weight(fmt, n_out, n_in)
        flops += 2.0 * m * n_out * n_in
    total += size * m * (2 * case["q"] + 2 * case["kv"])          # attention output in; q, k, v out
    total, flops = total * case["blocks"], flops * case["blocks"]
    total += size * m * 3 * h                                     # x in, residual and normed out
    if case["vocab"]:
        total += weight(_head_format(case), case["vocab"], h) + 4.0 * case["head_rows"] * case["vocab"]
        flops += 2.0 * case["head_rows"] * case["vocab"] * h
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Distances of a pass from the same pass in 64-bit arithmetic (activations rounded to their type between layers), over
    the listed and some drawn cases: bf16 0.8e-2, fp16 0.8e-3; fp32 0.7e-6 for one row on Q8_0, 1.4e-4 for one row on the
    K formats, whose decode reads activations as 15-bit fixed point per block, 5e-4 for several rows, which are scaled and
    rounded to fp16.  Allowed: about four times that, less for bf16."""
    if case["dtype"] != "f32":
        return {"rel": {"bf16": 2e-2, "f16": 3e-3}[case["dtype"]]}
    if case["rows"] > 1:
        return {"rel": 2e-3}
    return {"rel": 1e-5 if case["fmt"] == "q8_0" else 6e-4}
