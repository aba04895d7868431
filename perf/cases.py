"""Workloads of the NF4 streamed-weight path whose time is measured.

The path's users are a double-pass trainer over streamed NF4 layers (forward,
recompute, input gradients, weight gradients, re-quantization of what an
update changed) and programs that only run the forward on a few tokens.  Every
case goes through the public Python entry points.  Shapes are those of the 7B
and 70B decoder layers the benchmark uses, or generic ones beside them.

Inputs are made here in plain torch from a seed, the NF4 weights included
(normal values of weight scale, quantized by the codebook), so they do not
depend on the kernels under test, and ``exact`` can redo every product in 64
bits.
"""
import math

import torch

from aethelstream_amd import gemm, nf4, norm, stream

BLOCK = 64
GROUP = 256          # blocks per double-quant scale
SIGMA = 0.02         # weight scale

CODES = (-1.0, -0.6961928, -0.52507305, -0.3949175, -0.28444138, -0.18477343, -0.09105004, 0.0,
         0.0795803, 0.1609302, 0.2461123, 0.33791524, 0.44070983, 0.562617, 0.72295684, 1.0)

LAYER_7B = ((4096, 4096), (4096, 4096), (4096, 4096), (4096, 4096),
            (11008, 4096), (11008, 4096), (4096, 11008))


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------

def listed():
    return [
        # A single projection for one new token: the smallest call, all
        # latency (7B attention output).
        {"name": "fwd_one_token", "op": "fwd", "m": 1, "ns": "4096", "k": 4096, "block": BLOCK,
         "dq": True},
        # q/k/v of a 70B layer for a handful of sequences decoded together.
        {"name": "qkv_few_tokens", "op": "fwd", "m": 17, "ns": "8192,1024,1024", "k": 8192,
         "block": BLOCK, "dq": True},
        # The MLP block (norm, fused SwiGLU, down) on a short prompt, fp32
        # absmax as the reference's shards store it, generic widths.
        {"name": "mlp_short_prompt", "op": "mlp", "m": 100, "d": 5120, "ff": 13824, "dq": False},
        # gate/up of a 70B layer on a prompt of ragged length.
        {"name": "gate_up_ragged", "op": "fwd", "m": 777, "ns": "28672,28672", "k": 8192,
         "block": BLOCK, "dq": True},
        # The MLP block of a 7B layer at a training micro-batch.
        {"name": "mlp_training", "op": "mlp", "m": 4096, "d": 4096, "ff": 11008, "dq": True},
        # Input gradient of the 70B attention projections, small micro-batch.
        {"name": "dgrad_qkv_small_batch", "op": "dgrad", "m": 256, "ns": "8192,1024,1024",
         "k": 8192, "dq": True},
        # Input gradient of 70B gate/up at a full micro-batch: the largest.
        {"name": "dgrad_gate_up", "op": "dgrad", "m": 8192, "ns": "28672,28672", "k": 8192,
         "dq": True},
        # Weight gradients of 7B gate/up over two micro-batches, the second
        # accumulated onto the first.
        {"name": "wgrad_gate_up", "op": "wgrad", "m": 1000, "ns": "11008,11008", "k": 4096},
        # Re-quantization of an updated 70B gate matrix (bf16 values) into
        # its own double-quantized buffers.
        {"name": "requantize_update", "op": "requant", "rows": 28672, "cols": 8192, "bf16": True,
         "dq": True},
        # Quantization of an fp32 matrix with absmax blocks wider than 64,
        # which the shard index allows for each tensor; a row count that ends
        # in a partial launch.
        {"name": "quantize_block_128", "op": "quantize", "rows": 4099, "cols": 4096, "block": 128},
        # Dequantization of a whole 7B layer in one launch.
        {"name": "dequant_layer", "op": "dequant", "shapes": "7b", "f16": False, "dq": True},
        # Two 7B layers streamed from pinned host memory through the double
        # buffer, forward on 512 tokens.
        {"name": "stream_two_layers", "op": "stream", "m": 512, "layers": 2},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _multiple(rng, lo, hi, step):
    return max(lo, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    """A case of the ranges the listed ones stand for: forwards from 1 to
    8192 tokens, gradients from 64 (a micro-batch is not a decode step),
    any output width, reduction lengths that the formats allow."""
    biggest = max((work(c)["flops"], work(c)["bytes"]) for c in listed())
    while True:
        op = rng.choice(("fwd", "fwd", "mlp", "dgrad", "wgrad", "requant", "quantize", "dequant",
                         "stream"))
        case = {"op": op}
        if op == "fwd":
            count = rng.randint(1, 3)
            block = rng.choice((64, 64, 64, 128))
            case.update(m=_log_int(rng, 1, 8192),
                        ns=",".join(str(_log_int(rng, 512, 28672)) for _ in range(count)),
                        k=_multiple(rng, 1024, 28672, block), block=block,
                        dq=rng.random() < 0.6)
        elif op == "mlp":
            case.update(m=_log_int(rng, 1, 8192), d=_multiple(rng, 2048, 8192, 128),
                        ff=_multiple(rng, 4096, 28672, 64), dq=rng.random() < 0.6)
        elif op == "dgrad":
            count = rng.randint(1, 3)
            case.update(m=_log_int(rng, 64, 8192),
                        ns=",".join(str(_multiple(rng, 512, 28672, 64)) for _ in range(count)),
                        k=_multiple(rng, 1024, 28672, 64), dq=rng.random() < 0.6)
        elif op == "wgrad":
            count = rng.randint(1, 3)
            case.update(m=_log_int(rng, 64, 8192),
                        ns=",".join(str(_multiple(rng, 512, 28672, 8)) for _ in range(count)),
                        k=_multiple(rng, 1024, 16384, 8))
        elif op == "requant":
            case.update(rows=_log_int(rng, 512, 28672), cols=_multiple(rng, 1024, 8192, 64),
                        bf16=rng.random() < 0.5, dq=rng.random() < 0.7)
        elif op == "quantize":
            case.update(rows=_log_int(rng, 512, 16384), cols=_log_int(rng, 1000, 8192),
                        block=rng.choice((32, 64, 128, 256)))
        elif op == "dequant":
            case.update(shapes=";".join(f"{_log_int(rng, 512, 16384)}x{_multiple(rng, 1024, 8192, 64)}"
                                        for _ in range(rng.randint(1, 4))),
                        f16=rng.random() < 0.5, dq=rng.random() < 0.6)
            if case["f16"]:
                case["shapes"] = case["shapes"].split(";")[0]
        else:
            case.update(m=_log_int(rng, 1, 2048), layers=rng.randint(1, 3))
        w = work(case)
        if w["flops"] <= biggest[0] and w["bytes"] <= biggest[1]:
            return case


# --------------------------------------------------------------------------
# Inputs, in plain torch
# --------------------------------------------------------------------------

def _ints(text):
    return [int(v) for v in text.split(",")]


def _shapes(text):
    if text == "7b":
        return list(LAYER_7B)
    return [tuple(int(v) for v in s.split("x")) for s in text.split(";")]


def _normal(shape, seed, sigma, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, device="cuda", generator=g) * sigma).to(dtype)


def _quantized(rows, cols, seed, block, dq):
    """(packed bytes, absmax or None, (codes, scales) or None) of a normal
    matrix: nearest code of value / block absmax, even element in the high
    nibble; double-quantized absmax as an 8-bit code of 127 steps per group."""
    v = _normal((rows * cols // block, block), seed, SIGMA)
    absmax = v.abs().amax(1)
    v /= absmax.clamp(min=1e-8)[:, None]
    c = torch.tensor(CODES, device="cuda")
    idx = torch.bucketize(v, (c[:-1] + c[1:]) / 2, out_int32=True).to(torch.uint8).reshape(-1, 2)
    packed = (idx[:, 0] << 4) | idx[:, 1]
    if not dq:
        return packed, absmax, None
    nb = absmax.numel()
    groups = (nb + GROUP - 1) // GROUP
    padded = torch.zeros(groups * GROUP, device="cuda")
    padded[:nb] = absmax
    scale = padded.view(groups, GROUP).amax(1) / 127.0
    q = (padded.view(groups, GROUP) / scale[:, None]).round().clamp(0, 127).to(torch.uint8)
    return packed, None, (q.reshape(-1)[:nb].contiguous(), scale)


def _weight(rows, cols, seed, block=BLOCK, dq=True):
    packed, absmax, coded = _quantized(rows, cols, seed, block, dq)
    if coded is None:
        return nf4.Nf4Weight(packed=packed, absmax=absmax, shape=[rows, cols], block_size=block)
    return nf4.Nf4Weight(packed=packed, absmax=None, shape=[rows, cols], block_size=block,
                         absmax_q=coded[0], absmax_scale=coded[1], dq_group=GROUP)


def _product32(rows, cols, seed, block, dq):
    """code * absmax in fp32, the value every NF4 decode rounds."""
    packed, absmax, coded = _quantized(rows, cols, seed, block, dq)
    if coded is not None:
        q, scale = coded
        absmax = q.float() * scale.repeat_interleave(GROUP)[:q.numel()]
    nib = torch.stack((packed >> 4, packed & 15), 1).reshape(-1, block)
    return (torch.tensor(CODES, device="cuda")[nib.int()] * absmax[:, None]).view(rows, cols)


def _weight64(rows, cols, seed, block=BLOCK, dq=True):
    """The matrix the products use: the decoded weight is bf16 by definition."""
    return _product32(rows, cols, seed, block, dq).to(torch.bfloat16).double()


def _blob_layers(case, seed):
    layout = stream.LayerLayout([(f"w{i}", r, c) for i, (r, c) in enumerate(LAYER_7B)])
    pinned = []
    for l in range(case["layers"]):
        ws = [_weight(r, c, seed + 100 * l + i) for i, (r, c) in enumerate(LAYER_7B)]
        buf = stream.PinnedBuffer(layout.nbytes)
        layout.pack_into(buf.tensor, ws)
        pinned.append(buf)
    return layout, pinned


def prepare(case, seed):
    op = case["op"]
    seed = seed * 1000
    s = {"op": op}
    if op == "fwd":
        s["x"] = _normal((case["m"], case["k"]), seed, 1.0, torch.bfloat16)
        s["ws"] = [_weight(n, case["k"], seed + 1 + i, case["block"], case["dq"])
                   for i, n in enumerate(_ints(case["ns"]))]
    elif op == "mlp":
        d, ff = case["d"], case["ff"]
        s["x"] = _normal((case["m"], d), seed, 1.0)
        s["g"] = 1.0 + _normal((d,), seed + 1, 0.1)
        s["gate"], s["up"] = (_weight(ff, d, seed + 2 + i, BLOCK, case["dq"]) for i in range(2))
        s["down"] = _weight(d, ff, seed + 4, BLOCK, case["dq"])
    elif op == "dgrad":
        ns = _ints(case["ns"])
        s["dys"] = [_normal((case["m"], n), seed + i, 1e-3, torch.bfloat16)
                    for i, n in enumerate(ns)]
        s["ws"] = [_weight(n, case["k"], seed + 10 + i, BLOCK, case["dq"])
                   for i, n in enumerate(ns)]
    elif op == "wgrad":
        ns = _ints(case["ns"])
        s["batches"] = [([_normal((case["m"], n), seed + 10 * b + i, 1e-3, torch.bfloat16)
                          for i, n in enumerate(ns)],
                         _normal((case["m"], case["k"]), seed + 10 * b + 9, 1.0, torch.bfloat16))
                        for b in range(2)]
        s["outs"] = [torch.empty(n, case["k"], device="cuda") for n in ns]
    elif op == "requant":
        r, c = case["rows"], case["cols"]
        s["w"] = _weight(r, c, seed, BLOCK, case["dq"])
        s["values"] = _normal((r, c), seed + 1, SIGMA,
                              torch.bfloat16 if case["bf16"] else torch.float32)
    elif op == "quantize":
        s["values"] = _normal((case["rows"], case["cols"]), seed, SIGMA)
        s["block"] = case["block"]
    elif op == "dequant":
        s["f16"] = case["f16"]
        s["ws"] = [_weight(r, c, seed + i, BLOCK, case["dq"])
                   for i, (r, c) in enumerate(_shapes(case["shapes"]))]
        s["outs"] = [torch.empty(w.shape, device="cuda",
                                 dtype=torch.float16 if case["f16"] else torch.bfloat16)
                     for w in s["ws"]]
    else:
        s["x"] = _normal((case["m"], 4096), seed, 1.0, torch.bfloat16)
        s["layout"], s["pinned"] = _blob_layers(case, seed + 1)
        s["dbuf"] = stream.VramDoubleBuffer(s["layout"].nbytes)
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------

def run(s):
    op = s["op"]
    if op == "fwd":
        if len(s["ws"]) == 1:
            return [gemm.linear_fwd(s["x"], s["ws"][0])]
        return gemm.linear_fwd_grouped(s["x"], s["ws"])
    if op == "mlp":
        y, rms = norm.rms_norm_fwd(s["x"], s["g"])
        hidden = gemm.linear_swiglu(y, s["gate"], s["up"])
        return [y, rms, hidden, gemm.linear_fwd(hidden, s["down"])]
    if op == "dgrad":
        if len(s["ws"]) == 1:
            return [gemm.linear_dgrad(s["dys"][0], s["ws"][0])]
        return [gemm.linear_dgrad_sum(s["dys"], s["ws"])]
    if op == "wgrad":
        for i, (dys, x) in enumerate(s["batches"]):
            gemm.linear_wgrad_grouped(dys, x, s["outs"], accumulate=i > 0)
        return s["outs"]
    if op == "requant":
        w = nf4.requantize_(s["w"], s["values"])
        return [w.packed, w.absmax_q, w.absmax_scale] if w.double_quant else [w.packed, w.absmax]
    if op == "quantize":
        r = nf4.quantize_nf4(s["values"], s["block"])
        return [r.packed, r.absmax]
    if op == "dequant":
        if s["f16"]:
            return [nf4.dequant(s["ws"][0], out=s["outs"][0])]
        return nf4.dequant_batch(s["ws"], s["outs"])
    outs = []
    x = s["x"]

    def layer(_, w):
        q, k, v = gemm.linear_fwd_grouped(x, w[0:3])
        o = gemm.linear_fwd(q, w[3])
        hidden = gemm.linear_swiglu(x, w[4], w[5])
        outs.extend((q, k, v, o, hidden, gemm.linear_fwd(hidden, w[6])))

    stream.run_stack(s["pinned"], s["layout"], s["dbuf"], layer, torch.cuda.current_stream())
    return outs


# --------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# --------------------------------------------------------------------------

def _weight_bytes(rows, cols, block=BLOCK, dq=True):
    n = rows * cols
    blocks = n // block
    return n // 2 + (blocks + 4 * ((blocks + GROUP - 1) // GROUP) if dq else 4 * blocks)


def work(case):
    op = case["op"]
    if op == "fwd":
        m, k, ns = case["m"], case["k"], _ints(case["ns"])
        return {"bytes": 2 * m * k + sum(_weight_bytes(n, k, case["block"], case["dq"]) + 2 * m * n
                                         for n in ns),
                "flops": 2 * m * k * sum(ns)}
    if op == "mlp":
        m, d, ff = case["m"], case["d"], case["ff"]
        return {"bytes": 3 * _weight_bytes(ff, d, BLOCK, case["dq"]) + 4 * m * d + 4 * d
                + 2 * m * d + 4 * m + 2 * m * ff + 2 * m * d,
                "flops": 6 * m * d * ff}
    if op == "dgrad":
        m, k, ns = case["m"], case["k"], _ints(case["ns"])
        return {"bytes": 2 * m * k + sum(_weight_bytes(n, k, BLOCK, case["dq"]) + 2 * m * n
                                         for n in ns),
                "flops": 2 * m * k * sum(ns)}
    if op == "wgrad":
        m, k, ns = case["m"], case["k"], _ints(case["ns"])
        return {"bytes": 2 * 2 * m * (k + sum(ns)) + 4 * k * sum(ns),
                "flops": 2 * 2 * m * k * sum(ns)}
    if op == "requant":
        n = case["rows"] * case["cols"]
        return {"bytes": n * (2 if case["bf16"] else 4)
                + _weight_bytes(case["rows"], case["cols"], BLOCK, case["dq"]), "flops": 2 * n}
    if op == "quantize":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n + (n + 1) // 2 + 4 * ((n + case["block"] - 1) // case["block"]),
                "flops": 2 * n}
    if op == "dequant":
        shapes = _shapes(case["shapes"])
        n = sum(r * c for r, c in shapes)
        return {"bytes": 2 * n + sum(_weight_bytes(r, c, BLOCK, case["dq"]) for r, c in shapes),
                "flops": n}
    m, n = case["m"], sum(r * c for r, c in LAYER_7B)
    outs = 4 * 4096 + 11008 + 4096
    return {"bytes": 2 * m * 4096 + case["layers"] * (sum(_weight_bytes(r, c) for r, c in LAYER_7B)
                                                      + 2 * m * outs),
            "flops": case["layers"] * 2 * m * n}


def tolerance(case):
    """Codes, absmax and decoded weights are defined bit for bit.  A product
    is rounded once to bf16, which alone is 1.7e-3 from the 64-bit result
    (and one more such rounding in an MLP's hidden values); weight gradients
    stay fp32 over up to 16384 tokens."""
    op = case["op"]
    if op in ("requant", "quantize", "dequant"):
        return "exact"
    if op == "wgrad":
        return {"rel": 1e-5}
    if op in ("mlp", "stream"):
        return {"rel": 1e-2}
    return {"rel": 7e-3}


def _swiglu64(x, gate, up):
    g = x @ gate.t()
    g = g * torch.sigmoid(g)
    return g.mul_(x @ up.t())


def exact(case, seed):
    op = case["op"]
    seed = seed * 1000
    if op == "fwd":
        x = _normal((case["m"], case["k"]), seed, 1.0, torch.bfloat16).double()
        return [x @ _weight64(n, case["k"], seed + 1 + i, case["block"], case["dq"]).t()
                for i, n in enumerate(_ints(case["ns"]))]
    if op == "mlp":
        d, ff = case["d"], case["ff"]
        x = _normal((case["m"], d), seed, 1.0).double()
        g = (1.0 + _normal((d,), seed + 1, 0.1)).double()
        rms = (x.square().mean(1) + 1e-6).sqrt()
        y = x / rms[:, None] * g
        gate, up = (_weight64(ff, d, seed + 2 + i, BLOCK, case["dq"]) for i in range(2))
        hidden = _swiglu64(y, gate, up)
        return [y, rms, hidden, hidden @ _weight64(d, ff, seed + 4, BLOCK, case["dq"]).t()]
    if op == "dgrad":
        dx = torch.zeros(case["m"], case["k"], dtype=torch.float64, device="cuda")
        for i, n in enumerate(_ints(case["ns"])):
            dy = _normal((case["m"], n), seed + i, 1e-3, torch.bfloat16).double()
            dx += dy @ _weight64(n, case["k"], seed + 10 + i, BLOCK, case["dq"])
        return [dx]
    if op == "wgrad":
        xs = [_normal((case["m"], case["k"]), seed + 10 * b + 9, 1.0, torch.bfloat16).double()
              for b in range(2)]
        outs = []
        for i, n in enumerate(_ints(case["ns"])):
            dys = [_normal((case["m"], n), seed + 10 * b + i, 1e-3, torch.bfloat16).double()
                   for b in range(2)]
            outs.append(dys[0].t().contiguous() @ xs[0] + dys[1].t().contiguous() @ xs[1])
        return outs
    if op == "requant":
        v = _normal((case["rows"], case["cols"]), seed + 1, SIGMA,
                    torch.bfloat16 if case["bf16"] else torch.float32)
        absmax = v.abs().view(-1, BLOCK).amax(1).double()
        if not case["dq"]:
            return [None, absmax]
        groups = (absmax.numel() + GROUP - 1) // GROUP
        padded = torch.zeros(groups * GROUP, dtype=torch.float64, device="cuda")
        padded[:absmax.numel()] = absmax
        return [None, None, padded.view(groups, GROUP).amax(1) / 127.0]
    if op == "quantize":
        v = _normal((case["rows"], case["cols"]), seed, SIGMA).abs().reshape(-1)
        blocks = (v.numel() + case["block"] - 1) // case["block"]
        padded = torch.zeros(blocks * case["block"], device="cuda")
        padded[:v.numel()] = v
        return [None, padded.view(blocks, -1).amax(1).double()]
    if op == "dequant":
        return [_product32(r, c, seed + i, BLOCK, case["dq"]).double()
                for i, (r, c) in enumerate(_shapes(case["shapes"]))]
    x = _normal((case["m"], 4096), seed, 1.0, torch.bfloat16).double()
    outs = []
    for l in range(case["layers"]):
        w = [_weight64(r, c, seed + 1 + 100 * l + i) for i, (r, c) in enumerate(LAYER_7B)]
        q, k, v = (x @ w[i].t() for i in range(3))
        hidden = _swiglu64(x, w[4], w[5])
        outs += [q, k, v, q @ w[3].t(), hidden, hidden @ w[6].t()]
    return outs
