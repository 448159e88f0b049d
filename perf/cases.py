"""The workloads whose speed this repository is judged by, with their inputs and exact results.

An engine hands this library the quantized linear layers of a decoder: one
token at a time (decode), a few tokens (batched decode, speculative
verification), whole prompts (prefill), several prompts of different lengths
at once (ragged prefill), and tensors to be expanded to f32.  Layer widths and
formats are those of the repository's benchmark and of its tests, each FFN
with the format mix its quantization recipe gives it.

A case is one pass: every product of `layers` decoder layers, in order,
through the Exec mirror (`ops.Backend`) or, for a ragged batch and a tensor
expansion, the stateless entry points.  Each layer has weights of its own, as
in a model, so that a decode streams them from HBM.  Weights and images are
laid out once in `prepare`, where an engine loads its model.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import qwen35_amd
from qwen35_amd import ops, synth

#: GGUF type id, values per block, bytes per block
FORMATS = {
    "Q4_0": (2, 32, 18), "Q4_1": (3, 32, 20), "Q8_0": (8, 32, 34), "IQ4_NL": (20, 32, 18),
    "Q2_K": (10, 256, 84), "Q3_K": (11, 256, 110), "Q4_K": (12, 256, 144), "Q5_K": (13, 256, 176),
    "Q6_K": (14, 256, 210), "IQ4_XS": (23, 256, 136),
}
#: (gate / up, down) formats of common recipes (the 3-bit grid formats are left
#: out: they are the least used, and their grids would have to be restated here)
MIXES = [("Q8_0", "Q8_0"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q5_K", "Q5_K"), ("Q6_K", "Q6_K"),
         ("Q3_K", "Q5_K"), ("Q2_K", "Q3_K"), ("IQ4_XS", "Q5_K"), ("IQ4_XS", "IQ4_XS"), ("IQ4_NL", "IQ4_NL"),
         ("Q4_0", "Q4_0"), ("Q4_1", "Q4_1")]
#: the most operations a drawn pass may have: those of the largest listed case
MOST_OPS = 2 * 3 * 9728 * 2560 * 2048


def _ffn(name, gate, down, hidden, ffn, layers, tokens):
    return {"name": name, "kind": "ffn", "gate": gate, "down": down, "hidden": hidden, "ffn": ffn, "layers": layers,
            "tokens": tokens}


def listed():
    return [
        # one token through every FFN of the smallest model: the smallest calls
        # (4-8 MB of weights each), where launches and latency count
        _ffn("decode_small_q8_0", "Q8_0", "Q8_0", 1024, 3584, 24, 1),
        # one token of a 4B model in the common 4-bit recipe
        _ffn("decode_4b_q4_k", "Q4_K", "Q6_K", 2560, 9728, 8, 1),
        # one token of a 27B model, the same recipe
        _ffn("decode_27b_q4_k", "Q4_K", "Q6_K", 5120, 17408, 3, 1),
        # one token of a 27B model squeezed to about 3.5 bits
        _ffn("decode_27b_q3_k", "Q3_K", "Q5_K", 5120, 17408, 3, 1),
        # the output head, once for every decoded token: the largest single weight
        {"name": "head_iq4_nl", "kind": "linear", "type": "IQ4_NL", "rows": 248320, "cols": 2560, "layers": 1,
         "tokens": 1},
        # eight sequences decoded together (or eight draft tokens verified)
        _ffn("batch8_27b_q4_k", "Q4_K", "Q6_K", 5120, 17408, 3, 8),
        # a short prompt of an odd length
        _ffn("prompt37_4b_q5_k", "Q5_K", "Q6_K", 2560, 9728, 4, 37),
        # a prompt chunk of 512 tokens, 27B: the common recipe, and the 4-bit
        # codebook one
        _ffn("prefill512_27b_q4_k", "Q4_K", "Q6_K", 5120, 17408, 1, 512),
        _ffn("prefill512_27b_iq4_xs", "IQ4_XS", "Q5_K", 5120, 17408, 1, 512),
        # a long prompt chunk: the largest pass
        _ffn("prefill2048_4b_q4_k", "Q4_K", "Q6_K", 2560, 9728, 1, 2048),
        # eight prompts of 16..256 tokens packed into one launch
        {"name": "ragged_q8_0", "kind": "ragged", "type": "Q8_0", "rows": 3584, "cols": 1024, "weights": 2, "nseq": 8,
         "lo": 16, "hi": 256, "lengths": 0},
        # a whole tensor expanded to f32
        {"name": "expand_q6_k", "kind": "expand", "type": "Q6_K", "rows": 5120, "cols": 17408},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "prompt", "prompt", "head", "ragged", "expand"])
    if kind == "head":
        return {"kind": "linear", "type": rng.choice(["IQ4_NL", "Q4_K", "Q6_K", "Q8_0", "Q4_0"]),
                "rows": _log(rng, 6000, 248320), "cols": 256 * _log(rng, 4, 20), "layers": 1,
                "tokens": rng.choice([1, 1, 1, rng.randint(2, 16)])}
    if kind == "ragged":
        lo = rng.randint(1, 32)
        return {"kind": "ragged", "type": rng.choice(["Q8_0", "Q4_K", "IQ4_NL"]), "rows": _log(rng, 1000, 9728),
                "cols": 256 * _log(rng, 4, 10), "weights": 2, "nseq": rng.randint(2, 16), "lo": lo,
                "hi": lo + rng.randint(16, 224), "lengths": rng.randint(0, 999)}
    if kind == "expand":
        return {"kind": "expand", "type": rng.choice(sorted(FORMATS)), "rows": _log(rng, 1000, 20000),
                "cols": 256 * _log(rng, 4, 68)}
    gate, down = rng.choice(MIXES)
    hidden = 256 * _log(rng, 4, 20)
    ffn = 256 * max(hidden // 256, round(hidden / 256 * rng.uniform(2.5, 3.8)))
    tokens = 1 if kind == "decode" else rng.randint(2, 16) if kind == "batch" else _log(rng, 17, 4096)
    layers = max(1, min(24 if tokens == 1 else 3, round(4e8 / (3 * hidden * ffn * 0.6))))
    if tokens > 64:
        layers = 1
    tokens = min(tokens, MOST_OPS // (2 * 3 * hidden * ffn * layers))
    return {"kind": "ffn", "gate": gate, "down": down, "hidden": hidden, "ffn": ffn, "layers": layers,
            "tokens": tokens}


def _products(case):
    """(format, rows, cols) of every product of one layer."""
    if case["kind"] == "ffn":
        return [(case["gate"], case["ffn"], case["hidden"])] * 2 + [(case["down"], case["hidden"], case["ffn"])]
    return [(case["type"], case["rows"], case["cols"])] * case.get("weights", 1)


def _lengths(case):
    return [int(n) for n in synth.ragged_lengths(case["nseq"], case["lo"], case["hi"], seed=case["lengths"])]


def _tokens(case):
    return sum(_lengths(case)) if case["kind"] == "ragged" else case.get("tokens", 0)


def _row_bytes(fmt, cols):
    _, be, bb = FORMATS[fmt]
    return cols // be * bb


def work(case):
    """Bytes: each weight once, each activation vector in and each result out once in f32."""
    products, layers, t = _products(case), case.get("layers", 1), _tokens(case)
    wbytes = sum(rows * _row_bytes(fmt, cols) for fmt, rows, cols in products)
    if case["kind"] == "expand":
        return {"bytes": wbytes + 4 * case["rows"] * case["cols"], "flops": 0}
    inputs = 4 * t * (case["hidden"] + case["ffn"] if case["kind"] == "ffn" else case["cols"])
    outputs = 4 * t * sum(rows for _, rows, _ in products)
    return {"bytes": layers * (wbytes + inputs + outputs),
            "flops": layers * 2 * t * sum(rows * cols for _, rows, cols in products)}


# ---- inputs ---------------------------------------------------------------------------

def _f16_bytes(x):
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _weight(fmt, rows, cols, gen):
    """Packed rows of random values with block scales of a trained weight's size (`qwen35_amd.synth`'s rules)."""
    _, be, bb = FORMATS[fmt]
    n = rows * cols // be
    w = torch.randint(0, 256, (n, bb), dtype=torch.uint8, device="cuda", generator=gen)

    def normal(scale):
        return torch.randn(n, device="cuda", generator=gen) * scale

    at = {"Q6_K": 208, "Q3_K": 108, "Q2_K": 80}.get(fmt, 0)
    w[:, at:at + 2] = _f16_bytes(normal(2e-4 if fmt == "Q8_0" else 1e-3).abs())
    if fmt in ("Q4_K", "Q5_K"):
        w[:, 2:4] = _f16_bytes(normal(1e-3).abs())
    elif fmt == "Q2_K":
        w[:, 82:84] = _f16_bytes(normal(1e-3).abs())
    elif fmt == "Q4_1":
        w[:, 2:4] = _f16_bytes(normal(8e-3))
    elif fmt == "Q6_K":
        w[:, 192:208] = torch.randint(-64, 64, (n, 16), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
    elif fmt == "Q8_0":
        w[:, 2:] = torch.randint(-127, 128, (n, 32), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
    return w.reshape(rows, cols // be * bb)


def _inputs(case, seed):
    """Per layer: the weights in load order (gate and up in one tensor, so that they are adjacent) and the activations."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)
    made = []
    for _ in range(case.get("layers", 1)):
        if case["kind"] == "ffn":
            t, hidden, ffn = case["tokens"], case["hidden"], case["ffn"]
            weights = [_weight(case["gate"], 2 * ffn, hidden, gen), _weight(case["down"], hidden, ffn, gen)]
            acts = [torch.randn((t, hidden), device="cuda", generator=gen), torch.randn((t, ffn), device="cuda", generator=gen)]
        else:
            weights = [_weight(*p, gen) for p in _products(case)]
            sizes = _lengths(case) if case["kind"] == "ragged" else [case["tokens"]] if case["kind"] == "linear" else []
            acts = [torch.randn((n, case["cols"]), device="cuda", generator=gen) for n in sizes]
        made.append((weights, acts))
    return made


def prepare(case, seed):
    qwen35_amd.check("qhip_init", qwen35_amd.load().qhip_init(0))
    layers = _inputs(case, seed)
    state = {"case": case, "layers": layers}
    if case["kind"] not in ("ffn", "linear"):
        return state
    be = ops.Backend(0)
    t = case["tokens"]
    calls = []
    for weights, acts in layers:
        def load(fmt, rows, cols, w):
            lin = be.wrap_linear(FORMATS[fmt][0], rows, cols, w)
            be.prepare_linear(lin)
            return lin

        if case["kind"] == "ffn":
            hidden, ffn = case["hidden"], case["ffn"]
            gate = load(case["gate"], ffn, hidden, weights[0][:ffn])
            up = load(case["gate"], ffn, hidden, weights[0][ffn:])
            down = load(case["down"], hidden, ffn, weights[1])
            # at one token gate and up come back side by side
            gu = torch.empty((2, t, ffn), device="cuda")
            out = torch.empty((t, hidden), device="cuda")
            calls.append((gate, up, down, acts[0], acts[1], gu, out))
        else:
            lin = load(case["type"], case["rows"], case["cols"], weights[0])
            calls.append((lin, acts[0], torch.empty((t, case["rows"]), device="cuda")))
    state.update(be=be, calls=calls)
    return state


def run(state):
    """One pass; the outputs of every product, in order."""
    case = state["case"]
    kind = case["kind"]
    if kind == "ragged":
        (weights, seqs), = state["layers"]
        tt = FORMATS[case["type"]][0]
        xq, off, total = ops.quantize_ragged(tt, seqs, case["cols"])
        return [ops.mul_mat_ragged(tt, w, xq, off, len(seqs), total, case["rows"], case["cols"]) for w in weights]
    if kind == "expand":
        (weights, _), = state["layers"]
        tt, be_, _ = FORMATS[case["type"]]
        return ops.dequantize(tt, weights[0], case["rows"] * case["cols"] // be_)
    be, t = state["be"], case["tokens"]
    outs = []
    for call in state["calls"]:
        if kind == "linear":
            lin, x, out = call
            if t == 1:
                be.matvec(out, lin, x)
            else:
                be.matvec_batch_k(out, lin, x, t)
            outs.append(out)
            continue
        gate, up, down, x, h, gu, out = call
        if t == 1:
            be.matvec_pair(gu, gate, up, x)
            be.matvec(out, down, h)
        else:
            be.matvec_batch_k(gu[0], gate, x, t)
            be.matvec_batch_k(gu[1], up, x, t)
            be.matvec_batch_k(out, down, h, t)
        outs += [gu, out]
    return outs


def tolerance(case):
    # Products: the block integers are exact, the scales and the sums f32.  The
    # present kernels are 5e-8 to 1.5e-7 (2-norm) from 64 bits over the ranges of
    # draw(), and another order of the sums is as far on its own side; about four
    # times the sum of the two.  An expansion has one or two rounded operations a
    # value: the same bits.
    return "exact" if case["kind"] == "expand" else {"rel": 1e-6}


# ---- exact results ----------------------------------------------------------------------

_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _f16(w, at):
    return w[:, at:at + 2].contiguous().view(torch.float16).double()


def _k_scales(s):
    """The eight 6-bit scales and mins of 12 packed bytes."""
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    scale = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    least = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return scale.double(), least.double()


def _expand(fmt, w):
    """f64 values [blocks, values per block] of packed blocks."""
    def nibbles(q, step):
        """Groups of `step` bytes: their low nibbles, then their high ones."""
        q = q.reshape(q.shape[0], -1, step)
        return torch.stack([q & 15, q >> 4], 2).reshape(q.shape[0], -1)

    n = w.shape[0]
    if fmt == "Q8_0":
        return _f16(w, 0) * w[:, 2:].contiguous().view(torch.int8).double()
    if fmt == "Q4_0":
        return _f16(w, 0) * (nibbles(w[:, 2:], 16).double() - 8)
    if fmt == "Q4_1":
        return _f16(w, 0) * nibbles(w[:, 4:], 16).double() + _f16(w, 2)
    codes = torch.tensor(_IQ4, dtype=torch.float64, device=w.device)
    if fmt == "IQ4_NL":
        return _f16(w, 0) * codes[nibbles(w[:, 2:], 16).long()]
    if fmt == "IQ4_XS":
        high = w[:, 2].int() | (w[:, 3].int() << 8)
        sub = [((w[:, 4 + i // 2].int() >> (4 * (i % 2))) & 15) | (((high >> (2 * i)) & 3) << 4) for i in range(8)]
        scale = torch.stack(sub, 1).double() - 32
        v = codes[nibbles(w[:, 8:], 16).long()].reshape(n, 8, 32)
        return (_f16(w, 0) * scale)[:, :, None].mul(v).reshape(n, 256)
    if fmt in ("Q4_K", "Q5_K"):
        scale, least = _k_scales(w[:, 4:16])
        q = nibbles(w[:, 48 if fmt == "Q5_K" else 16:], 32).reshape(n, 8, 32).int()
        if fmt == "Q5_K":
            q = q + 16 * torch.stack([(w[:, 16:48].int() >> i) & 1 for i in range(8)], 1)
        v = (_f16(w, 0) * scale)[:, :, None] * q.double() - (_f16(w, 2) * least)[:, :, None]
        return v.reshape(n, 256)
    if fmt == "Q6_K":
        ql, qh = w[:, :128].reshape(n, 2, 64).int(), w[:, 128:192].reshape(n, 2, 32).int()
        low = torch.cat([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)
        q = low | (torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 2) << 4)
        scale = w[:, 192:208].contiguous().view(torch.int8).double() * _f16(w, 208)
        return (scale[:, :, None] * (q.reshape(n, 16, 16).double() - 32)).reshape(n, 256)
    if fmt == "Q3_K":
        mask, qs, s = w[:, :32].int(), w[:, 32:96].reshape(n, 2, 32).int(), w[:, 96:108].int()
        low = torch.stack([(qs >> (2 * i)) & 3 for i in range(4)], 2).reshape(n, 8, 32)
        q = low - 4 * (1 - torch.stack([(mask >> i) & 1 for i in range(8)], 1))
        packed = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        top = torch.cat([(s[:, 8:12] >> (2 * i)) & 3 for i in range(4)], 1)
        scale = (packed | (top << 4)).double() - 32
        return ((_f16(w, 108) * scale)[:, :, None] * q.reshape(n, 16, 16).double()).reshape(n, 256)
    assert fmt == "Q2_K"
    s, qs = w[:, :16], w[:, 16:80].reshape(n, 2, 32).int()
    q = torch.stack([(qs >> (2 * i)) & 3 for i in range(4)], 2).reshape(n, 16, 16).double()
    scale, least = _f16(w, 80) * (s & 15).double(), _f16(w, 82) * (s >> 4).double()
    return (scale[:, :, None] * q - least[:, :, None]).reshape(n, 256)


def _activation(fmt, x):
    """x as the products see it: quantized to 8 bits per block (f32 arithmetic), then back, in f64."""
    be = 32 if FORMATS[fmt][1] == 32 else 256
    v = x.cpu().numpy().reshape(-1, be)
    most = np.abs(v).max(1, keepdims=True)
    scale = np.where(most > 0, most / np.float32(127), np.float32(1)).astype(np.float32)
    inverse = np.where(most > 0, np.float32(1) / scale, np.float32(0)).astype(np.float32)
    scaled = v * inverse
    if be == 32:
        q = np.clip(np.trunc(scaled + np.copysign(np.float32(0.5), scaled)), -128, 127)
        scale = scale.astype(np.float16)
    else:
        wide = scaled.astype(np.float64)
        q = np.clip(np.copysign(np.floor(np.abs(wide) + 0.5), wide), -127, 127)
    y = q.astype(np.float64) * scale.astype(np.float64)
    return torch.from_numpy(y.reshape(x.shape)).to(x.device)


def _product(fmt, w, x):
    """x . W^T in f64; w [rows, row bytes], x the activation as the products see it."""
    rows, cols = w.shape[0], x.shape[1]
    _, _, bb = FORMATS[fmt]
    out = torch.empty((x.shape[0], rows), dtype=torch.float64, device=x.device)
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        part = _expand(fmt, w[r:r + step].reshape(-1, bb)).reshape(-1, cols)
        out[:, r:r + step] = x @ part.t()
    return out


def exact(case, seed):
    layers = _inputs(case, seed)
    kind = case["kind"]
    if kind == "expand":
        w = layers[0][0][0]
        _, _, bb = FORMATS[case["type"]]
        step = max(1, (1 << 26) // case["cols"])
        return torch.cat([_expand(case["type"], w[r:r + step].reshape(-1, bb)).reshape(-1)
                          for r in range(0, w.shape[0], step)])
    if kind == "ragged":
        (weights, seqs), = layers
        x = _activation(case["type"], torch.cat(seqs))
        return [_product(case["type"], w, x) for w in weights]
    outs = []
    for weights, acts in layers:
        if kind == "linear":
            outs.append(_product(case["type"], weights[0], _activation(case["type"], acts[0])))
            continue
        t, ffn = case["tokens"], case["ffn"]
        gu = _product(case["gate"], weights[0], _activation(case["gate"], acts[0]))
        outs.append(torch.stack([gu[:, :ffn], gu[:, ffn:]]).reshape(2, t, ffn))
        outs.append(_product(case["down"], weights[1], _activation(case["down"], acts[1])))
    return outs
