"""The work a program does through xn_amd, as measurable cases.

A case is one call (or, for the decode step, one replay) of the package's
public entry points on device-resident GGUF weights:

  linear    QLinear.forward: (m, k) f32 rows through one n x k weight
  group     matmul_t_group: q, k and v projections of one activation
  mlp       mlp_t: the SwiGLU block (gate, up, down)
  step      DecodeStep.replay: every projection of a captured decode step
  quantize  QTensor.quantize_f32 + dequantize: making a quantized weight from
            f32 and reading it back

`listed` holds the ordinary ones, `draw` others of the same ranges.  Weights
are GGUF blocks of every device dtype made from random integer fields with
the spread that quantized N(0, 0.02) weights have; activations are normal
rows whose channels differ in scale, as normalised hidden states do.
"""
import math

import torch

from xn_amd.decode import DecoderWeights, DecodeStep, LayerWeights
from xn_amd.quantized import GgmlDType, QLinear, QTensor, matmul_t_group, mlp_t

DEV = "cuda"

# elements and bytes of one GGUF block
BLOCK = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q5_0": (32, 22), "Q5_1": (32, 24), "Q8_0": (32, 34),
         "Q2K": (256, 84), "Q3K": (256, 110), "Q4K": (256, 144), "Q5K": (256, 176), "Q6K": (256, 210)}
K_TYPES = ("Q2K", "Q3K", "Q4K", "Q5K", "Q6K")


def listed():
    return [
        # one token through one GPU's share of a feed-forward split 8 ways: the smallest call
        {"name": "linear_q4k_m1_4096x1792", "op": "linear", "dtype": "Q4K", "m": 1, "k": 4096, "n": 1792},
        # one token through a square Q8_0 projection
        {"name": "linear_q8_0_m1_4096x4096", "op": "linear", "dtype": "Q8_0", "m": 1, "k": 4096, "n": 4096},
        # one token through the gate projection of an 8B model, the benchmark's headline
        {"name": "linear_q4k_m1_4096x14336", "op": "linear", "dtype": "Q4K", "m": 1, "k": 4096, "n": 14336},
        # one token through a whole Q4_0 feed-forward block
        {"name": "mlp_q4_0_m1", "op": "mlp", "dtype": "Q4_0", "down": "Q4_0", "m": 1, "k": 4096, "f": 14336, "n": 4096},
        # the q, k and v projections for four sequences
        {"name": "group_qkv_q4k_m4", "op": "group", "dtype": "Q4K", "m": 4, "k": 4096, "n": 4096, "kv": 1024},
        # the feed-forward block of a Q4_K_M model for sixteen sequences
        {"name": "mlp_q4k_q6k_m16", "op": "mlp", "dtype": "Q4K", "down": "Q6K", "m": 16, "k": 4096, "f": 14336, "n": 4096},
        # a Q5_K projection at a ragged batch (a short prompt)
        {"name": "linear_q5k_m37_4096x6144", "op": "linear", "dtype": "Q5K", "m": 37, "k": 4096, "n": 6144},
        # the reference's own benchmark shape: 125 frames through a Q8_0 layer
        {"name": "linear_q8_0_m125_4096x1024", "op": "linear", "dtype": "Q8_0", "m": 125, "k": 4096, "n": 1024},
        # a 512-token prompt through a Q4_0 gate projection
        {"name": "linear_q4_0_m512_4096x14336", "op": "linear", "dtype": "Q4_0", "m": 512, "k": 4096, "n": 14336},
        # a 512-token prompt through a Q4_K gate projection, the benchmark's prefill
        {"name": "linear_q4k_m512_4096x14336", "op": "linear", "dtype": "Q4K", "m": 512, "k": 4096, "n": 14336},
        # a 2048-token prompt through a Q6_K projection: the largest product
        {"name": "linear_q6k_m2048_4096x14336", "op": "linear", "dtype": "Q6K", "m": 2048, "k": 4096, "n": 14336},
        # all projections of one token's decode step, eight layers and the head, as one graph
        {"name": "step_q4k_q6k_b1", "op": "step", "m": 1, "layers": 8, "hidden": 4096, "kv": 1024, "f": 14336,
         "vocab": 128256},
    ]


# The largest product and weight that a drawn case holds; the types with a
# scale per 32 elements and the rarer K types are served at prompts of a few
# hundred rows.
MAX_MNK = {"Q4K": 2048 * 4096 * 14336, "Q6K": 2048 * 4096 * 14336}
MAX_MNK_OTHER = 512 * 4096 * 14336
MAX_NK = 4096 * 28672


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(["linear", "group", "mlp", "quantize"], [11, 3, 4, 2])[0]
    if op == "quantize":
        dt = rng.choice(["Q4_0", "Q8_0", "Q4K", "Q6K"])
        return {"op": op, "dtype": dt, "k": 256 * _log_int(rng, 2, 32), "n": _log_int(rng, 256, 6000)}
    dt = rng.choices(["Q4K", "Q6K", "Q8_0", "Q4_0", "Q5K", "Q4_1", "Q5_0", "Q5_1", "Q2K", "Q3K"],
                     [6, 4, 4, 4, 2, 1, 1, 1, 1, 1])[0]
    step = 256 if dt in K_TYPES else 64
    k = step * _log_int(rng, 1024 // step, 14336 // step)
    limit = MAX_MNK.get(dt, MAX_MNK_OTHER)
    m = _log_int(rng, 1, 2048)
    if op == "linear":
        n = _log_int(rng, 512, min(28672, MAX_NK // k))
        return {"op": op, "dtype": dt, "m": max(1, min(m, limit // (n * k))), "k": k, "n": n}
    if op == "group":
        n = 128 * rng.randint(8, 48)
        return {"op": op, "dtype": dt, "m": max(1, min(m, limit // (2 * n * k))), "k": k, "n": n,
                "kv": 128 * rng.randint(2, 8)}
    k = min(k, 8192)
    f = 256 * rng.randint(8, 56)
    down = "Q6K" if dt == "Q4K" and rng.random() < 0.7 else dt
    return {"op": op, "dtype": dt, "down": down, "m": max(1, min(m, limit // (3 * f * k))), "k": k, "f": f, "n": k}


# ---------------------------------------------------------------------------
# Weights: integer fields of every block of an n x k weight, the GGUF bytes
# they pack into, and the value they stand for.

def _rng(seed, part=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 10007 + part)
    return g


def _normal_levels(g, shape, lo, hi, mid, sd):
    """Whole numbers lo..hi, normal around mid."""
    v = torch.empty(shape, dtype=torch.float32, device=DEV).normal_(mid, sd, generator=g)
    return v.round_().clamp_(lo, hi).to(torch.uint8 if lo >= 0 else torch.int8)


def _scale(g, nb, unit):
    """An f16 scale for each block, around `unit`."""
    v = torch.empty(nb, dtype=torch.float32, device=DEV).normal_(0.0, 0.15, generator=g)
    return (torch.exp(v) * unit).half()


def _uniform(g, shape, lo, hi):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int16)


class Fields:
    """q: levels as they multiply (nb, elements); sc, mn: sub-block scales and
    mins (nb, subs) or None; d, dmin: f16 of each block or None; add: the f16
    constant of Q4_1 / Q5_1 or None."""

    def __init__(self, q, d, sc=None, mn=None, dmin=None, add=None):
        self.q, self.d, self.sc, self.mn, self.dmin, self.add = q, d, sc, mn, dmin, add

    def values(self, n, k):
        """The weight in 64 bits (without `add`)."""
        w = self.q.double()
        if self.sc is not None:
            nb, subs = self.sc.shape
            w = w.view(nb, subs, -1) * self.sc.double()[:, :, None]
            w = w * self.d.double()[:, None, None]
            if self.mn is not None:
                w = w - (self.dmin.double()[:, None] * self.mn.double())[:, :, None]
        else:
            w = w * self.d.double()[:, None]
        return w.reshape(n, k)


def _f16_bytes(h):
    return h.view(torch.uint8).view(-1, 2)


def _nibbles(q):
    """32 levels -> 16 bytes: byte i holds elements i and i + 16."""
    return q[:, :16] | (q[:, 16:] << 4)


def _pairs32(q):
    """256 levels 0..15 -> 128 bytes: byte 32p + l holds elements 64p + l and 64p + 32 + l."""
    q = q.view(-1, 4, 2, 32)
    return (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)


def _scales_k4(sc, mn):
    """Eight 6-bit scales and mins -> 12 bytes."""
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    a = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    b = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    c = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return torch.cat([a, b, c], 1)


def _high_bits32(q):
    """Bit 4 of 32 levels -> 4 bytes, element e at bit e."""
    b = ((q >> 4) & 1).view(-1, 4, 8).int()
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], device=DEV, dtype=torch.int32)
    return (b * w).sum(2).to(torch.uint8)


def _make_fields(dtype, n, k, g):
    """(GGUF bytes (nb, block bytes) uint8, Fields) of a random weight."""
    be, _ = BLOCK[dtype]
    nb = n * k // be
    if dtype == "Q8_0":
        q, d = _normal_levels(g, (nb, 32), -127, 127, 0, 55), _scale(g, nb, 0.02 / 55)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], 1), Fields(q, d)
    if dtype == "Q4_0":
        q, d = _normal_levels(g, (nb, 32), 0, 15, 8, 3.5), _scale(g, nb, 0.02 / 3.5)
        return torch.cat([_f16_bytes(d), _nibbles(q)], 1), Fields(q.to(torch.int8) - 8, d)
    if dtype == "Q5_0":
        q, d = _normal_levels(g, (nb, 32), 0, 31, 16, 7), _scale(g, nb, 0.02 / 7)
        return (torch.cat([_f16_bytes(d), _high_bits32(q), _nibbles(q & 15)], 1), Fields(q.to(torch.int8) - 16, d))
    if dtype in ("Q4_1", "Q5_1"):
        top = 15 if dtype == "Q4_1" else 31
        q, d = _normal_levels(g, (nb, 32), 0, top, top / 2, top / 4), _scale(g, nb, 0.08 / top)
        add = (-d.float() * (top / 2)).half()
        parts = [_f16_bytes(d), _f16_bytes(add)] + ([_high_bits32(q)] if top == 31 else []) + [_nibbles(q & 15)]
        return torch.cat(parts, 1), Fields(q, d, add=add)
    if dtype in ("Q4K", "Q5K"):
        top = 15 if dtype == "Q4K" else 31
        q = _normal_levels(g, (nb, 256), 0, top, top / 2, top / 4)
        sc, mn = _uniform(g, (nb, 8), 24, 64), _uniform(g, (nb, 8), 24, 64)
        d, dmin = _scale(g, nb, 0.08 / top / 44), _scale(g, nb, 0.04 / 44)
        head = [_f16_bytes(d), _f16_bytes(dmin), _scales_k4(sc, mn)]
        if top == 31:  # byte l: bit 2p of element 64p + l, bit 2p + 1 of element 64p + 32 + l
            b = ((q >> 4) & 1).view(-1, 8, 32).int()
            w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], device=DEV, dtype=torch.int32)
            head.append((b * w[None, :, None]).sum(1).to(torch.uint8))
        return torch.cat(head + [_pairs32(q & 15)], 1), Fields(q, d, sc, mn, dmin)
    if dtype == "Q6K":
        q = _normal_levels(g, (nb, 256), 0, 63, 32, 14)
        sc = _uniform(g, (nb, 16), 60, 128) * (1 - 2 * _uniform(g, (nb, 16), 0, 2))
        d = _scale(g, nb, 0.02 / 14 / 94)
        e = q.view(-1, 2, 4, 32)  # element 128h + 32i + l
        low = torch.stack([(e[:, :, 0] & 15) | ((e[:, :, 2] & 15) << 4), (e[:, :, 1] & 15) | ((e[:, :, 3] & 15) << 4)], 2)
        high = (e[:, :, 0] >> 4) | ((e[:, :, 1] >> 4) << 2) | ((e[:, :, 2] >> 4) << 4) | ((e[:, :, 3] >> 4) << 6)
        return (torch.cat([low.reshape(-1, 128), high.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], 1),
                Fields(q.to(torch.int8) - 32, d, sc))
    # element 128h + 32i + l: two bits at byte 32h + l, bits 2i
    q = _normal_levels(g, (nb, 256), 0, 3 if dtype == "Q2K" else 7, 1.5 if dtype == "Q2K" else 4, 0.9 if dtype == "Q2K" else 1.7)
    e = (q & 3).view(-1, 2, 4, 32)
    low = (e[:, :, 0] | (e[:, :, 1] << 2) | (e[:, :, 2] << 4) | (e[:, :, 3] << 6)).reshape(-1, 64)
    if dtype == "Q2K":
        sc, mn = _uniform(g, (nb, 16), 5, 16), _uniform(g, (nb, 16), 5, 16)
        d, dmin = _scale(g, nb, 0.02 / 10), _scale(g, nb, 0.03 / 10)
        both = (sc | (mn << 4)).to(torch.uint8)
        return torch.cat([both, low, _f16_bytes(d), _f16_bytes(dmin)], 1), Fields(q, d, sc, mn, dmin)
    # Q3K: bit 2 of element 32j + l at byte l, bit j; 16 six-bit scales
    b = (q >> 2).view(-1, 8, 32).int()
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], device=DEV, dtype=torch.int32)
    high = (b * w[None, :, None]).sum(1).to(torch.uint8)
    sc = _uniform(g, (nb, 16), 0, 64)
    s = sc.to(torch.uint8)
    first = (s[:, :8] & 15) | ((s[:, 8:] & 15) << 4)
    t = s >> 4
    last = t[:, 0:4] | (t[:, 4:8] << 2) | (t[:, 8:12] << 4) | (t[:, 12:16] << 6)
    d = _scale(g, nb, 0.02 / 1.7 / 18)
    return (torch.cat([high, low, first, last, _f16_bytes(d)], 1), Fields(q.to(torch.int8) - 4, d, sc - 32))


def _qtensor(dtype, n, k, seed, part):
    blocks, _ = _make_fields(dtype, n, k, _rng(seed, part))
    return QTensor.from_gguf_bytes(blocks.reshape(-1).cpu().numpy(), (n, k), GgmlDType[dtype], DEV)


def _rows(m, k, seed, part=999):
    g = _rng(seed, part)
    spread = torch.exp(0.4 * torch.randn(k, generator=g, device=DEV))
    return torch.randn((m, k), generator=g, device=DEV) * spread


# ---------------------------------------------------------------------------
# The measured calls.

def _layer_shapes(case):
    d, kv, f = case["hidden"], case["kv"], case["f"]
    return [("Q4K", d, d), ("Q4K", kv, d), ("Q4K", kv, d), ("Q4K", d, d), ("Q4K", f, d), ("Q4K", f, d), ("Q6K", d, f)]


def _weights(case):
    """(dtype, rows, columns) of each weight of a case, in order."""
    op = case["op"]
    if op == "linear":
        return [(case["dtype"], case["n"], case["k"])]
    if op == "group":
        return [(case["dtype"], r, case["k"]) for r in (case["n"], case["kv"], case["kv"])]
    if op == "mlp":
        dt, k, f = case["dtype"], case["k"], case["f"]
        return [(dt, f, k), (dt, f, k), (case["down"], case["n"], f)]
    return _layer_shapes(case) * case["layers"] + [("Q6K", case["vocab"], case["hidden"])]


def _rest_of_model(point, layer, bufs):
    """Attention, norms and residuals are outside the quantized path: what
    they would write (attn, x_next) stands in the step's buffers."""


def prepare(case, seed):
    op = case["op"]
    if op == "quantize":
        w = torch.empty((case["n"], case["k"]), dtype=torch.float32, device=DEV).normal_(0.0, 0.02, generator=_rng(seed))
        return {"op": op, "w": w, "dtype": GgmlDType[case["dtype"]]}
    qts = [_qtensor(dt, n, k, seed, i) for i, (dt, n, k) in enumerate(_weights(case))]
    m = case["m"]
    x = _rows(m, qts[0].shape()[1], seed)
    if op == "linear":
        return {"op": op, "layer": QLinear(qts[0]), "x": x}
    if op == "group":
        outs = [torch.empty((m, q.shape()[0]), device=DEV) for q in qts]
        return {"op": op, "qts": qts, "x": x, "m": m, "k": case["k"], "outs": outs}
    if op == "mlp":
        return {"op": op, "qts": qts, "x": x, "m": m, "h": torch.empty((m, case["f"]), device=DEV),
                "y": torch.empty((m, case["n"]), device=DEV)}
    layers = [LayerWeights(*qts[7 * i:7 * i + 7]) for i in range(case["layers"])]
    step = DecodeStep(DecoderWeights(layers, qts[-1]), m, torch.device(DEV, torch.cuda.current_device()), _rest_of_model)
    step.x.copy_(x)
    for i, b in enumerate(step.bufs):
        b["attn"].copy_(_rows(m, case["hidden"], seed, 1000 + 2 * i))
        b["x_next"].copy_(_rows(m, case["hidden"], seed, 1001 + 2 * i))
    step.capture()
    return {"op": op, "step": step}


def _step_outputs(step):
    return [step.logits] + [b[name] for b in step.bufs for name in ("q", "k", "v", "o", "h", "down")]


def run(state):
    op = state["op"]
    if op == "linear":
        return state["layer"].forward(state["x"])
    if op == "group":
        matmul_t_group(state["qts"], state["m"], state["k"], state["x"], state["outs"])
        return state["outs"]
    if op == "mlp":
        gate, up, down = state["qts"]
        mlp_t(gate, up, down, state["m"], state["x"], state["h"], state["y"])
        return [state["h"], state["y"]]
    if op == "step":
        state["step"].replay(torch.cuda.current_stream())
        return _step_outputs(state["step"])
    return QTensor.quantize_f32(state["w"], dtype=state["dtype"]).dequantize()


def work(case):
    if case["op"] == "quantize":
        be, bb = BLOCK[case["dtype"]]
        count = case["n"] * case["k"]
        return {"bytes": 2 * (4 * count) + 2 * (count // be * bb), "flops": 2 * count}
    m, nbytes, flops = case["m"], 0, 0
    for dt, n, k in _weights(case):
        be, bb = BLOCK[dt]
        nbytes += n * k // be * bb
        flops += 2 * m * n * k
    if case["op"] == "linear":
        nbytes += 4 * m * (case["k"] + case["n"])
    elif case["op"] == "group":
        nbytes += 4 * m * (case["k"] + case["n"] + 2 * case["kv"])
    elif case["op"] == "mlp":
        nbytes += 4 * m * (case["k"] + case["f"] + case["n"])
    else:
        d = case["hidden"]
        nbytes += 4 * m * (d + case["layers"] * (3 * d + 2 * case["kv"] + case["f"]) + case["vocab"])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    op = case["op"]
    if op == "quantize":  # whole levels and f16 scales: the same bytes as the CPU quantizer's
        return "exact"
    # an f32 rounding of o or h moves some of the 8-bit levels they are quantized to
    if op == "step":  # measured 3.8e-3, 1.4e-2
        return {"rel": 1.5e-2, "max": 6e-2}
    if op == "mlp":  # measured 4.6e-4, 6.1e-3
        return {"rel": 2e-3, "max": 2.5e-2}
    if case["dtype"] == "Q4K":  # 16-bit halves of the min term (measured 4.8e-6, 1.9e-5)
        return {"rel": 2e-5, "max": 8e-5}
    return {"rel": 5e-7, "max": 2.5e-6}  # 32-bit sums (measured 1.1e-7, 6.2e-7)


# ---------------------------------------------------------------------------
# The same products in 64 bits.  The activation is quantized as the format
# says (Q8_K or Q8_0 blocks: whole levels and one scale), which is part of
# what the product is; everything after that is plain 64-bit arithmetic.

def _round_away(t):
    return torch.sign(t) * torch.floor(t.abs() + 0.5)


def _quantized_rows(dtype, x):
    """f32 rows -> (d * levels, block sums as Q8_1 keeps them), 64 bits."""
    m, k = x.shape
    x = x.float()
    if dtype in K_TYPES:
        b = x.view(m, -1, 256)
        at = b.abs().argmax(2, keepdim=True)
        top = torch.gather(b, 2, at).double()
        iscale = torch.where(top != 0, -128.0 / top, torch.zeros_like(top)).float()
        q = _round_away((iscale * b).double()).clamp(max=127.0)
        d = torch.where(iscale != 0, 1.0 / iscale.double(), torch.zeros_like(top)).float().double()
        return (q * d).view(m, k), None
    b = x.view(m, -1, 32)
    d = (b.abs().amax(2, keepdim=True).double() / 127.0).float()
    inv = torch.where(d != 0, 1.0 / d.double(), torch.zeros_like(d, dtype=torch.float64)).float()
    q = _round_away((b * inv).double())
    d16 = d.half()
    s = (q.sum(2, keepdim=True).float().half().float() * d16.float()).half()
    return (q * d16.double()).view(m, k), s.double()[:, :, 0]


def _product(dtype, n, k, seed, part, x):
    _, f = _make_fields(dtype, n, k, _rng(seed, part))
    a, s = _quantized_rows(dtype, x)
    y = a @ f.values(n, k).t()
    if f.add is not None:
        y += s @ f.add.double().view(n, -1).t()
    return y


def _mlp64(shapes, seed, part, x):
    g = _product(*shapes[0], seed, part, x)
    u = _product(*shapes[1], seed, part + 1, x)
    h = g / (1.0 + torch.exp(-g)) * u
    return h, _product(*shapes[2], seed, part + 2, h)


def exact(case, seed):
    op = case["op"]
    if op == "quantize":  # defined by its f32 search, not by a 64-bit value
        return None
    ws = _weights(case)
    x = _rows(case["m"], ws[0][2], seed)
    if op == "linear":
        return _product(*ws[0], seed, 0, x)
    if op == "group":
        return [_product(*w, seed, i, x) for i, w in enumerate(ws)]
    if op == "mlp":
        return list(_mlp64(ws, seed, 0, x))
    outs = []
    for i in range(case["layers"]):
        p = 7 * i
        qkv = [_product(*ws[p + j], seed, p + j, x) for j in range(3)]
        o = _product(*ws[p + 3], seed, p + 3, _rows(case["m"], case["hidden"], seed, 1000 + 2 * i))
        outs += qkv + [o, *_mlp64(ws[p + 4:p + 7], seed, p + 4, o)]
        x = _rows(case["m"], case["hidden"], seed, 1001 + 2 * i)
    return [_product(*ws[-1], seed, len(ws) - 1, x)] + outs
