"""The workloads this framework's speed is judged by: packed-weight matmuls as an inference program calls them.

Five kinds of call, each through the Python host layer on bf16 or fp16 activations that are already on the device:

  linear   one projection of any payload format, `load_quant_linear(dtype, blob)` and then `lin(x)`
  ffn      a dense feed-forward block: gate/up with SwiGLU, then down (`nint_ffn_decode` / `nvq_ffn_swiglu_down`)
  layer    the five projections of one decoder layer, each in a format of its own (a mixed-precision file)
  head     the LM head of a greedy decode step with its logits (`nint_matmul_argmax`)
  moe      a feed-forward block of routed mixed-bit experts and a shared one (`nint_moe_ffn_forward`)

`rows` is the number of activation rows of the call: 1 is a decode step of one sequence, up to a few dozen a batched
decode or speculative step, hundreds to 2048 a prefill chunk.  Payloads are drawn in the packed domain -- every bit
pattern of the code streams is a valid payload -- with anchors that make the weights roughly N(0, 0.02); activations are
N(0, 1) with one channel in a thousand scaled by 20, as hidden states have them.
"""
from __future__ import annotations

import math
import struct

import numpy as np
import torch

from tyloquant_amd import formats as F
from tyloquant_amd import runtime as R
from tyloquant_amd import runtime_moe as RM
from tyloquant_amd import runtime_vq as RV
from tyloquant_amd import synth

# name -> (bits, groupsize, sub_bits) of the NINT profiles files are written in
NINT = {"NINT2-16": (2, 16, 5), "NINT3-24": (3, 24, 5), "NINT4-24": (4, 24, 6), "NINT4-32": (4, 32, 6),
        "NINT5-28": (5, 28, 7), "NINT6-24": (6, 24, 7), "NINT8-48": (8, 48, 7)}
OTHER = ("NINT8-0", "NVQ3J-512", "NVQ2J", "NEPQ1-S", "MXFP4", "MXFP8")
DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}
MAX_FLOPS = 6.0e11          # no drawn case multiplies more than the largest listed one


def listed():
    return [
        # one projection of a small model at batch 1: launch latency and the host path are most of it
        dict(name="linear_nint3_row1", kind="linear", format="NINT3-24", out=4096, k=4096, rows=1, dtype="bf16"),
        # the LM head of a decode step: the largest single tensor a step reads
        dict(name="head_nint4_row1", kind="head", format="NINT4-32", out=151936, k=4096, rows=1, dtype="bf16"),
        # a dense feed-forward block at batch 1, 4-bit integers and 3-bit vectors: the body of every decode step
        dict(name="ffn_nint4_row1", kind="ffn", format="NINT4-32", hidden=4096, inter=12288, rows=1, dtype="bf16"),
        dict(name="ffn_nvq3j_row1", kind="ffn", format="NVQ3J-512", hidden=5120, inter=17408, rows=1, dtype="bf16"),
        # a mixed-format decoder layer in batched decode, and the same in prefill
        dict(name="layer_mixed_rows13", kind="layer", formats="NINT5-28,NVQ3J-512,NEPQ1-S,NINT3-24,NVQ2J",
             hidden=4096, inter=12288, rows=13, dtype="bf16"),
        dict(name="layer_mixed_rows1024", kind="layer", formats="NINT5-28,NVQ2J,NEPQ1-S,NVQ3J-512,NINT3-24",
             hidden=4096, inter=12288, rows=1024, dtype="bf16"),
        # prefill chunks of an odd length on the formats whose bytes come from other ecosystems
        dict(name="linear_mxfp4_rows601", kind="linear", format="MXFP4", out=12288, k=4096, rows=601, dtype="bf16"),
        dict(name="linear_nint8_0_rows333", kind="linear", format="NINT8-0", out=4096, k=12288, rows=333, dtype="fp16"),
        # a full prefill chunk through a dense feed-forward block: the most arithmetic
        dict(name="ffn_nint4_rows2048", kind="ffn", format="NINT4-32", hidden=4096, inter=12288, rows=2048, dtype="bf16"),
        # routed experts: one token, a batched decode step that hits every expert, a prefill chunk
        dict(name="moe_row1", kind="moe", experts=64, top_k=8, hidden=4096, inter=2048, rows=1, dtype="bf16"),
        dict(name="moe_rows61", kind="moe", experts=64, top_k=8, hidden=4096, inter=2048, rows=61, dtype="bf16"),
        dict(name="moe_rows2048", kind="moe", experts=128, top_k=8, hidden=2048, inter=1024, rows=2048, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("linear",) * 5 + ("ffn",) * 2 + ("layer", "head", "moe", "moe"))
        c = dict(kind=kind, rows=_log_int(rng, 1, 2048), dtype=rng.choice(("bf16", "bf16", "fp16")))
        if kind == "linear":
            c.update(format=rng.choice(tuple(NINT) + OTHER), out=_log_int(rng, 1024, 17408),
                     k=128 * _log_int(rng, 8, 136))
        elif kind == "ffn":
            c.update(format=rng.choice(("NINT4-32", "NINT3-24", "NINT5-28", "NVQ3J-512")),
                     hidden=128 * rng.randint(16, 40), inter=128 * rng.randint(32, 136))
        elif kind == "layer":
            c.update(formats=",".join(rng.choice(("NINT3-24", "NINT4-24", "NINT5-28") + OTHER) for _ in range(5)),
                     hidden=128 * rng.randint(16, 32), inter=128 * rng.randint(32, 96))
        elif kind == "head":
            c.update(format=rng.choice(("NINT4-32", "NINT5-28", "NINT6-24")), out=rng.randint(32000, 151936),
                     k=128 * rng.randint(16, 32), rows=_log_int(rng, 1, 16))
        else:
            hidden, inter, experts = rng.choice(((4096, 2048, 64), (2048, 1024, 128), (2048, 768, 128), (2880, 1440, 32)))
            c.update(experts=experts, top_k=rng.choice((2, 4, 8)), hidden=hidden, inter=inter)
        if work(c)["flops"] <= MAX_FLOPS:
            return c


# ---- payloads ------------------------------------------------------------------------------------------------------
def _nint_blob(rng, profile, out, k):
    """A NINT payload with uniform codes and sub-scales; the anchors centre the weights and give them sigma 0.02."""
    bits, gs, sub = profile
    ng = -(-k // gs)
    levels, centre = (1 << sub) - 1, ((1 << bits) - 1) / 2
    spread = lambda n: ((n + 1) ** 2 - 1) / 12
    var = (spread(levels) + (levels / 2) ** 2) * (spread(2 * centre) + centre ** 2) - (levels / 2 * centre) ** 2
    ns = (rng.uniform(0.7, 1.3, out) * 0.02 / math.sqrt(var + centre ** 2 * spread(levels))).astype(np.float16)
    nm = (ns.astype(np.float32) * centre).astype(np.float16)
    nbytes = 2 * ((out * ng * sub + 7) // 8) + (out * ng * gs * bits + 7) // 8
    streams = rng.integers(0, 1 << 64, (nbytes + 7) // 8, dtype=np.uint64).view(np.uint8)[:nbytes]
    head = struct.pack("<BBiii", bits, sub, gs, 0, k) + struct.pack("<I2qII", 2, out, k, out, ng)
    return b"".join((head, ns.tobytes(), nm.tobytes(), streams.tobytes()))


def _blob(seed, fmt, out, k):
    """(dtype, blob) of an [out, k] tensor."""
    if fmt in NINT:
        return fmt.split("-")[0], _nint_blob(np.random.default_rng(seed), NINT[fmt], out, k)
    if fmt == "NINT8-0":
        return synth.nint8_zero_blob(seed, out, k)
    if fmt == "NVQ3J-512":
        return synth.nvq3j512_blob(seed, out, k)
    if fmt == "NVQ2J":
        return synth.nvq2j_blob(seed, out, k)
    if fmt == "NEPQ1-S":
        return synth.nepq1_blob(seed, fmt, out, k)
    return synth.mx_blob(seed, fmt, out, k)


def _expert_bits(experts):
    """Bit widths of a mixed-bit expert tensor: a tenth at 2, four tenths each at 3 and 4, a tenth at 5."""
    return np.random.default_rng(4).choice([2, 3, 4, 5], size=experts, p=[0.1, 0.4, 0.4, 0.1])


def _moe_weight(seed, experts, out, k):
    rng, bits, pools = np.random.default_rng(seed), _expert_bits(experts), []
    for b in (2, 3, 4, 5):
        ids = np.flatnonzero(bits == b).astype(np.int32)
        if len(ids):
            pools.append((ids, f"NINT{b}", _nint_blob(rng, synth.MOE_PROFILES[b], len(ids) * out, k)))
    return RM.NintMoeWeight.from_blob(F.nintm_blob(experts, out, k, pools))


def _linear(seed, fmt, out, k):
    return R.load_quant_linear(*_blob(seed, fmt, out, k))


def _activations(seed, rows, k, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn(rows, k, generator=g, device="cuda")
    x[:, torch.randperm(k, generator=g, device="cuda")[:max(1, k // 1000)]] *= 20.0
    return x.to(DTYPE[dtype])


def _layer(c):
    """(format, out, k) of the projections of a decoder layer: fused q/k/v, attention output, gate, up, down."""
    h, i = c["hidden"], c["inter"]
    return list(zip(c["formats"].split(","), (h + h // 2, h, i, i, h), (h, h, h, h, i)))


# ---- the calls -------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    c, s, rows, dt = case, 1000 * seed, case["rows"], case["dtype"]
    if c["kind"] == "linear":
        return dict(kind="linear", lin=_linear(s, c["format"], c["out"], c["k"]), x=_activations(s + 9, rows, c["k"], dt))
    if c["kind"] == "head":
        return dict(kind="head", w=_linear(s, c["format"], c["out"], c["k"]).weight, x=_activations(s + 9, rows, c["k"], dt))
    if c["kind"] == "ffn":
        h, i = c["hidden"], c["inter"]
        x = _activations(s + 9, rows, h, dt)
        if c["format"] in NINT:
            return dict(kind="ffn", gate_up=_linear(s, c["format"], 2 * i, h).weight, down=_linear(s + 1, c["format"], h, i).weight, x=x)
        gate, up, down = (_linear(s + j, c["format"], *shape).weight for j, shape in enumerate(((i, h), (i, h), (h, i))))
        return dict(kind="nvq_ffn", gate=gate, up=up, down=down, x=x)
    if c["kind"] == "layer":
        return dict(kind="layer", lins=[_linear(s + j, *p) for j, p in enumerate(_layer(c))],
                    x=_activations(s + 9, rows, c["hidden"], dt), hidden=_activations(s + 8, rows, c["inter"], dt))
    e, h, i = c["experts"], c["hidden"], c["inter"]
    g = torch.Generator(device="cuda")
    g.manual_seed(s + 7)
    return dict(kind="moe", gate_up=_moe_weight(s, e, 2 * i, h), down=_moe_weight(s + 1, e, h, i), top_k=c["top_k"],
                shared=(_linear(s + 2, "NINT4-24", 2 * i, h).weight, _linear(s + 3, "NINT4-24", h, i).weight),
                x=_activations(s + 9, rows, h, dt), logits=torch.randn(rows, e, generator=g, device="cuda"))


def run(state):
    s = state
    if s["kind"] == "linear":
        return s["lin"](s["x"])
    if s["kind"] == "head":
        return R.nint_matmul_argmax(s["w"], s["x"], return_logits=True)
    if s["kind"] == "ffn":
        return R.nint_ffn_decode(s["gate_up"], s["down"], s["x"])
    if s["kind"] == "nvq_ffn":
        return RV.nvq_ffn_swiglu_down(s["gate"], s["up"], s["down"], s["x"])
    if s["kind"] == "layer":
        return [lin(x) for lin, x in zip(s["lins"], (s["x"],) * 4 + (s["hidden"],))]
    return RM.nint_moe_ffn_forward(s["gate_up"], s["down"], s["x"], s["logits"], s["top_k"], normalize=True, shared=s["shared"])


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _payload(fmt, out, k):
    """Bytes of a tensor in its file (without headers and tables of a few KB)."""
    groups = -(-k // 24)
    if fmt in NINT:
        bits, gs, sub = NINT[fmt]
        return out * (4 + -(-k // gs) * (2 * sub + gs * bits) / 8)
    return out * {"NINT8-0": k * 34 / 32, "NVQ3J-512": 2 + groups / 2 + k / 4 * 9 / 8 + k / 8 * 7 / 8,
                  "NVQ2J": 2 + groups / 2 + k / 8 + k / 8 * 7 / 8,
                  "NEPQ1-S": 2 + groups * 5 / 8 + k / 8 * 9 / 8 + -(-groups // 4),
                  "MXFP4": k / 2 + k / 32, "MXFP8": k + k / 128 / 128}[fmt]


def work(case):
    c, m = case, case["rows"]
    mm = lambda fmt, out, k: (_payload(fmt, out, k), 2.0 * m * out * k)
    if c["kind"] in ("linear", "head"):
        b, f = mm(c["format"], c["out"], c["k"])
        return {"bytes": b + m * (2 * c["k"] + 4 * c["out"]), "flops": f}
    if c["kind"] == "layer":
        parts = [mm(*p) for p in _layer(c)]
        return {"bytes": sum(b for b, _ in parts) + m * (2 * c["hidden"] + 2 * c["inter"] + 4 * sum(o for _, o, _ in _layer(c))),
                "flops": sum(f for _, f in parts)}
    h, i = c["hidden"], c["inter"]
    if c["kind"] == "ffn":
        (b0, f0), (b1, f1) = mm(c["format"], 2 * i, h), mm(c["format"], h, i)
        return {"bytes": b0 + b1 + m * 6 * h, "flops": f0 + f1}
    # the experts a batch hits on average, at the mean size of an expert, and the shared one
    e, k = c["experts"], c["top_k"]
    name = {2: "NINT2-16", 3: "NINT3-24", 4: "NINT4-24", 5: "NINT5-28"}
    each = sum(_payload(name[int(b)], 2 * i, h) + _payload(name[int(b)], h, i) for b in _expert_bits(e)) / e
    hit = e * (1.0 - (1.0 - k / e) ** m)
    shared = _payload("NINT4-24", 2 * i, h) + _payload("NINT4-24", h, i)
    return {"bytes": hit * each + shared + m * (6 * h + 4 * e), "flops": 2.0 * m * (k + 1) * 3 * h * i}


# Largest relative difference (2-norm) another correct implementation would show: about four times what the paths differ
# from the same sums over the dequantized weights in 64 bits.  The weights of EXACT are products of small integers and
# powers of two that fp16 or bf16 hold exactly, so only 32-bit sums differ (up to 6e-6 seen); those of ROUNDED are rounded
# once to fp16 where they meet the matrix cores (2.4e-4 seen), NVQ2J and NINT8-0 only in batches; a feed-forward block
# rounds its hidden row to fp16 (2.1e-4 seen) on top of that (4.7e-4 seen).
EXACT = ("NINT2-16", "NINT3-24", "NINT4-24", "NINT4-32", "NEPQ1-S", "MXFP4", "MXFP8")
IN_BATCHES = ("NVQ2J", "NINT8-0")


def tolerance(case):
    if case["kind"] in ("layer", "moe"):
        return {"rel": 1e-3}
    exact = case["format"] in EXACT or (case["format"] in IN_BATCHES and case["rows"] <= 32)
    if case["kind"] == "ffn":
        return {"rel": 1e-3 if exact else 2e-3}
    return {"rel": 2.5e-5 if exact else 1e-3}
