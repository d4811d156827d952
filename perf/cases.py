"""The work a program has this library do, as cases that can be timed: linears, gated projections, a decoder layer's
linears as a chain, and expert FFNs, from one token to a long prompt.

A case is a dict of plain values:
  kind "linear"  `layers` independent W4A16 linears [n][k] at t rows through W4a16Dec.lin_forward, the path chosen by the
                 library (out_f16: f16 or f32 results); glu: lin_forward_glu, the fused gate|up projection with SiLU * up
  kind "chain"   `layers` decoder layers (QKV, O, gate|up, down) through chain_forward / chain_forward_fused
  kind "moe"     `layers` expert FFNs: moe_route on the layer's router logits, then moe_ffn
`group` and `bf16` are the scale group and the scale type.  A pass runs as many layers as a step of a model would have
in a row, each with weights of its own, so that decode steps find their weights in HBM and not in a cache.
"""
import math
import weakref

import numpy as np
import torch

from llm170_amd import gen, ops

# Layer shapes of the repository's benchmark and tests (n, k): the 27B dense layer (QKV, O, gate|up, down) and an 8B-like one
DENSE = [(7168, 5120), (5120, 5120), (34816, 5120), (5120, 17408), (6144, 4096), (4096, 4096), (22016, 4096), (4096, 11008)]


def listed():
    return [
        # one token through the smallest linear of the benchmark: latency and launches, a decode step of one sequence
        {"name": "linear_t1_4096", "kind": "linear", "n": 4096, "k": 4096, "group": 128, "bf16": False, "t": 1, "layers": 16,
         "glu": False, "out_f16": True},
        # one token through the widest projection of the 27B layer: the weight stream of a decode step
        {"name": "glu_t1_27b", "kind": "linear", "n": 34816, "k": 5120, "group": 128, "bf16": False, "t": 1, "layers": 2,
         "glu": True, "out_f16": True},
        # a decode step of four sequences through whole 27B layers
        {"name": "chain_t4_27b", "kind": "chain", "hidden": 5120, "n_qkv": 7168, "n_ff": 17408, "group": 128, "t": 4,
         "layers": 4, "fused": True},
        # sixteen sequences, the down projection: few output rows, a long k
        {"name": "linear_t16_down_27b", "kind": "linear", "n": 5120, "k": 17408, "group": 128, "bf16": False, "t": 16,
         "layers": 4, "glu": False, "out_f16": False},
        # an odd batch through a dense linear of an expert model (group 32, bf16 scales)
        {"name": "linear_t37_g32_bf16", "kind": "linear", "n": 5120, "k": 2048, "group": 32, "bf16": True, "t": 37,
         "layers": 16, "glu": False, "out_f16": False},
        # a serving batch of 64 sequences through the widest projection
        {"name": "glu_t64_27b", "kind": "linear", "n": 34816, "k": 5120, "group": 128, "bf16": False, "t": 64, "layers": 2,
         "glu": True, "out_f16": True},
        # a short prompt of ragged length through a whole 27B layer
        {"name": "chain_t300_27b", "kind": "chain", "hidden": 5120, "n_qkv": 7168, "n_ff": 17408, "group": 128, "t": 300,
         "layers": 2, "fused": True},
        # a long prompt chunk through the widest projection: the largest call
        {"name": "glu_t4096_27b", "kind": "linear", "n": 34816, "k": 5120, "group": 128, "bf16": False, "t": 4096,
         "layers": 1, "glu": True, "out_f16": True},
        # one token through expert FFNs (128 experts, 8 chosen): latency again, eight experts' weights
        {"name": "moe_t1", "kind": "moe", "n_exp": 128, "top_k": 8, "h": 2048, "n_ff": 768, "group": 32, "bf16": False,
         "t": 1, "layers": 6},
        # a serving batch: nearly every expert is hit by a few tokens (bf16 scales, as such checkpoints hold)
        {"name": "moe_t64_bf16", "kind": "moe", "n_exp": 128, "top_k": 8, "h": 2048, "n_ff": 768, "group": 32, "bf16": True,
         "t": 64, "layers": 2},
        # a prompt of ragged length, bf16 scales
        {"name": "moe_t517_bf16", "kind": "moe", "n_exp": 128, "top_k": 8, "h": 2048, "n_ff": 768, "group": 32, "bf16": True,
         "t": 517, "layers": 2},
        # a long prompt chunk, f16 scales
        {"name": "moe_t2048", "kind": "moe", "n_exp": 128, "top_k": 8, "h": 2048, "n_ff": 768, "group": 32, "bf16": False,
         "t": 2048, "layers": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "chain", "moe", "moe"])
    if kind == "linear":
        if rng.random() < 0.5:
            n, k = rng.choice(DENSE)
        else:
            n, k = _log_int(rng, 512, 40000), 128 * _log_int(rng, 8, 136)
        glu = rng.random() < 0.3
        if glu:
            n = max(32, n // 32 * 32)
        elif rng.random() < 0.7:
            n = max(16, n // 16 * 16)
        t = _log_int(rng, 1, 4096)
        while 2.0 * t * n * k > 1.4e12:
            t = (t * 3) // 4
        group, bf16 = rng.choice([(128, False), (128, False), (32, True), (32, False)])
        layers = 1 if t > 256 else max(1, min(16, math.ceil(1.2e8 / (n * k / 2))))
        return {"kind": kind, "n": n, "k": k, "group": group, "bf16": bf16, "t": t, "layers": layers, "glu": glu,
                "out_f16": glu or rng.random() < 0.5}
    if kind == "chain":
        hidden, n_qkv, n_ff = rng.choice([(5120, 7168, 17408), (4096, 6144, 11008), (2560, 3840, 6912), (2048, 2560, 5632)])
        t = _log_int(rng, 1, 1000)
        return {"kind": kind, "hidden": hidden, "n_qkv": n_qkv, "n_ff": n_ff, "group": 128, "t": t,
                "layers": 4 if t <= 64 else 2, "fused": rng.random() < 0.7}
    n_exp, top_k, h, n_ff = rng.choice([(128, 8, 2048, 768), (64, 6, 2048, 1408), (32, 4, 2048, 1024), (8, 2, 4096, 3584)])
    group, bf16 = rng.choice([(32, False), (32, True), (32, True), (128, False)])
    return {"kind": kind, "n_exp": n_exp, "top_k": top_k, "h": h, "n_ff": n_ff, "group": group, "bf16": bf16,
            "t": _log_int(rng, 1, 2048), "layers": 1}


class _Program:
    """A program's one library context, shared by every state that is alive, and the name slots its models use."""

    def __init__(self):
        self.dec = ops.W4a16Dec()
        self.slots = []
        self.taken = 0

    def slot(self):
        if self.slots:
            return self.slots.pop()
        self.taken += 1
        return self.taken - 1


_live = weakref.WeakValueDictionary()


def _program():
    p = _live.get("program")
    if p is None:
        p = _live["program"] = _Program()
    return p


class _State:
    """What a program holds for one model: the registered weights (by name), its inputs and its result buffers."""

    def __init__(self, case, program, slot):
        self.case, self.program, self.slot = case, program, slot
        self.dec = program.dec
        weakref.finalize(self, program.slots.append, slot)  # the names are used again by the next model


def _words(g, *shape):
    """Packed int4 weights: eight uniform nibbles per word."""
    return torch.randint(-2**31, 2**31, shape, dtype=torch.int64, device="cuda", generator=g).to(torch.int32).cpu().numpy().view(np.uint32)


def _scales(g, bf16, *shape):
    s = torch.rand(shape, device="cuda", generator=g) * 0.018 + 0.002
    return s.to(torch.bfloat16 if bf16 else torch.float16).view(torch.int16).cpu().numpy().view(np.uint16)


def _normal(g, *shape, dtype=torch.float16):
    return torch.randn(shape, device="cuda", generator=g).to(dtype)


def prepare(case, seed):
    p = _program()
    s = _State(case, p, p.slot())
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dec, t, layers, prefix = s.dec, case["t"], case["layers"], "m%d" % s.slot
    s.names = ["%s.%d" % (prefix, i) for i in range(layers)]
    if case["kind"] == "linear":
        n, k, group = case["n"], case["k"], case["group"]
        for i, name in enumerate(s.names):
            if case["bf16"]:
                dec.upload_lin_g(name, _words(g, n, k // 8), _scales(g, True, n, k // group), n, k, group, True)
            else:
                dec.upload_lin_synth(name, n, k, group, gen.shape_seed(n, k, seed, 2 * i), gen.shape_seed(n, k, seed, 2 * i + 1))
            dec.drop_raw(name)
        s.x = [_normal(g, t, k) for _ in s.names]
        s.y = [torch.empty(t, n // 2 if case["glu"] else n, device="cuda", dtype=torch.float16 if case["out_f16"] else torch.float32)
               for _ in s.names]
    elif case["kind"] == "chain":
        seeds = dec.upload_chain_synth(prefix, layers, case["hidden"], case["n_qkv"], case["n_ff"], case["group"], seed=seed)
        for name in seeds:
            dec.drop_raw(name)
            dec.row_norm_max(name)  # part of loading a model whose chain runs fused
        s.prefix = prefix
        s.x = _normal(g, t, case["hidden"])
        s.y = torch.empty(t, case["hidden"], device="cuda", dtype=torch.float16)
    else:
        e, h, n_ff, group, bf16 = case["n_exp"], case["h"], case["n_ff"], case["group"], case["bf16"]
        for name in s.names:
            dec.upload_experts(name, _words(g, e, 2 * n_ff, h // 8), _scales(g, bf16, e, 2 * n_ff, h // group),
                               _words(g, e, h, n_ff // 8), _scales(g, bf16, e, h, n_ff // group), e, h, n_ff, group, bf16)
        s.x = [_normal(g, t, h) for _ in s.names]
        s.logits = [_normal(g, t, e, dtype=torch.float32) for _ in s.names]
        s.idx = [torch.empty(t, case["top_k"], device="cuda", dtype=torch.int32) for _ in s.names]
        s.wt = [torch.empty(t, case["top_k"], device="cuda", dtype=torch.float32) for _ in s.names]
        s.y = [torch.empty(t, h, device="cuda", dtype=torch.float32) for _ in s.names]
    torch.cuda.synchronize()  # the library launches on a stream of its own
    return s


def run(s):
    c, dec, t = s.case, s.dec, s.case["t"]
    if c["kind"] == "linear":
        for name, x, y in zip(s.names, s.x, s.y):
            if c["glu"]:
                dec.lin_forward_glu(name, x.data_ptr(), y.data_ptr(), t)
            else:
                dec.lin_forward(name, x.data_ptr(), y.data_ptr(), t, out_f16=c["out_f16"])
        return s.y
    if c["kind"] == "chain":
        step = dec.chain_forward_fused if c["fused"] else dec.chain_forward
        step(s.prefix, 0, c["layers"], s.x.data_ptr(), t, s.y.data_ptr())
        return s.y
    for name, x, lg, idx, wt, y in zip(s.names, s.x, s.logits, s.idx, s.wt, s.y):
        dec.moe_route(lg.data_ptr(), t, c["n_exp"], c["top_k"], idx.data_ptr(), wt.data_ptr())
        dec.moe_ffn(name, x.data_ptr(), idx.data_ptr(), wt.data_ptr(), t, c["top_k"], y.data_ptr())
    return s.y, s.idx, s.wt


def _weights(n, k, group):
    return n * k // 2 + 2 * n * (k // group)


def work(case):
    t, layers = case["t"], case["layers"]
    if case["kind"] == "linear":
        n, k = case["n"], case["k"]
        out = t * (n // 2 if case["glu"] else n) * (2 if case["out_f16"] else 4)
        return {"bytes": layers * (_weights(n, k, case["group"]) + 2 * t * k + out), "flops": 2.0 * layers * t * n * k}
    if case["kind"] == "chain":
        h, q, f, g = case["hidden"], case["n_qkv"], case["n_ff"], case["group"]
        mats = [(q, h), (h, h), (2 * f, h), (h, f)]
        return {"bytes": layers * sum(_weights(n, k, g) for n, k in mats) + 4 * t * h,
                "flops": 2.0 * layers * t * sum(n * k for n, k in mats)}
    e, h, f, g, top = case["n_exp"], case["h"], case["n_ff"], case["group"], case["top_k"]
    hit = e * (1.0 - (1.0 - top / e) ** t)  # experts that t tokens reach
    return {"bytes": layers * (hit * (_weights(2 * f, h, g) + _weights(h, f, g)) + t * (2 * h + 4 * h + 4 * e + 8 * top)),
            "flops": 2.0 * layers * t * top * 3 * f * h}


def tolerance(case):
    # each bound is about four times the measured distance of two correct evaluations
    if case["kind"] == "linear":
        # f32 results: sums of up to 17408 products in another order differ by 2e-7 to 7e-7 (the lane order of the
        # repository's oracle); f16 results: their rounding, 2.1e-4 against 64-bit values, at most one unit per value
        return {"rel": 8e-4, "max": 4e-3} if case["out_f16"] else {"rel": 1.5e-6, "max": 1e-5}
    if case["kind"] == "chain":
        return {"rel": 2e-3, "max": 8e-2}  # f16 hand-overs rounded before or after their 1/rms factor: 5.8e-4, 2.1e-2
    return {"rel": 1.5e-3, "max": 8e-3, "differ": 0.0}  # f16 gate, up, activation, expert outputs: 4e-4, 2e-3 against 64 bits
