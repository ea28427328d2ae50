"""The work that a program using this framework has it do, as cases that can be timed and compared.

Every case goes through the package's device operators (`rocmforge_amd.ops`) the way an inference program calls
them: quantised weights resident on the GPU, new activations for every pass.  The kinds of work:

  project   one projection of a decode step, y = x . W^T for 1..8 sequences; with "norm" the RMSNorm before it is
            part of the call
  mlp       the SwiGLU block of a decode step (RMSNorm, gate, up, activation, down) for 1..8 sequences
  prompt    one projection of a prompt (or of more sequences than a decode kernel takes) on fp16 activations
  qkv       the three attention projections of a prompt: the activations arranged once, multiplied three times
  mx        one projection of a prompt on the block-scaled matrix cores: activations re-encoded, then multiplied
  dequant   a weight tensor to float32, as a loader does for tensors that it does not keep packed

`listed()` holds fixed sizes, `draw()` more of the same ranges.
"""
from __future__ import annotations

import math

import torch

from rocmforge_amd import _lib, ops
from rocmforge_amd import quantize as Q

FORMATS = {name: fmt for fmt, name in Q.NAMES.items()}
DECODE = ("Q4_0", "Q8_0", "Q4_K", "Q6_K", "MXFP4", "MXFP6_E2M3", "GGUF_Q4_0", "GGUF_Q8_0", "GGUF_Q4_K", "GGUF_Q6_K")
PROMPT = ("Q4_0", "Q8_0", "Q4_K", "Q6_K", "GGUF_Q4_0", "GGUF_Q8_0", "GGUF_Q4_K", "GGUF_Q6_K")
LOADER = DECODE + ("Q2_K", "Q3_K", "Q5_K")
MX = ("MXFP4", "MXFP6_E2M3")

# multiply-adds of the largest prompt projection that is listed
MOST_PROMPT = 512 * 14336 * 4096


def listed():
    return [
        # The smallest call: one projection of a 0.5-billion-parameter model, one sequence.  Latency.
        {"name": "decode_small", "kind": "project", "fmt": "Q4_0", "m": 1, "n": 4864, "k": 896, "norm": False},
        # The MLP projection of an 8-billion-parameter model for one sequence: the framework's headline shape.
        {"name": "decode_one", "kind": "project", "fmt": "Q4_K", "m": 1, "n": 14336, "k": 4096, "norm": False},
        # The same model's square projections for eight sequences decoded together.
        {"name": "decode_eight", "kind": "project", "fmt": "Q8_0", "m": 8, "n": 4096, "k": 4096, "norm": False},
        # The vocabulary projection, once per generated token; GGUF files keep that tensor in Q6_K.
        {"name": "vocabulary", "kind": "project", "fmt": "GGUF_Q6_K", "m": 1, "n": 128256, "k": 4096, "norm": False},
        # The MLP block of one layer for one sequence, weights as a GGUF file holds them.
        {"name": "mlp_one", "kind": "mlp", "fmt": "GGUF_Q4_K", "down": "GGUF_Q4_K", "m": 1, "hidden": 4096, "inter": 14336},
        # The MLP block of a 13-billion-parameter model for a few sequences; mixed files keep the down projection in Q6_K.
        {"name": "mlp_few", "kind": "mlp", "fmt": "GGUF_Q4_K", "down": "GGUF_Q6_K", "m": 5, "hidden": 5120, "inter": 13824},
        # A short turn of a conversation (or a few dozen sequences decoded together).
        {"name": "prompt_short", "kind": "prompt", "fmt": "GGUF_Q4_K", "m": 37, "n": 4096, "k": 4096, "out": "f16"},
        # A 512-token prompt through the MLP projection of the 8-billion-parameter model.
        {"name": "prompt_512", "kind": "prompt", "fmt": "Q4_K", "m": 512, "n": 14336, "k": 4096, "out": "f16"},
        # A ragged prompt through the down projection of the 13-billion-parameter model, float32 for the residual.
        {"name": "prompt_ragged", "kind": "prompt", "fmt": "Q8_0", "m": 333, "n": 5120, "k": 13824, "out": "f32"},
        # Q, K and V of one layer for a medium prompt with grouped heads: one input, three weights.
        {"name": "attention_in", "kind": "qkv", "fmt": "GGUF_Q4_K", "m": 160, "hidden": 4096, "n": 4096, "kv": 1024},
        # The largest: a 2048-token prompt through the MLP projection of a 70-billion-parameter model in MXFP4.
        {"name": "prompt_mx", "kind": "mx", "fmt": "MXFP4", "m": 2048, "n": 28672, "k": 8192},
        # One weight tensor of the 8-billion-parameter model to float32.
        {"name": "load", "kind": "dequant", "fmt": "Q6_K", "n": 14336, "k": 4096},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _width(rng, lo, hi):
    """The width of an output: mostly a multiple of 64, sometimes any number (vocabularies, split tensors)."""
    return _log(rng, lo, hi, 64 if rng.random() < 0.75 else 1)


def draw(rng):
    kind = rng.choice(("project",) * 4 + ("mlp",) * 2 + ("prompt",) * 3 + ("qkv", "mx", "dequant"))
    if kind == "project":
        fmt = rng.choice(DECODE)
        k = _log(rng, 512, 14336, Q.BLOCK_ELEMS[FORMATS[fmt]])
        if rng.random() < 0.15:                                    # a vocabulary
            return {"kind": kind, "fmt": fmt, "m": 1, "n": _width(rng, 32000, 131072), "k": min(k, 4096), "norm": False}
        return {"kind": kind, "fmt": fmt, "m": rng.choice((1, 1, 1, 2, 3, 4, 6, 8)), "n": _width(rng, 512, 16384), "k": k,
                "norm": rng.random() < 0.25}
    if kind == "mlp":
        fmt = rng.choice(DECODE)
        hidden = _log(rng, 768, 5120, 256)
        return {"kind": kind, "fmt": fmt, "down": rng.choice((fmt, fmt, "GGUF_Q6_K", "Q8_0")), "m": rng.choice((1, 1, 1, 2, 4, 5, 8)),
                "hidden": hidden, "inter": hidden * rng.randint(10, 14) // 4 // 256 * 256}
    if kind == "prompt":
        fmt = rng.choice(PROMPT)
        m, k = _log(rng, 9, 2048), _log(rng, 768, 14336, 256)
        return {"kind": kind, "fmt": fmt, "m": m, "n": _width(rng, 768, max(769, min(14336, MOST_PROMPT // (m * k)))), "k": k,
                "out": rng.choice(("f16", "f16", "f32"))}
    if kind == "qkv":
        hidden = _log(rng, 768, 5120, 256)
        return {"kind": kind, "fmt": rng.choice(PROMPT), "m": _log(rng, 9, 1024), "hidden": hidden, "n": hidden,
                "kv": hidden // rng.choice((1, 4, 8))}
    if kind == "mx":
        m, k = _log(rng, 16, 2048), _log(rng, 1024, 8192, 128)
        return {"kind": kind, "fmt": rng.choice(MX), "m": m, "n": _width(rng, 1024, 28672), "k": k}
    n = _log(rng, 768, 28672, 64)
    return {"kind": kind, "fmt": rng.choice(LOADER), "n": n, "k": _log(rng, 768, 8192, 256)}


# ---- inputs: what quantising zero-mean weights of deviation 0.02 gives in each layout, made on the GPU ----------------


def _codes(g, shape, middle, spread, top):
    """Codes of normally distributed weights: integers 0..top around `middle`."""
    return torch.randn(shape, generator=g, device="cuda").mul_(spread).add_(middle).round_().clamp_(0, top).to(torch.uint8)


def _near(g, shape, value, sign=False):
    """Scales that differ from block to block as the largest weight of a block does."""
    v = value * (0.75 + 0.5 * torch.rand(shape, generator=g, device="cuda"))
    return v * (torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1) if sign else v


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _random(g, shape, top=256):
    return torch.randint(0, top, shape, generator=g, device="cuda", dtype=torch.uint8)


def _pack6(c):
    """[..., 4j] 6-bit codes -> [..., 3j] bytes, a little-endian bit stream."""
    c = c.view(*c.shape[:-1], -1, 4)
    b = torch.stack((c[..., 0] | (c[..., 1] << 6), (c[..., 1] >> 2) | (c[..., 2] << 4), (c[..., 2] >> 4) | (c[..., 3] << 2)), -1)
    return b.view(*c.shape[:-2], -1)


def _mx_blocks(g, fmt, blocks, std):
    """The reference's packer: a power-of-two scale from the block's largest value, then the nearest code."""
    v = torch.randn((blocks, 32), generator=g, device="cuda") * std
    e = v.abs().amax(1).log2().round()
    v = v / e.exp2()[:, None]
    if fmt == "MXFP4":
        code = (v.abs() > 0.75).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
        body = (code[:, 0::2] << 4) | code[:, 1::2]
    else:
        table = torch.tensor([(1 + j / 8) * 2.0 ** (x - 1) for x in range(4) for j in range(8)], device="cuda")
        code = torch.bucketize(v.abs().clamp(0.5, 7.5), (table[1:] + table[:-1]) / 2).to(torch.uint8) | ((v < 0).to(torch.uint8) << 5)
        body = _pack6(code)
    return torch.cat((_bytes(e.to(torch.int8)[:, None]), body), 1)


def _blocks(g, fmt, blocks):
    if fmt in ("MXFP4", "MXFP6_E2M3"):
        return _mx_blocks(g, fmt, blocks, 0.02)
    if fmt in ("Q4_0", "GGUF_Q4_0"):
        c = _codes(g, (blocks, 32), 8, 3.3, 15)
        d = _near(g, (blocks, 1), 0.006, True)
        if fmt == "Q4_0":
            return torch.cat((_bytes(d), c[:, 0::2] | (c[:, 1::2] << 4)), 1)
        return torch.cat((_bytes(d.half()), c[:, :16] | (c[:, 16:] << 4)), 1)
    if fmt in ("Q8_0", "GGUF_Q8_0"):
        c = _codes(g, (blocks, 32), 128, 53.0, 255)
        d = _near(g, (blocks, 1), 0.00038)
        return torch.cat((_bytes(d), c), 1) if fmt == "Q8_0" else torch.cat((_bytes(d.half()), c ^ 0x80), 1)
    if fmt == "Q4_K":                                              # integer minimums beside one-sided codes, 28 bytes apart
        out = _random(g, (blocks, 256))
        out[:, 0:16] = _bytes(_near(g, (blocks, 8), 0.015, True).half())
        out[:, 16:24] = _random(g, (blocks, 8), 5) - 2
        return out
    if fmt in ("Q6_K", "Q3_K", "Q5_K", "Q2_K"):
        out = _random(g, (blocks, 256))
        out[:, 0:32] = _bytes(_near(g, (blocks, 16), 0.0013, True).half())
        if fmt == "Q6_K":
            out[:, 32:224] = _pack6((_codes(g, (blocks, 256), 32, 13.0, 63) - 32) & 63)
        elif fmt == "Q2_K":
            out[:, 32:64] = _bytes(_near(g, (blocks, 16), 0.002).half())
        return out
    if fmt == "GGUF_Q4_K":
        c = _codes(g, (blocks, 4, 2, 32), 7.5, 3.4, 15)
        sc, mn = _codes(g, (blocks, 8), 50, 6.0, 63), _codes(g, (blocks, 8), 50, 6.0, 63)
        head = torch.cat((_bytes(_near(g, (blocks, 1), 1.2e-4).half()), _bytes(_near(g, (blocks, 1), 9e-4).half())), 1)
        scales = torch.cat((sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)), 1)
        return torch.cat((head, scales, (c[:, :, 0] | (c[:, :, 1] << 4)).reshape(blocks, 128)), 1)
    c = _codes(g, (blocks, 2, 4, 32), 32, 13.0, 63)                # GGUF_Q6_K
    lo, hi = c & 15, c >> 4
    ql = torch.cat((lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)), 2).reshape(blocks, 128)
    qh = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(blocks, 64)
    sc = _codes(g, (blocks, 16), 100, 12.0, 127)
    return torch.cat((ql, qh, sc, _bytes(_near(g, (blocks, 1), 1.5e-5).half())), 1)


def _weights(g, fmt, n, k):
    blocks = n * k // Q.BLOCK_ELEMS[FORMATS[fmt]]
    step = (1 << 26) // Q.BLOCK_ELEMS[FORMATS[fmt]]                # in pieces: the codes take far more room than the bytes
    out = torch.empty((blocks, Q.BLOCK_BYTES[FORMATS[fmt]]), dtype=torch.uint8, device="cuda")
    for at in range(0, blocks, step):
        out[at:at + step] = _blocks(g, fmt, min(step, blocks - at))
    return out.view(-1)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def prepare(case, seed):
    c, kind = case, case["kind"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = {"case": c, "f": FORMATS[c["fmt"]]}
    if kind == "project":
        s.update(w=_weights(g, c["fmt"], c["n"], c["k"]), x=_normal(g, c["m"], c["k"]))
        if c["norm"]:
            s["norm"] = 1 + 0.1 * _normal(g, c["k"])
    elif kind == "mlp":
        s.update(gate=_weights(g, c["fmt"], c["inter"], c["hidden"]), up=_weights(g, c["fmt"], c["inter"], c["hidden"]),
                 down=_weights(g, c["down"], c["hidden"], c["inter"]), x=_normal(g, c["m"], c["hidden"]), norm=1 + 0.1 * _normal(g, c["hidden"]))
    elif kind == "prompt":
        s.update(w=_weights(g, c["fmt"], c["n"], c["k"]), a=_normal(g, c["m"], c["k"]).half())
    elif kind == "qkv":
        s.update(w=[_weights(g, c["fmt"], n, c["hidden"]) for n in (c["n"], c["kv"], c["kv"])], a=_normal(g, c["m"], c["hidden"]).half())
    elif kind == "mx":
        w = _weights(g, c["fmt"], c["n"], c["k"])
        s.update(w=ops.MxOperand(s["f"], w, c["n"], c["k"]), a=_mx_blocks(g, "MXFP4", c["m"] * c["k"] // 32, 1.0).view(-1))
    else:
        s["w"] = _weights(g, c["fmt"], c["n"], c["k"])
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "project":
        if c["norm"]:
            return ops.rms_norm_gemv(s["f"], s["w"], s["x"], s["norm"], 1e-5, c["n"], c["k"])
        return ops.gemv(s["f"], s["w"], s["x"], c["n"], c["k"])
    if kind == "mlp":
        return ops.mlp_swiglu(s["f"], s["gate"], s["up"], FORMATS[c["down"]], s["down"], s["x"], s["norm"], 1e-5, c["hidden"], c["inter"])
    if kind == "prompt":
        return ops.gemm_f16(s["f"], s["w"], s["a"], c["n"], c["k"], torch.float16 if c["out"] == "f16" else torch.float32)
    if kind == "qkv":
        a = ops.ArrangedA(s["a"])
        return [ops.gemm_f16_arranged(s["f"], w, a, n) for w, n in zip(s["w"], (c["n"], c["kv"], c["kv"]))]
    if kind == "mx":
        return ops.gemm_mx(ops.MxOperand(Q.MXFP4, s["a"], c["m"], c["k"], _lib.MX_FP4_UNCHECKED), s["w"])
    return ops.dequant(s["f"], s["w"], c["n"] * c["k"])


def work(case):
    c, kind = case, case["kind"]

    def packed(fmt, n, k):
        return Q.packed_bytes(FORMATS[fmt], n * k)

    if kind == "project":
        return {"bytes": packed(c["fmt"], c["n"], c["k"]) + 4 * (c["m"] * (c["n"] + c["k"]) + (c["k"] if c["norm"] else 0)),
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind == "mlp":
        h, i = c["hidden"], c["inter"]
        return {"bytes": 2 * packed(c["fmt"], i, h) + packed(c["down"], h, i) + 4 * (2 * c["m"] * h + h), "flops": 6 * c["m"] * h * i}
    if kind == "prompt":
        return {"bytes": packed(c["fmt"], c["n"], c["k"]) + 2 * c["m"] * c["k"] + (2 if c["out"] == "f16" else 4) * c["m"] * c["n"],
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind == "qkv":
        n = c["n"] + 2 * c["kv"]
        return {"bytes": packed(c["fmt"], n, c["hidden"]) + 2 * c["m"] * (c["hidden"] + n), "flops": 2 * c["m"] * n * c["hidden"]}
    if kind == "mx":
        per_weight = 33 / 64 if c["fmt"] == "MXFP4" else 33 / 32   # an element code, and a scale byte for every 32 of them
        return {"bytes": int(per_weight * c["n"] * c["k"]) + c["m"] * c["k"] // 32 * 17 + 2 * c["m"] * c["n"], "flops": 2 * c["m"] * c["n"] * c["k"]}
    return {"bytes": packed(c["fmt"], c["n"], c["k"]) + 4 * c["n"] * c["k"], "flops": c["n"] * c["k"]}


def tolerance(case):
    """About four times what the results differ from the same contraction in 64 bits ("rel", "max" as measured):
    float32 projections 1.1e-6, 3.2e-6 and MLP blocks 2.2e-6, 1.1e-5 (22 bits per activation and float32 sums); prompts in
    float32 1.1e-6, 5.5e-6 (Q4_K, whose products q * scale are rounded to fp16 once: 2.0e-5, 9.5e-5), in fp16 2.1e-4, 5.3e-4;
    bfloat16 results 1.8e-3, 3.2e-3.  Dequantisation has no freedom."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "project":
        return {"rel": 5e-6, "max": 1.5e-5}
    if kind == "mlp":
        return {"rel": 1e-5, "max": 4e-5}
    if kind == "mx":
        return {"rel": 7e-3, "max": 1.3e-2}
    if case.get("out") == "f32":
        return {"rel": 8e-5, "max": 4e-4} if case["fmt"] == "Q4_K" else {"rel": 5e-6, "max": 2.5e-5}
    return {"rel": 8e-4, "max": 2e-3}
