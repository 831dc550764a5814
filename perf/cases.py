"""The work that a program built on this package has it do, as cases that can be timed and checked.

Each case is one pass through the public entry points of lastengine_amd.Engine over weights that stay on
the GPU, as an inference engine makes it between two of its own kernels:

  matmul   one weight matrix: a single projection, or the output head, at one token or a few
  dense    the quantized matmuls of dense transformer layers: at one token q, k and v over a pointer
           table, o, gate and up as one matrix, and down with the SwiGLU formed inside it; at more tokens
           (speculative verify, batches, prompt processing) the same matrices through the GEMM
  int8     the same at one token in the int8 activation mode (RMSNorm and quantization fused)
  moe      routed expert layers, from one token to prompt size
  dequant  rows of a matrix to fp32 (embedding rows, loading)

`layers` counts layers with weights of their own, as a model has them: one pass then streams from HBM what a
model's pass streams, instead of finding one matrix in the caches.
"""
import base64
import math

import numpy as np
import torch

import lastengine_amd as le

TYPES = {"Q4_0": 2, "Q8_0": 8, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ2_XXS": 16, "IQ3_XXS": 18, "IQ2_S": 22}
# values and bytes of a block (the GGUF layouts)
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q3_K": (256, 110), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210),
         "IQ2_XXS": (256, 66), "IQ3_XXS": (256, 98), "IQ2_S": (256, 82)}
EPS = 1e-5


def row_bytes(ty, cols):
    v, b = BLOCK[ty]
    return cols // v * b


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: one k or v projection at hidden 2048, where the launch is most of the time
        {"name": "kv_projection", "kind": "matmul", "ty": "Q4_K", "rows": 1024, "cols": 2048, "tokens": 1},
        # the output head at one token
        {"name": "head_q8_0", "kind": "matmul", "ty": "Q8_0", "rows": 32000, "cols": 4096, "tokens": 1},
        # decode: four layers of the benchmark's dense model (Q4_K, Q6_K down)
        {"name": "decode_q4_k", "kind": "dense", "layers": 4, "tokens": 1, "hidden": 4096, "q_rows": 4096, "kv_rows": 1024,
         "ff": 14336, "ty_attn": "Q4_K", "ty_ffn": "Q4_K", "ty_down": "Q6_K"},
        # decode of a low-bit quantization (the benchmark's IQ types)
        {"name": "decode_iq", "kind": "dense", "layers": 4, "tokens": 1, "hidden": 4096, "q_rows": 4096, "kv_rows": 1024,
         "ff": 14336, "ty_attn": "IQ2_S", "ty_ffn": "IQ2_XXS", "ty_down": "IQ3_XXS"},
        # decode in the int8 activation mode, at widths whose super-block counts are odd or hardly divide
        {"name": "decode_int8", "kind": "int8", "layers": 4, "tokens": 1, "hidden": 2560, "q_rows": 2560, "kv_rows": 640,
         "ff": 6912, "ty_attn": "Q5_K", "ty_ffn": "Q4_K", "ty_down": "Q6_K"},
        # speculative verify: four drafted tokens through two layers
        {"name": "verify_4", "kind": "dense", "layers": 2, "tokens": 4, "hidden": 4096, "q_rows": 4096, "kv_rows": 1024,
         "ff": 14336, "ty_attn": "Q4_K", "ty_ffn": "Q4_K", "ty_down": "Q6_K"},
        # a batch of decoding requests, an odd count, on a smaller model in a mix of types
        {"name": "batch_37", "kind": "dense", "layers": 2, "tokens": 37, "hidden": 3072, "q_rows": 3072, "kv_rows": 768,
         "ff": 8192, "ty_attn": "Q5_K", "ty_ffn": "Q4_K", "ty_down": "Q6_K"},
        # prompt processing: 512 tokens through one layer of the benchmark's dense model
        {"name": "prompt_512", "kind": "dense", "layers": 1, "tokens": 512, "hidden": 4096, "q_rows": 4096, "kv_rows": 1024,
         "ff": 14336, "ty_attn": "Q4_K", "ty_ffn": "Q4_K", "ty_down": "Q6_K"},
        # expert layers (128 experts, top 8): one token, a small batch, prompt size
        {"name": "moe_1", "kind": "moe", "layers": 2, "tokens": 1, "n_exp": 128, "k": 8, "hidden": 2048, "ff": 768,
         "ty_gate": "Q4_K", "ty_down": "Q6_K", "tables": False},
        {"name": "moe_12", "kind": "moe", "layers": 2, "tokens": 12, "n_exp": 128, "k": 8, "hidden": 2048, "ff": 768,
         "ty_gate": "Q4_K", "ty_down": "Q6_K", "tables": True},
        {"name": "moe_prompt_2048", "kind": "moe", "layers": 1, "tokens": 2048, "n_exp": 128, "k": 8, "hidden": 2048, "ff": 768,
         "ty_gate": "Q4_K", "ty_down": "Q6_K", "tables": False},
        # a quarter of an output head's rows to fp32
        {"name": "dequant_rows", "kind": "dequant", "ty": "Q6_K", "rows": 8000, "cols": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sb(rng, lo, hi):
    """A width: a multiple of 256 from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, _log(rng, lo, hi) // 256 * 256))


def _layer(rng, kind, tokens, types):
    hidden = _sb(rng, 1024, 4096)
    q_rows = rng.choice([hidden, hidden, min(4096, 2 * hidden)])
    kv_rows = q_rows // rng.choice([1, 2, 4])
    case = {"kind": kind, "layers": 1, "tokens": tokens, "hidden": hidden, "q_rows": q_rows, "kv_rows": kv_rows,
            "ff": _sb(rng, 2 * hidden, 14336 * hidden // 4096 // 256 * 256), "ty_attn": rng.choice(types), "ty_ffn": rng.choice(types),
            "ty_down": rng.choice(types)}
    if tokens == 1:  # about a model's worth of bytes, as far as four layers go
        case["layers"] = max(1, min(4, -(-(100 << 20) // _layer_bytes(case))))
    return case


def draw(rng):
    common, every = ["Q4_K", "Q5_K", "Q6_K", "Q8_0"], list(TYPES)
    kind = rng.choice(["matmul", "dense", "dense", "batch", "batch", "int8", "moe", "moe", "dequant"])
    if kind == "matmul":
        return {"kind": "matmul", "ty": rng.choice(every), "rows": _log(rng, 512, 40000), "cols": _sb(rng, 1024, 8192),
                "tokens": rng.choice([1, 1, 1, rng.randint(2, 8)])}
    if kind == "dense":
        return _layer(rng, "dense", 1, rng.choice([common, every]))
    if kind == "batch":
        return _layer(rng, "dense", _log(rng, 2, 512), rng.choice([common, every]))
    if kind == "int8":
        return _layer(rng, "int8", 1, common)
    if kind == "moe":
        n_exp = _log(rng, 8, 128)
        g, d = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q8_0", "Q8_0"), ("IQ2_XXS", "IQ3_XXS"), (rng.choice(every), rng.choice(every))])
        return {"kind": "moe", "layers": 1, "tokens": _log(rng, 1, 2048), "n_exp": n_exp, "k": rng.randint(1, min(8, n_exp)),
                "hidden": _sb(rng, 1024, 2048), "ff": _sb(rng, 256, 768), "ty_gate": g, "ty_down": d, "tables": rng.random() < 0.5}
    return {"kind": "dequant", "ty": rng.choice(every), "rows": _log(rng, 64, 8000), "cols": _sb(rng, 1024, 4096)}


# ---------------------------------------------------------------- inputs

# root mean square of a weight's integer code (sub-block scale times quant, in units of the super-block scale d)
_CODE_RMS = {"Q4_0": 4.6, "Q8_0": 74.0, "Q3_K": 42.0, "Q4_K": 169.0, "Q5_K": 338.0, "Q6_K": 1369.0, "IQ2_XXS": 40.0, "IQ3_XXS": 125.0, "IQ2_S": 40.0}


def _weights(gen, ty, rows, cols):
    """Blocks of a matrix: every code uniform, and per-block scales that give weights of about N(0, 0.03),
    the offsets of Q4_K and Q5_K centring them as a quantizer of centred weights leaves them."""
    v, bb = BLOCK[ty]
    q = torch.randint(0, 256, (rows * (cols // v), bb), dtype=torch.uint8, device="cuda", generator=gen)
    n = q.shape[0]
    d = (0.03 / _CODE_RMS[ty]) * (0.5 + torch.rand(n, device="cuda", generator=gen))
    if ty in ("Q4_0", "Q6_K", "Q3_K"):  # these take the sign of the block's largest value
        d = torch.where(torch.rand(n, device="cuda", generator=gen) < 0.5, d, -d)
    at = {"Q3_K": 108, "Q6_K": 208}.get(ty, 0)
    q[:, at:at + 2] = d.half().view(torch.uint8).reshape(n, 2)
    if ty in ("Q4_K", "Q5_K"):
        q[:, 2:4] = (d * (7.5 if ty == "Q4_K" else 15.5)).half().view(torch.uint8).reshape(n, 2)
        q[:, 8:12] = q[:, 4:8]  # mins of the first four sub-blocks, and the high bits of the others
        q[:, 12:16] = (q[:, 12:16] & 15) * 17
    return q.reshape(-1)


def _acts(gen, *shape):
    """Normalised activations: N(0, 1) with the few strong channels that real ones have."""
    x = torch.randn(*shape, device="cuda", generator=gen)
    return x * (1.0 + 7.0 * (torch.rand(shape[-1], device="cuda", generator=gen) < 0.004))


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _mats(case):
    """(name, type, rows, cols) of a layer's matrices."""
    h, ff, q, kv = case["hidden"], case["ff"], case["q_rows"], case["kv_rows"]
    a = case["ty_attn"]
    return [("q", a, q, h), ("k", a, kv, h), ("v", a, kv, h), ("o", a, h, q), ("gate_up", case["ty_ffn"], 2 * ff, h),
            ("down", case["ty_down"], h, ff)]


def _layer_bytes(case):
    return sum(r * row_bytes(t, c) for _, t, r, c in _mats(case))


_engine = None


def engine():
    global _engine
    if _engine is None:
        _engine = le.Engine()
    return _engine


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    eng = engine()
    kind, s = case["kind"], {"case": case}
    if kind == "matmul":
        m = case["tokens"]
        s["w"] = _weights(gen, case["ty"], case["rows"], case["cols"])
        s["x"] = _acts(gen, m, case["cols"])
        s["y"] = _empty(m, case["rows"])
        if m > 1:
            s["ws"] = _empty(max(16, eng.gemm_workspace_size_rows(TYPES[case["ty"]], m, case["rows"], case["cols"])), dtype=torch.uint8)
    elif kind in ("dense", "int8"):
        m, mats = case["tokens"], _mats(case)
        s["layers"] = []
        if m > 1:
            s["ws"] = _empty(max(eng.gemm_workspace_size_rows(TYPES[t], m, r, c) for _, t, r, c in mats), dtype=torch.uint8)
        for _ in range(case["layers"]):
            lay = {"w": {n: _weights(gen, t, r, c) for n, t, r, c in mats},
                   "x_attn": _acts(gen, m, case["hidden"]), "x_o": _acts(gen, m, case["q_rows"]), "x_ffn": _acts(gen, m, case["hidden"])}
            if m > 1 or kind == "int8":
                lay["x_down"] = _acts(gen, m, case["ff"])
            if m > 1:
                lay["y"] = {n: _empty(m, r) for n, _, r, _ in mats}
            else:
                q, kv, rb = case["q_rows"], case["kv_rows"], row_bytes(case["ty_attn"], case["hidden"])
                base = [lay["w"]["q"].data_ptr() + j * kv * rb for j in range(q // kv)] + [lay["w"][n].data_ptr() for n in "kv"]
                lay["qkv"] = torch.tensor(base, dtype=torch.int64, device="cuda")
                lay["y"] = {"qkv": _empty(q + 2 * kv), "o": _empty(case["hidden"]), "gate_up": _empty(2 * case["ff"]),
                            "down": _empty(case["hidden"])}
            if kind == "int8":
                lay["norm"] = [1.0 + 0.1 * torch.randn(case["hidden"], device="cuda", generator=gen) for _ in range(2)]
                for n, c in (("attn", case["hidden"]), ("o", case["q_rows"]), ("ffn", case["hidden"]), ("down", case["ff"])):
                    lay["q8_" + n] = (_empty(c, dtype=torch.int8), _empty(c // 32), _empty(c // 32, dtype=torch.int32))
                lay["n_attn"], lay["n_ffn"] = _empty(case["hidden"]), _empty(case["hidden"])
            s["layers"].append(lay)
    elif kind == "moe":
        n, e, k, h, ff = case["tokens"], case["n_exp"], case["k"], case["hidden"], case["ff"]
        tg, td = case["ty_gate"], case["ty_down"]
        s["layers"] = []
        s["ws"] = torch.zeros(max(eng.moe_workspace_size(n, k, ff), eng.moe_prefill_workspace_size(n, k, e, h, ff)), dtype=torch.uint8, device="cuda")
        for _ in range(case["layers"]):
            lay = {"gate": _weights(gen, tg, e * ff, h), "up": _weights(gen, tg, e * ff, h), "down": _weights(gen, td, e * h, ff),
                   "x": _acts(gen, n, h), "out": _empty(n, h), "idx": _empty(n, k, dtype=torch.int32), "wt": _empty(n, k)}
            # router logits: some experts are chosen more often than others
            lay["logits"] = torch.randn(n, e, device="cuda", generator=gen) + 0.5 * torch.randn(e, device="cuda", generator=gen)
            if case["tables"]:
                for name, ty, r, c in (("gate", tg, ff, h), ("up", tg, ff, h), ("down", td, h, ff)):
                    lay[name + "_ptrs"] = lay[name].data_ptr() + torch.arange(e, dtype=torch.int64, device="cuda") * (r * row_bytes(ty, c))
            s["layers"].append(lay)
    else:
        s["w"] = _weights(gen, case["ty"], case["rows"], case["cols"])
        s["y"] = _empty(case["rows"], case["cols"])
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    case, eng = s["case"], engine()
    kind = case["kind"]
    if kind == "matmul":
        ty, r, c = TYPES[case["ty"]], case["rows"], case["cols"]
        if case["tokens"] == 1:
            eng.mv(ty, s["w"], s["x"], s["y"], r, c)
        else:
            eng.gemm(ty, s["w"], s["x"], case["tokens"], s["y"], r, c, ws=s["ws"])
        return s["y"]
    if kind == "dequant":
        eng.dequant_rows(TYPES[case["ty"]], s["w"], s["y"], case["rows"], case["cols"])
        return s["y"]
    out = []
    if kind == "moe":
        tg, td = TYPES[case["ty_gate"]], TYPES[case["ty_down"]]
        shape = (case["n_exp"], case["k"], case["hidden"], case["ff"])
        for lay in s["layers"]:
            if case["tables"]:
                eng.moe_ptrs(tg, tg, td, lay["gate_ptrs"], lay["up_ptrs"], lay["down_ptrs"], *shape, lay["logits"], lay["x"], case["tokens"],
                             lay["out"], lay["idx"], lay["wt"], ws=s["ws"])
            else:
                eng.moe(tg, tg, td, lay["gate"], lay["up"], lay["down"], *shape, lay["logits"], lay["x"], case["tokens"], lay["out"],
                        lay["idx"], lay["wt"], ws=s["ws"])
            out.append({"out": lay["out"], "idx": lay["idx"], "wt": lay["wt"]})
        return out
    ta, tf, td = TYPES[case["ty_attn"]], TYPES[case["ty_ffn"]], TYPES[case["ty_down"]]
    h, ff, q, kv, m = case["hidden"], case["ff"], case["q_rows"], case["kv_rows"], case["tokens"]
    for lay in s["layers"]:
        w, y = lay["w"], lay["y"]
        if kind == "int8":
            a, o, f, d = (lay["q8_" + n] for n in ("attn", "o", "ffn", "down"))
            eng.rms_quant(lay["x_attn"], lay["norm"][0], lay["n_attn"], *a, h, EPS)
            eng.mv_q8(ta, lay["qkv"], *a, y["qkv"], kv, h, 0, q // kv + 2)
            eng.quant_x(lay["x_o"], *o, q // 32)
            eng.mv_q8(ta, None, *o, y["o"], h, q, 0, 1, w=w["o"])
            eng.rms_quant(lay["x_ffn"], lay["norm"][1], lay["n_ffn"], *f, h, EPS)
            eng.mv_q8(tf, None, *f, y["gate_up"], 2 * ff, h, 0, 1, w=w["gate_up"])
            eng.quant_x(lay["x_down"], *d, ff // 32)
            eng.mv_q8(td, None, *d, y["down"], h, ff, 0, 1, w=w["down"])
            out.append({**y, "n_attn": lay["n_attn"], "n_ffn": lay["n_ffn"], "q8": a + f})
        elif m == 1:
            eng.mv_ptrs(ta, lay["qkv"], lay["x_attn"], y["qkv"], kv, h, 0, q // kv + 2)
            eng.mv(ta, w["o"], lay["x_o"], y["o"], h, q)
            eng.mv(tf, w["gate_up"], lay["x_ffn"], y["gate_up"], 2 * ff, h)
            eng.mv_swiglu(td, w["down"], y["gate_up"], y["down"], h, ff)
            out.append(y)
        else:
            for n, ty, x, r, c in (("q", ta, "x_attn", q, h), ("k", ta, "x_attn", kv, h), ("v", ta, "x_attn", kv, h), ("o", ta, "x_o", h, q),
                                   ("gate_up", tf, "x_ffn", 2 * ff, h), ("down", td, "x_down", h, ff)):
                eng.gemm(ty, w[n], lay[x], m, y[n], r, c, ws=s["ws"])
            out.append(y)
    return out


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "dequant":
        return {"bytes": case["rows"] * (row_bytes(case["ty"], case["cols"]) + 4 * case["cols"]), "flops": 0}
    m = case["tokens"]
    if kind == "matmul":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * row_bytes(case["ty"], c) + 4 * m * (r + c), "flops": 2 * m * r * c}
    if kind == "moe":
        e, k, h, ff = case["n_exp"], case["k"], case["hidden"], case["ff"]
        used = e * (1.0 - (1.0 - k / e) ** m)  # experts that some token is routed to, on average
        per = 2 * ff * row_bytes(case["ty_gate"], h) + h * row_bytes(case["ty_down"], ff)
        return {"bytes": case["layers"] * (int(used * per) + m * (8 * h + 4 * e + 8 * k)), "flops": case["layers"] * 6 * m * k * h * ff}
    mats = _mats(case)
    io = sum(4 * m * (r + c) for _, _, r, c in mats)
    return {"bytes": case["layers"] * (_layer_bytes(case) + io), "flops": case["layers"] * 2 * m * sum(r * c for _, _, r, c in mats)}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    # measured against exact() (relative 2-norm), and about four times that stated:
    if kind == "int8":  # 1e-7..4e-7, unless a normalised value lies at a rounding boundary and takes the other integer
        return {"rel": 1e-4, "max": 5e-3, "differ": 1e-3}
    if kind == "moe":  # decode kernels (15-bit activations) 1.1e-4, grouped matrix-core form (fp16 activations) 4e-4
        grouped = case["tokens"] > 8 or (case["ty_gate"], case["ty_down"]) not in _MOE_DECODE
        return {"rel": 1.6e-3, "max": 1.6e-2} if grouped else {"rel": 4e-4, "max": 4e-3}
    if case["tokens"] == 1:  # 15-bit activations per 32 values: 5e-5, down after the SwiGLU 1.1e-4
        return {"rel": 4e-4, "max": 4e-3}
    return {"rel": 1e-3, "max": 1e-2}  # fp16 activations: 2.5e-4


_MOE_DECODE = {("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q6_K", "Q6_K"), ("Q8_0", "Q8_0"), ("IQ2_XXS", "IQ3_XXS"), ("IQ2_XXS", "IQ2_XXS"),
               ("IQ3_XXS", "IQ3_XXS")}


# ---------------------------------------------------------------- the same in 64 bits

# IQ grids of the GGUF formats: entry i holds the levels of its values as digits in base 3 (IQ2_XXS, IQ2_S:
# 8 values of 8, 25, 43) or base 8 (IQ3_XXS: 4 values), lowest first
IQ2_XXS = (
    "AAACAAQABgAIAAoADAASABQAGAAaABwAHgAkACoALgAwADYAOAA+AEoAUgBUAFoAXgBsAIoAlgCiAKQAtgDaAPQA9gD8AAYBCAEOARABFAEgASoBLAEy"
    "AT4BRAFGAUoBVgFkAXgBegGEAZwBngGwAc4B4AHmAeoB7AHyAf4BAgIEAgoCDAIiAjoCUgKKApQC2gLcAuIC7AL0AgYDEgMYAxwDKgMwAzwDTgNWA2AD"
    "kAOaA8wD0gPeA+ID7gMCBCwETARuBHwEwATCBMgE2gT2BBAFFAVYBYYFsgW0BboF0AXgBegF6gUcBiQGVAZWBqYGqAauBsAGzgb2BhIHJgeGB54Hqgfa"
    "B1gIjAiOCJQImgieCKAIpgisCLQIuAjCCMQIygjcCO4ICgkSCRYJLgk2CU4JVglgCX4JhAmQCbQJxAnaCeQJIApyCnQKegqMCpAKwgrsCvAK+goyC1IL"
    "ZAtqC24LdAt2C5oLoAu4C9ILAAxGDJYMmAywDPoMIA1KDVQNWg16DbYN8g1ADkYOWA5wDo4Otg7uDgwPMA80D4oPjA+6D0AQFhEYER4RMhFOEWoRdhGC"
    "EcIRChIMEhISFhIkEjYSWhJ6EpwSshLGEtgS/hJQE6gT8hP4EwQUChQ4FE4UdhSwFOIU9hQAFVgVDBY4FsoW7BYCFyAXahfKF9IYAhk=")
IQ3_XXS = (
    "AAACAAQACQALAA8AEAASABkAIgA7AD0AQQBDAEgASgBRAFUAWABaAGEAbAB4AIAAggCEAIkAkACSAJkAmwCfAKkArwC9AMEAxwDIAMoA1QD4AAsBHwEk"
    "AS8BOwE9AUEBRwFaAWoBnQG0AcgBzAHOAeMB8QEBAgMCCAIKAhECEwIYAhoCHAInAigCQAJCAkkCUAJSAoECgwKIAooCkQKYAroCwALCAtAC2QLmAvYC"
    "AQMFAygDUANUA2YDeQOFA9ID4AMABAIECQQLBBAEEgQWBBkEIgRBBEMERQRIBEoEUQRYBHMEdwR4BIAEggSJBI8EkASSBJ8EoAStBMEEyATMBPgE/AQd"
    "BSsFQwVXBWEFfAXBBcMFzgXlBQEGCAYKBhEGEwYoBjUGOgZABkIGUAZZBmQGZgaBBoMGiAaVBqoGugbJBtsGGAcnBzoHQAdGB1IHbQeMB54HswfbB/AH"
    "BAgPCB0IHwgrCC8IfAiQCJ8IoAiwCLYIxwjlCAQJKQk0CVUJYwl4CcUJyAnKCdgJCgohCjgKQApGClYKbQqMCpoKugrCCusKCAsTCxcLOgtCC1kLqAvU"
    "C+ILFAwkDCYMNAxRDHEMjwy0DNgM3gwkDUUNag2bDcMN0Q0DDgUOBw4IDhoOKg5WDmAOig6lDqoOwA7NDtsO8A4RDyEPQA9CD1QPmA8=")
IQ2_S = (
    "AAACAAQABgAIAAoADAAOABAAEgAUABYAGAAcAB4AIAAiACQAJgAoACoALgAwADIANAA2ADgAOgA8AEAAQgBIAEwAUABSAFQAVgBYAFoAXABeAGAAZABm"
    "AGwAbgBwAHIAdgB4AHoAfAB+AIIAhACIAIoAkACSAJQAmgCcAKIApACmAKgArACuALQAvAC+AMAAwgDEAMYAygDYANwA4ADkAOwA9AD2APgA+gD8AP4A"
    "AAECAQYBCAEKAQwBDgEQARIBFAEWARgBGgEcAR4BIAEiASQBKgEsAS4BMAEyATYBOAE8AT4BRAFGAUgBSgFMAU4BUAFSAVQBVgFaAVwBYAFiAWQBZgFo"
    "AWoBbAFuAXIBdAF6AXwBfgGAAYQBhgGMAZYBmAGaAZwBngGiAbABtAG2AboBvAHCAcwBzgHUAeYB6AHqAewB8AHyAfQB9gH4AfwBAAICAgQCBgIIAgoC"
    "DAIOAhACFAIWAhwCIAIoAjYCOAI6AkACQgJEAkYCSgJSAlYCWAJcAl4CZAJuAnYCiAKSApQCnAKgAqICrALOAtoC3ALeAuAC4gLkAuYC6ALsAu4C8AL0"
    "AvYC+AL6Av4CAAMCAwQDBgMIAwoDDAMQAxIDFAMYAxwDHgMiAyQDKgMsAy4DMAMyAzQDNgM4AzoDPAM+A0ADQgNGA0gDSgNMA04DUANSA1QDWANaA2AD"
    "YgNkA2YDagNsA3wDfgOCA4QDiAOOA5ADlgOaA6ADogOyA7QDugPMA84D0APSA9YD2APaA9wD3gPiA+QD6APqA+wD7gPwA/ID9AP2A/oD/AMCBAQEBgQI"
    "BAwEDgQUBB4EIAQiBCQEJgQoBCoELAQwBDIEOAQ6BDwEPgRCBEQESgRUBFYEXARuBHIEdAR4BHoEgASKBIwEkgSkBL4EwATCBMQExgTIBMwEzgTSBNoE"
    "3ATeBOAE5ATmBOwE9gT4BBAFEgUUBRYFGgUcBSIFLAUuBTQFRAVaBWQFagV8BYoFsgW0BbYFuAW8Bb4FwAXCBcQFyAXMBc4F0AXWBdgF2gXiBegF8AX0"
    "BQIGBAYGBgwGDgYQBhYGHgYgBiIGKAYqBjAGOgY8BkIGVAZcBmgGbAZuBnIGeAaQBpIGogamBqgGqgasBq4Gsga0BrgGugbABsIGxAbGBsoGzAbSBtwG"
    "3gbkBvYG+gb8BgAHAgcIBxIHFAcaBygHLAdIB0oHUAdiB3IHmAecB6IHpAe0B7YHvAfWB+gH6gfsB/IHLAhCCE4Iagh2CHgIjAiOCJAIkgiUCJYImAia"
    "CJwIngigCKIIpgioCKoIrAiuCLAIsgi0CLYIuAi6CLwIwgjECMoIzgjQCNQI1gjcCN4I4AjiCOYI6AjqCOwI7gjwCPII+Aj6CPwI/ggACQIJBAkGCQoJ"
    "DAkSCRQJFgkYCRwJHgkkCS4JMAk2CTgJOgk8CUIJSAlMCU4JUglUCVoJZAlmCX4JgAmCCYQJhgmICYoJjAmOCZAJkgmUCZYJmgmcCZ4JoAmiCaQJpgmo"
    "CawJrgm0CbYJuAm6Cb4JwAnGCdAJ0gnUCdYJ2AnaCdwJ3gniCeQJ6gnsCe4J8An0CfYJ/AkECgYKCAoOCiAKIgokCiYKKgosCjIKPAo+CkQKVgpsCnIK"
    "dAp4CnoKfAp+CoAKhAqGCowKjgqQCpIKlgqYCp4KqgqwCsIKxArGCsgKzArOCtQK3grgCuYK+AoGCxQLFgscCy4LZAtmC2gLagtuC3ALcgt0C3YLeAt6"
    "C3wLgAuCC4QLhguIC4oLjAuOC5ILlAuaC5wLngugC6QLpgu2C7gLugu8C74LwAvCC8QLyAvKC9AL0gvUC9YL2gvcC+IL7AvuC/QLBgwKDAwMEAwSDBgM"
    "IgwkDCoMOgw8DFgMWgxcDF4MYAxiDGQMZgxqDGwMcgx0DHYMeAx8DH4MhAyODJAMlgyoDKoMrAyuDLIMtAy6DMQMxgzMDN4M+gz8DAINEA0UDUoNTA1O"
    "DVANVA1WDVwNZg1oDW4Ndg2ADZwNng2kDbYN7A38DSYOOg4+DkAOQg5GDkgOSg5MDlAOUg5YDlwOXg5iDmQOag52DnwOjg6QDpIOlA6YDpoOoA6qDqwO"
    "sg7EDtQO4g7oDvoOCA8oDzAPNA82DzoPPA9CD0wPTg9UD2YPgg+ED4oPnA+kD7QPwg/SDxQQJBAmECwQVBBoEHQQjhDiEA4RFhEYERoRHBEgESIRJhEo"
    "ESwRMhE0EToRPBE+EUARRBFMEVARVhFYEWgRahFuEXARchF0EXYRehF8EYIRhBGGEYgRjBGOEZ4RoBGmEbYRuBG8EcARwhHEEdQR1hHcEQoSDBIOEhAS"
    "EhIUEhYSGBIcEiQSJhIoEioSLhIwEjYSQBJCEkgSWhJcEl4SYBJkEmYSbBJ2EngSfhKQEpgSrBKuErQSxBLGEvwSABMGEwgTGBMaEyATRhNOE1ATaBN+"
    "E7ITyBPKE9YT6BPwE/IT9hP4E/oT/BP+EwQUChQMFA4UEBQUFBYUHBQmFCgULhRAFEQUShRMFFwUXhRkFGwUkhSUFJoUrBTeFOIU5BTmFOgU7BTuFPQU"
    "/hQAFQYVGBUmFTQVNhU8FU4VeBV8FYQVpBW0FdYV2BXeFewV8BUkFiYWSBZMFrYWyBbMFtAW1BbcFuIW5BbmFuwWEhcYFzQXShdsF3IXfheCF4QXohem"
    "F6gXuBe8F74XxBfWF/gXBhgMGBwYghi2GMYY+BgmGToZVhlYGWIZZBloGYwZoBk=")


def _grid(text, levels, n, device):
    code = torch.from_numpy(np.frombuffer(base64.b64decode(text), dtype="<u2").astype(np.int64)).to(device)
    lv = torch.tensor(levels, dtype=torch.float64, device=device)
    return torch.stack([lv[code // len(levels) ** j % len(levels)] for j in range(n)], 1)


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _k4(b):
    """(scales, mins) of the 12 packed bytes of Q4_K and Q5_K, eight each."""
    b = b.to(torch.int16)
    sc = torch.cat([b[:, 0:4] & 63, (b[:, 8:12] & 15) | (b[:, 0:4] >> 6 << 4)], 1)
    mn = torch.cat([b[:, 4:8] & 63, (b[:, 8:12] >> 4) | (b[:, 4:8] >> 6 << 4)], 1)
    return sc.double(), mn.double()


def _bits(b, n=8):
    return (b.to(torch.int32).unsqueeze(-1) >> torch.arange(n, device=b.device, dtype=torch.int32)) & 1


def _signs7(idx):
    """Signs of the 7-bit sign index: its bits, and an eighth that makes the count of minus signs even."""
    s = _bits(idx, 7)
    return 1.0 - 2.0 * torch.cat([s, s.sum(-1, keepdim=True) & 1], -1).double()


def _dequant(ty, q):
    """Blocks q (n, bytes) to values (n, values), in 64 bits."""
    n = q.shape[0]
    if ty in ("Q4_0", "Q8_0"):
        d = _f16(q[:, :2])
        if ty == "Q8_0":
            return d * q[:, 2:].contiguous().view(torch.int8).double()
        return d * (torch.cat([q[:, 2:] & 15, q[:, 2:] >> 4], 1).double() - 8.0)
    if ty in ("Q4_K", "Q5_K"):
        d, dm = _f16(q[:, 0:2]), _f16(q[:, 2:4])
        sc, mn = _k4(q[:, 4:16])
        qs = q[:, -128:].reshape(n, 4, 32)
        v = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if ty == "Q5_K":
            v = v + (_bits(q[:, 16:48]).transpose(1, 2).to(torch.uint8) << 4)
        return ((d * sc).unsqueeze(-1) * v.double() - (dm * mn).unsqueeze(-1)).reshape(n, 256)
    if ty == "Q6_K":
        ql, qh = q[:, :128].reshape(n, 2, 2, 32), q[:, 128:192].reshape(n, 2, 32)
        v = torch.stack([(ql[:, :, j & 1] >> (4 * (j >> 1)) & 15) | (qh >> (2 * j) & 3) << 4 for j in range(4)], 2)
        sc = q[:, 192:208].contiguous().view(torch.int8).double()
        return ((_f16(q[:, 208:210]) * sc).unsqueeze(-1) * (v.reshape(n, 16, 16).double() - 32.0)).reshape(n, 256)
    if ty == "Q3_K":
        hm, qs, s = q[:, :32], q[:, 32:96].reshape(n, 2, 32), q[:, 96:108].to(torch.int16)
        lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        hi = torch.cat([s[:, 8:12] >> (2 * j) & 3 for j in range(4)], 1)
        sc = (lo | hi << 4).double() - 32.0
        v = torch.stack([qs >> (2 * j) & 3 for j in range(4)], 2).reshape(n, 8, 32).double() - 4.0 * (1 - _bits(hm).transpose(1, 2)).double()
        return ((_f16(q[:, 108:110]) * sc).unsqueeze(-1) * v.reshape(n, 16, 16)).reshape(n, 256)
    d = _f16(q[:, :2])
    if ty == "IQ2_S":
        qh = q[:, 66:74].to(torch.int64)
        hi = torch.stack([qh << (8 - 2 * j) & 0x300 for j in range(4)], -1).reshape(n, 32)
        g = _grid(IQ2_S, [8, 25, 43], 8, q.device)[q[:, 2:34].long() | hi]
        s = 1.0 - 2.0 * _bits(q[:, 34:66]).double()
        sc = torch.stack([q[:, 74:82] & 15, q[:, 74:82] >> 4], -1).reshape(n, 16).double()
        return ((d * (0.5 + sc) * 0.25).unsqueeze(-1) * (g * s).reshape(n, 16, 16)).reshape(n, 256)
    if ty == "IQ2_XXS":
        r = q[:, 2:].reshape(n, 8, 8)
        g = _grid(IQ2_XXS, [8, 25, 43], 8, q.device)[r[:, :, :4].long()]
        aux, step = r[:, :, 4:].contiguous().view(torch.int32), 0.25
    else:
        g = _grid(IQ3_XXS, [4, 12, 20, 28, 36, 44, 52, 62], 4, q.device)[q[:, 2:66].long()].reshape(n, 8, 4, 8)
        aux, step = q[:, 66:].reshape(n, 8, 4).contiguous().view(torch.int32), 0.5
    aux = aux.reshape(n, 8).long() & 0xFFFFFFFF
    s = _signs7(torch.stack([aux >> (7 * j) & 127 for j in range(4)], -1))
    return ((d * (0.5 + (aux >> 28).double()) * step).reshape(n, 8, 1, 1) * (g * s)).reshape(n, 256)


def _times(ty, w, rows, cols, x):
    """x . W^T in 64 bits for x (tokens, cols), some rows of W at a time."""
    v, bb = BLOCK[ty]
    q = w.reshape(rows, cols // v, bb)
    step = max(1, (16 << 20) // cols)
    return torch.cat([x @ _dequant(ty, q[r:r + step].reshape(-1, bb)).reshape(-1, cols).T for r in range(0, rows, step)], 1)


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _q8(x):
    """x after the int8 quantization per 32 values."""
    v = x.reshape(-1, 32)
    d = v.abs().amax(1, keepdim=True) / 127.0
    return (torch.round(torch.where(d > 0, v / d, torch.zeros_like(v))) * d).reshape(x.shape)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "matmul":
        return _times(case["ty"], s["w"], case["rows"], case["cols"], s["x"].double())
    if kind == "dequant":
        v, bb = BLOCK[case["ty"]]
        return _dequant(case["ty"], s["w"].reshape(-1, bb)).reshape(case["rows"], case["cols"])
    out = []
    if kind == "moe":
        e, k, h, ff = case["n_exp"], case["k"], case["hidden"], case["ff"]
        tg, td = case["ty_gate"], case["ty_down"]
        for lay in s["layers"]:
            p, idx = torch.softmax(lay["logits"].double(), -1).topk(k, -1)
            wt = p / p.sum(-1, keepdim=True)
            x, y = lay["x"].double(), torch.zeros(case["tokens"], h, dtype=torch.float64, device="cuda")
            gate, up, down = (lay[n].reshape(e, -1) for n in ("gate", "up", "down"))
            for i in range(e):
                t, j = (idx == i).nonzero(as_tuple=True)
                if t.numel():
                    a = _silu_mul(_times(tg, gate[i], ff, h, x[t]), _times(tg, up[i], ff, h, x[t]))
                    y.index_add_(0, t, wt[t, j].unsqueeze(1) * _times(td, down[i], h, ff, a))
            out.append({"out": y, "idx": idx.to(torch.int32), "wt": wt})
        return out
    mats = {n: (t, r, c) for n, t, r, c in _mats(case)}
    for lay in s["layers"]:
        x = {n: lay["x_" + n].double() for n in ("attn", "o", "ffn")}
        nx = {}
        if kind == "int8":
            nx = {"n_" + n: _norm(x[n], w.double()).reshape(-1) for n, w in zip(("attn", "ffn"), lay["norm"])}
            x = {"attn": _q8(nx["n_attn"]).reshape(1, -1), "o": _q8(x["o"]), "ffn": _q8(nx["n_ffn"]).reshape(1, -1)}
        y = {n: _times(t, lay["w"][n], r, c, x["attn" if n in "qkv" else "o" if n == "o" else "ffn"]) for n, (t, r, c) in mats.items() if n != "down"}
        if "x_down" in lay:
            xd = lay["x_down"].double()
            xd = _q8(xd) if kind == "int8" else xd
        else:
            xd = _silu_mul(*y["gate_up"].chunk(2, -1))
        y["down"] = _times(mats["down"][0], lay["w"]["down"], mats["down"][1], mats["down"][2], xd)
        if case["tokens"] == 1:
            y["qkv"] = torch.cat([y.pop(n) for n in "qkv"], 1)
            y = {n: v.reshape(-1) for n, v in y.items()}
        out.append({**y, **nx, "q8": None} if kind == "int8" else y)
    return out
