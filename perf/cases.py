"""What the speed of this package is judged by: one call of a public operator, as an inference program makes it.

The operators are the ones a program runs while it serves a weight-quantised model: the GPTQ 3-bit product at batch
1 (decode of one sequence), at small batches (decode of several) and with a prompt's tokens as rows (prefill); 4-bit
weights expanded and made (NF4 / FP4 dequantisation and quantisation); the 8-bit dynamic-map quantiser; the LUT-GEMM
and AQLM matrix-vector products; the int8 activation quantisers; the dense and integer gemv; the microscaling fp4
round trip.  Operators that a program runs once per model (the weight packers) are not here.

listed() holds the shapes of the benchmark and of the tests, from the smallest call to the largest; draw() gives
other sizes, types and options of the same operators.  Sizes follow what the operators accept; where any size is
accepted, odd ones are among them.
"""
import math

import torch

import hecbench_amd as hq

F16, F32, BF16, I8, U8, I16, I32 = (torch.float16, torch.float32, torch.bfloat16, torch.int8, torch.uint8, torch.int16,
                                    torch.int32)
FLOATS = {"f16": F16, "f32": F32, "bf16": BF16}
SIZE = {"f16": 2, "f32": 4, "bf16": 2}

# the largest product of M, K and N of a batched 3-bit product, and the most elements of a streaming operator
GEMM_MOST = 1021 * 8192 * 28672
STREAM_MOST = 1 << 27


def listed():
    return [
        # the smallest product: a narrow layer of a small model, one token; launch and call overhead count
        {"name": "q3_decode_1024x512", "op": "q3_matvec", "K": 1024, "N": 512, "x": "f32"},
        # one token through a feed-forward layer: the benchmark's headline shape, fp16 activations
        {"name": "q3_decode_4096x11008", "op": "q3_matvec", "K": 4096, "N": 11008, "x": "f16"},
        # 64 sequences decoded together through a wide layer
        {"name": "q3_batch64_8192x28672", "op": "q3_gemm", "M": 64, "K": 8192, "N": 28672},
        # a prompt's tokens through the same layer; a prompt has any length
        {"name": "q3_prefill1021_8192x28672", "op": "q3_gemm", "M": 1021, "K": 8192, "N": 28672},
        # a 4-bit weight matrix expanded for a dense product
        {"name": "nf4_dequant_4096x4096", "op": "nf4_dequant", "n": 4096 * 4096, "blocksize": 64, "table": 0},
        # a layer's fp16 weights quantised on load
        {"name": "nf4_quantize_4096x11008", "op": "nf4_quantize", "n": 4096 * 11008, "blocksize": 64, "table": 0,
         "x": "f16"},
        # an optimizer state or tensor of any length quantised to the dynamic 8-bit map
        {"name": "dynamic8_10000019", "op": "dynamic8", "n": 10000019},
        # one token through a binary-coded layer of three planes
        {"name": "lut_4096x16384_q3", "op": "lut", "K": 4096, "N": 16384, "bits": 3, "group": 128, "bias": True},
        # one token through a code-book layer
        {"name": "aqlm_4096x4096", "op": "aqlm", "M": 4096, "K": 4096, "books": 1},
        # a prefill's activations quantised per token with zero point, at a hidden size that is no multiple of anything
        {"name": "int8_dynamic_azp_4096x5137", "op": "int8_dynamic", "tokens": 4096, "hidden": 5137, "x": "bf16",
         "azp": True},
        # one token through a 4-bit integer layer
        {"name": "gemv_int4_16384x16384", "op": "gemv_int4", "rows": 16384, "n": 16384},
        # an activation or weight tensor rounded to microscaling fp4
        {"name": "mxfp4_4096x4096", "op": "mxfp4", "n": 4096 * 4096, "x": "bf16"},
    ]


def _between(rng, lo, hi, step=1):
    """A multiple of step from lo to hi, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    op = rng.choice(["q3_matvec", "q3_batch", "q3_prefill", "nf4_dequant", "nf4_quantize", "dynamic8", "lut", "aqlm",
                     "int8_dynamic", "int8_static", "gemv_fp16", "gemv_int8", "gemv_int4", "mxfp4"])
    if op == "q3_matvec":
        return {"op": op, "K": _between(rng, 512, 49152, 32), "N": _between(rng, 128, 28672, 4),
                "x": rng.choice(["f16", "f32"])}
    if op == "q3_batch":
        return {"op": "q3_gemm", "M": _between(rng, 2, 64), "K": _between(rng, 1024, 16384, 32),
                "N": _between(rng, 512, 28672, 4)}
    if op == "q3_prefill":
        M, K = _between(rng, 65, 2048), _between(rng, 1024, 8192, 32)
        return {"op": "q3_gemm", "M": M, "K": K, "N": _between(rng, 512, min(28672, GEMM_MOST // (M * K)), 4)}
    if op in ("nf4_dequant", "nf4_quantize"):
        c = {"op": op, "n": _between(rng, 4096, STREAM_MOST), "blocksize": rng.choice([32, 64, 128, 256, 1024, 4096]),
             "table": rng.choice([0, 1])}
        if op == "nf4_quantize":
            c["x"] = rng.choice(["f16", "f32"])
        return c
    if op == "dynamic8":
        return {"op": op, "n": _between(rng, 4096, STREAM_MOST)}
    if op == "lut":
        group = rng.choice([32, 64, 128, 128, 256])
        return {"op": op, "K": _between(rng, 1024, 16384, max(group, 128)), "N": _between(rng, 512, 28672),
                "bits": rng.choice([1, 2, 3, 3, 4]), "group": group, "bias": rng.choice([True, True, False])}
    if op == "aqlm":
        return {"op": op, "M": _between(rng, 512, 28672), "K": _between(rng, 1024, 16384, 64), "books": rng.choice([1, 1, 3])}
    if op in ("int8_dynamic", "int8_static"):
        hidden = _between(rng, 128, 16384)
        return {"op": op, "tokens": _between(rng, 1, min(8192, STREAM_MOST // hidden)), "hidden": hidden,
                "x": rng.choice(["f16", "bf16", "f32"]), "azp": rng.choice([True, False])}
    if op.startswith("gemv"):
        return {"op": op, "rows": _between(rng, 512, 28672), "n": _between(rng, 512, 16384, 32)}
    return {"op": op, "n": _between(rng, 4096, STREAM_MOST, 32), "x": rng.choice(["f16", "bf16"])}


def prepare(case, seed):
    hq.init()
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def normal(*shape, dtype=F32, scale=1.0):
        t = torch.empty(shape, dtype=dtype, device=dev).normal_(generator=g)
        return t.mul_(scale) if scale != 1.0 else t

    def bits(*shape, dtype):
        lo, hi = (0, 256) if dtype == U8 else (torch.iinfo(dtype).min, torch.iinfo(dtype).max + 1)
        return torch.randint(lo, hi, shape, dtype=dtype, device=dev, generator=g)

    s, op = dict(case), case["op"]
    if op in ("q3_matvec", "q3_gemm"):
        K, N = s["K"], s["N"]
        s["qweight"] = bits(3 * K // 32, N, dtype=I32)  # every 96-bit string is 32 codes
        s["scales"] = torch.rand(N, device=dev, generator=g).mul_(0.01).add_(0.002)
        s["zeros"] = s["scales"] * torch.randint(2, 6, (N,), device=dev, generator=g)
        s["in"] = normal(K, dtype=FLOATS[s["x"]]) if op == "q3_matvec" else normal(s["M"], K, dtype=F16)
    elif op == "nf4_dequant":
        s["packed"] = bits((s["n"] + 1) // 2, dtype=U8)
        s["absmax"] = torch.rand(-(-s["n"] // s["blocksize"]), device=dev, generator=g).mul_(0.2).add_(0.01)
    elif op == "nf4_quantize":
        s["in"] = normal(s["n"], dtype=FLOATS[s["x"]], scale=0.02)
    elif op == "dynamic8":
        s["code"] = hq.dynamic_map().to(dev)
        s["in"] = normal(s["n"], scale=0.2)
    elif op == "lut":
        K, N, nb, G = s["K"], s["N"], s["bits"], s["group"]
        s["bW"] = bits(K // 32, nb, N, dtype=I32)
        s["alpha"] = torch.rand(K // G, nb, N, device=dev, generator=g).mul_(0.02).add_(0.001).half()
        s["q_bias"] = normal(K // G, N, dtype=F16, scale=0.01) if s["bias"] else None
        s["in"] = normal(K, dtype=F16)
    elif op == "aqlm":
        M, K, nb = s["M"], s["K"], s["books"]
        s["codes"] = bits(M, K // 8, dtype=I16)
        s["codebooks"] = normal(nb, 65536, 8, dtype=F16, scale=0.1)
        s["bounds"] = [M] * 4 if nb == 1 else [M // 3, 2 * (M // 3), M, M]
        s["scales"] = torch.rand(M, device=dev, generator=g).mul_(0.1).add_(0.05).half()
        s["in"] = normal(K, dtype=F16)
    elif op in ("int8_dynamic", "int8_static"):
        s["in"] = normal(s["tokens"], s["hidden"], dtype=FLOATS[s["x"]])
    elif op.startswith("gemv"):
        rows, n = s["rows"], s["n"]
        s["mat"] = (normal(rows, n, dtype=F16, scale=0.02) if op == "gemv_fp16" else
                    bits(rows, n, dtype=I8) if op == "gemv_int8" else bits(rows, n // 2, dtype=U8))
        s["in"] = normal(n, dtype=F16)
    else:
        s["in"] = normal(s["n"], dtype=FLOATS[s["x"]])
    return s


def run(s):
    op = s["op"]
    if op == "q3_matvec":
        return hq.q3_matvec(s["in"], s["qweight"], s["scales"], s["zeros"])
    if op == "q3_gemm":
        return hq.q3_gemm(s["in"], s["qweight"], s["scales"], s["zeros"])
    if op == "nf4_dequant":
        return hq.dequant_4bit(s["packed"], s["absmax"], s["n"], s["blocksize"], s["table"])
    if op == "nf4_quantize":
        return hq.quantize_4bit(s["in"], s["blocksize"], s["table"])
    if op == "dynamic8":
        return hq.quantize_dynamic8(s["code"], s["in"])
    if op == "lut":
        return hq.lut_matmul(s["in"], s["bW"], s["alpha"], s["q_bias"], s["group"])
    if op == "aqlm":
        return hq.code1x16_matvec(s["codes"], s["in"], s["codebooks"], s["bounds"], 65536, s["scales"])
    if op == "int8_dynamic":
        return hq.dynamic_scaled_int8_quant(s["in"], s["azp"])
    if op == "int8_static":
        return hq.static_scaled_int8_quant(s["in"], 0.03, 7 if s["azp"] else None)
    if op == "gemv_fp16":
        return hq.gemv_fp16(s["mat"], s["in"])
    if op == "gemv_int8":
        return hq.gemv_int8(s["mat"], s["in"], 0.01, 3.0)
    if op == "gemv_int4":
        return hq.gemv_int4(s["mat"], s["in"], 0.05, 8.0)
    return hq.mxfp4_qdq(s["in"])


def work(c):
    op, flops = c["op"], 0
    if op in ("q3_matvec", "q3_gemm"):
        M, K, N = c.get("M", 1), c["K"], c["N"]
        moved = 3 * K * N // 8 + 8 * N + M * K * SIZE[c.get("x", "f16")] + 4 * M * N
        flops = 2 * M * K * N
    elif op == "nf4_dequant":
        moved = c["n"] // 2 + 4 * (c["n"] // c["blocksize"]) + 2 * c["n"]
    elif op == "nf4_quantize":
        moved = c["n"] // 2 + 4 * (c["n"] // c["blocksize"]) + SIZE[c["x"]] * c["n"]
    elif op == "dynamic8":
        moved = 5 * c["n"] + 1024
    elif op == "lut":
        K, N, nb, G = c["K"], c["N"], c["bits"], c["group"]
        moved = K * N * nb // 8 + 2 * (K // G) * N * (nb + (1 if c["bias"] else 0)) + 2 * K + 2 * N
        flops = 2 * K * N * nb
    elif op == "aqlm":
        M, K = c["M"], c["K"]
        moved = 2 * M * (K // 8) + c["books"] * (1 << 20) + 2 * K + 4 * M
        flops = 2 * M * K
    elif op in ("int8_dynamic", "int8_static"):
        moved = c["tokens"] * c["hidden"] * (SIZE[c["x"]] + 1)
        if op == "int8_dynamic":
            moved += c["tokens"] * (8 if c["azp"] else 4)
    elif op.startswith("gemv"):
        moved = int(c["rows"] * c["n"] * {"gemv_fp16": 2, "gemv_int8": 1, "gemv_int4": 0.5}[op]) + 2 * c["n"] + 2 * c["rows"]
        flops = 2 * c["rows"] * c["n"]
    else:
        moved = 4 * c["n"]
    return {"bytes": moved, "flops": flops}


def tolerance(c):
    op = c["op"]
    if op in ("q3_matvec", "q3_gemm"):
        # fp32 results of sums over K fp16 or fp32 activations; a matrix core's fp32 accumulation rounds every
        # partial sum, over a long K by a few 1e-5 of the result
        return {"rel": 2e-5 if op == "q3_matvec" else 1e-4}
    if op in ("lut", "aqlm") or op.startswith("gemv"):
        return {"rel": 1e-3}  # fp32 sums, one rounding to fp16 (half a unit in the last place is 4.9e-4)
    return "exact"  # codes, scales and once-rounded products: every correct implementation gives the same
