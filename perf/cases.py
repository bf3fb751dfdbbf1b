"""What is timed when the speed of this backend is judged: the calls a host interpreter or a serving loop makes of it,
over the range of sizes, types and options they are made with.

A case is a dict of plain values; `kind` names the entry point:

  a16    one tpu.A16MatMul on device tensors (a16mm_launch), 4- or 8-bit weights: decode (few rows) and prefill (many)
  block  a decoder block as a device-resident op list: float32 in through set_tensor, invoke, float32 out of every
         output through get_tensor, the calling convention of the interpreter classes
  i8     one quantized tpu.MatMul with requantization on device tensors (i8mm_launch)
  mlp    a quantized two-layer perceptron on device tensors: Cast to int8, MatMul + ReLU, MatMul, Cast back
  dyn    tpu.A16MatMul with dynamic activation quantization (a16mm_dq_launch)
  dyn2   tpu.MatMul of two activations, both quantized dynamically (matmul_dq_launch)
  f8     tpu.MatMul on 8-bit-float codes with output requantization (f8mm_launch)
  op     tpu.A16MatMul through the operator boundary: float32 host tensors in and out (A16MatMul.inference)
"""
import importlib

import numpy as np
import torch

amd = importlib.import_module("tpu-mlir_amd")
clib = importlib.import_module("tpu-mlir_amd.clib")


def listed():
    return [
        # one projection for one token: the smallest call there is, launch and host cost against 7 MB of weights
        dict(name="w4_decode_1x2048x6144", kind="a16", bits=4, M=1, K=2048, N=6144, g=64, f16=False),
        # a Llama-7B decoder block for one token, activations resident, the interpreter's float32 view at both ends
        dict(name="w4_block_decode_1", kind="block", M=1, hidden=4096, mlp=11008, g=128),
        # an MLP up-projection for a batch of 32 tokens, 8-bit weights with one scale per channel
        dict(name="w8_decode_32x4096x11008", kind="a16", bits=8, M=32, K=4096, N=11008, g=0, f16=False),
        # a projection while a prompt of 2048 tokens is read
        dict(name="w4_prefill_2048x4096x4096", kind="a16", bits=4, M=2048, K=4096, N=4096, g=128, f16=False),
        # a prompt of odd length through a grouped 8-bit up-projection, F16 mode
        dict(name="w8_prefill_777x4096x11008", kind="a16", bits=8, M=777, K=4096, N=11008, g=64, f16=True),
        # a small quantized layer: int8 in and out, per-channel requantization
        dict(name="i8_256x1024x1024", kind="i8", M=256, K=1024, N=1024, rt=True, unsigned=False, per_channel=True),
        # the largest quantized product
        dict(name="i8_4096x4096x4096", kind="i8", M=4096, K=4096, N=4096, rt=True, unsigned=False, per_channel=True),
        # a quantized perceptron of ragged sizes, weights [K, N] as tpu.MatMul stores them, asymmetric middle activation
        dict(name="i8_mlp_333x1000x3000", kind="mlp", M=333, hidden=1000, mlp=3000),
        # a prompt of 512 tokens through a projection with dynamically quantized activations
        dict(name="dyn_prefill_512x4096x4096", kind="dyn", bits=4, dq="INT", M=512, K=4096, N=4096, g=128),
        # attention scores of 2048 positions by 2048, 128 wide, both sides quantized dynamically
        dict(name="dyn2_scores_2048x128x2048", kind="dyn2", dq="INT8", M=2048, K=128, N=2048, g=64, rt=True),
        # the largest 8-bit-float product, per-channel output scales
        dict(name="f8_4096x4096x4096", kind="f8", M=4096, K=4096, N=4096, rt=True, per_channel=True),
        # what an interpreter that keeps its tensors as host floats pays for a 128-token projection
        dict(name="op_128x4096x4096", kind="op", M=128, K=4096, N=4096, g=128),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step, spread over the logarithm of [lo, hi]."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def _fits(c):
    w = work(c)
    return w["flops"] <= 137.5e9 and w["bytes"] <= 120e6


def draw(rng):
    while True:
        c = _draw(rng)
        if _fits(c):
            return c


def _draw(rng):
    kind = rng.choice(["a16", "a16", "a16", "a16", "block", "i8", "i8", "mlp", "dyn", "dyn2", "f8", "op"])
    if kind == "a16":
        bits = rng.choice([4, 4, 8])
        g = rng.choice([32, 64, 128, 128]) if bits == 4 else rng.choice([0, 0, 64, 128])
        return dict(kind=kind, bits=bits, M=_log(rng, 1, 2048), K=_log(rng, 1024, 11008, g or 64),
                    N=_log(rng, 512, 11008), g=g, f16=rng.random() < 0.3)
    if kind == "block":
        h = _log(rng, 1024, 4096, 128)
        return dict(kind=kind, M=_log(rng, 1, 32), hidden=h, mlp=int(h * rng.uniform(2.0, 2.7)) // 128 * 128, g=128)
    if kind == "i8":
        return dict(kind=kind, M=_log(rng, 1, 4096), K=_log(rng, 256, 8192), N=_log(rng, 256, 8192),
                    rt=rng.random() < 0.5, unsigned=rng.random() < 0.3, per_channel=rng.random() < 0.7)
    if kind == "mlp":
        h = _log(rng, 200, 2048)
        return dict(kind=kind, M=_log(rng, 16, 2048), hidden=h, mlp=h * rng.choice([2, 3, 4]))
    if kind == "dyn":
        bits, dq = rng.choice([(4, "INT"), (4, "INT"), (8, "INT"), (4, "F4"), (8, "F8E4M3")])
        return dict(kind=kind, bits=bits, dq=dq, M=_log(rng, 1, 1024), K=_log(rng, 1024, 8192, 128),
                    N=_log(rng, 512, 8192), g=rng.choice([64, 128, 128]))
    if kind == "dyn2":
        return dict(kind=kind, dq=rng.choice(["INT8", "INT8", "INT4"]), M=_log(rng, 16, 2048),
                    K=rng.choice([64, 128, 128, 256, 512, 1024]), N=_log(rng, 16, 2048), g=rng.choice([32, 64]),
                    rt=rng.random() < 0.6)
    if kind == "f8":
        return dict(kind=kind, M=_log(rng, 1, 4096), K=_log(rng, 256, 8192, 16), N=_log(rng, 256, 8192),
                    rt=rng.random() < 0.7, per_channel=rng.random() < 0.7)
    return dict(kind=kind, M=_log(rng, 1, 512), K=_log(rng, 1024, 4096, 128), N=_log(rng, 512, 4096), g=128)


# ---- inputs -----------------------------------------------------------------------------------------------------
def _f16_bits(a, f16):
    """Non-negative float32 values as bf16 or f16 bit patterns."""
    if f16:
        return a.astype(np.float16).view(np.uint16)
    return torch.from_numpy(a).bfloat16().view(torch.int16).numpy().view(np.uint16)


def _a16_arrays(rng, bits, K, N, g, f16, dq="INT"):
    """Packed weights with every code drawn evenly, scales |N(0, .01)| (4-bit) / |N(0, .005)| (8-bit), one zero point a
    group: what a converted checkpoint's projection holds."""
    G = K // g if g else 1
    if bits == 4:
        w = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8)
        zp = rng.integers(0, 16, size=(N, G), dtype=np.uint8)
        scale = np.abs(rng.standard_normal((N, G), dtype=np.float32)) * 0.01 + 1e-4
    else:
        w = rng.integers(-127, 128, size=(N, K), dtype=np.int8)
        zp = np.zeros((N, G), dtype=np.uint8)
        scale = np.abs(rng.standard_normal((N, G), dtype=np.float32)) * 0.005 + 1e-5
    if dq == "F8E4M3":
        w = w.view(np.uint8) & np.uint8(0xD7)  # finite codes of moderate size
    if dq != "INT":
        zp[:] = 0  # the producer of float codes writes no zero points
    return w, _f16_bits(scale.astype(np.float32), f16), zp


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _i8(gen, shape, lo=-128, hi=128, dtype=torch.int8):
    return torch.randint(lo, hi, shape, generator=gen, device="cuda", dtype=torch.int32).to(dtype)


def _q31(gen, N, out_dtype, zp=0):
    mult = torch.randint(1 << 30, (1 << 31) - 1, (N,), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    shift = torch.randint(8, 17, (N,), generator=gen, device="cuda", dtype=torch.int32)
    return amd.RequantDesc(clib.RQ_QDM, clib.ROUND_HALF_AWAY_FROM_ZERO, out_dtype=out_dtype, multiplier=mult,
                           shift=shift, zp=zp)


def _bias_i32(gen, N):
    return torch.randint(-65536, 65537, (N,), generator=gen, device="cuda", dtype=torch.int32)


def prepare(case, seed):
    c = case
    rng, gen = np.random.default_rng(int(seed)), _gen(seed)
    kind = c["kind"]
    if kind in ("a16", "dyn"):
        f16 = bool(c.get("f16", False))
        w, scale, zp = _a16_arrays(rng, c["bits"], c["K"], c["N"], c["g"], f16, c.get("dq", "INT"))
        weight = amd.A16Weight(w, scale, zp, None, K=c["K"], N=c["N"], weight_bits=c["bits"], q_group_size=c["g"],
                               dtype=clib.DT_F16 if f16 else clib.DT_BF16)
        x = torch.randn((c["M"], c["K"]), generator=gen, device="cuda").to(torch.float16 if f16 else torch.bfloat16)
        return dict(kind=kind, w=weight, x=x, dq={"INT": clib.DQ_INT, "F4": clib.DQ_F4, "F8E4M3": clib.DQ_F8E4M3}[c.get("dq", "INT")])
    if kind == "block":
        M, h, f = c["M"], c["hidden"], c["mlp"]
        m = amd.Module()
        m.add_tensor("x", clib.ST_F32, (M, h)).add_tensor("xb", clib.ST_BF16, (M, h))
        chain = [("q", "xb", h, h), ("k", "xb", h, h), ("v", "xb", h, h), ("o", "q", h, h), ("gate", "o", h, f),
                 ("up", "o", h, f), ("down", "gate", f, h)]
        for name, _, _, n in chain:
            m.add_tensor(name, clib.ST_BF16, (M, n))
        m.add_cast("x", "xb", in_type=clib.ST_F32, out_type=clib.ST_BF16)
        for name, src, k, n in chain:
            m.add_a16matmul(src, name, *_a16_arrays(rng, 4, k, n, c["g"], False), None, K=k, N=n, weight_bits=4,
                            q_group_size=c["g"])
        return dict(kind=kind, m=m, x=rng.standard_normal((M, h), dtype=np.float32))
    if kind == "i8":
        M, K, N = c["M"], c["K"], c["N"]
        a = _i8(gen, (M, K), 0, 256, torch.uint8) if c["unsigned"] else _i8(gen, (M, K))
        b = _i8(gen, (N, K) if c["rt"] else (K, N))
        if c["per_channel"]:
            rq = _q31(gen, N, clib.DT_I8)
        else:  # one multiplier and shift for the whole tensor (outputs of about 40 steps), an output zero point
            rq = amd.RequantDesc(clib.RQ_MULTIPLIER_SHIFT, clib.ROUND_HALF_UP, out_dtype=clib.DT_I8,
                                 multiplier=int(rng.uniform(0.8, 1.25) * 40 * 2 ** 20 / (74 * 74 * K ** 0.5)), shift=20,
                                 zp=-3)
        return dict(kind=kind, a=a, b=b, bias=_bias_i32(gen, N), rq=rq, rt=c["rt"], zp=117 if c["unsigned"] else 0)
    if kind == "mlp":
        M, h, f = c["M"], c["hidden"], c["mlp"]
        return dict(kind=kind, x=torch.randn((M, h), generator=gen, device="cuda"), b1=_i8(gen, (h, f)), b2=_i8(gen, (f, h)),
                    bias1=_bias_i32(gen, f), bias2=_bias_i32(gen, h), rq1=_q31(gen, f, clib.DT_U8, zp=9), zp1=9,
                    rq2=_q31(gen, h, clib.DT_I8))
    if kind == "dyn2":
        left = torch.randn((c["M"], c["K"]), generator=gen, device="cuda").bfloat16()
        right = torch.randn((c["N"], c["K"]) if c["rt"] else (c["K"], c["N"]), generator=gen, device="cuda").bfloat16()
        return dict(kind=kind, left=left, right=right, rt=c["rt"], g=c["g"], dq={"INT8": clib.DQ_INT8, "INT4": clib.DQ_INT4}[c["dq"]])
    if kind == "f8":
        M, K, N = c["M"], c["K"], c["N"]
        a = torch.randn((M, K), generator=gen, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
        b = torch.randn((N, K) if c["rt"] else (K, N), generator=gen, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
        bias = torch.randn(N, generator=gen, device="cuda")
        scales = torch.rand(N, generator=gen, device="cuda", dtype=torch.float64) * 1.5 + 0.5 if c["per_channel"] else None
        return dict(kind=kind, a=a, b=b, bias=bias, scales=scales, rt=c["rt"])
    # op: the interpreter's float tensors; init is its one-time call
    w, scale, zp = _a16_arrays(rng, 4, c["K"], c["N"], c["g"], False)
    op = amd.A16MatMul(c["K"], c["N"], 4, c["g"]).init(w, (scale.astype(np.uint32) << 16).view(np.float32), zp)
    x = torch.from_numpy(rng.standard_normal((c["M"], c["K"]), dtype=np.float32)).bfloat16().float().numpy()
    return dict(kind=kind, op=op, x=x)


# ---- one pass ---------------------------------------------------------------------------------------------------
def run(state):
    s = state
    kind = s["kind"]
    if kind == "a16":
        return amd.a16mm_launch(s["w"], s["x"])
    if kind == "block":
        m = s["m"]
        m.set_tensor("x", s["x"])
        m.invoke()
        return {name: m.get_tensor(name) for name in m.output_names}
    if kind == "i8":
        return amd.i8mm_launch(s["a"], s["b"], s["bias"], right_transpose=s["rt"], input_zp=s["zp"], rq=s["rq"])
    if kind == "mlp":
        a = amd.cast_launch(s["x"], in_type=clib.ST_F32, out_type=clib.ST_I8, out_quant=True, scale=0.03)
        a = amd.i8mm_launch(a, s["b1"], s["bias1"], do_relu=True, rq=s["rq1"])
        a = amd.i8mm_launch(a, s["b2"], s["bias2"], input_zp=s["zp1"], rq=s["rq2"])
        return a, amd.cast_launch(a, in_type=clib.ST_I8, out_type=clib.ST_F32, in_quant=True, scale=0.05)
    if kind == "dyn":
        return amd.a16mm_dq_launch(s["w"], s["x"], dq_type=s["dq"])
    if kind == "dyn2":
        return amd.matmul_dq_launch(s["left"], s["right"], right_transpose=s["rt"], q_group_size=s["g"], dq_type=s["dq"])
    if kind == "f8":
        if s["scales"] is None:
            return amd.f8mm_launch(s["a"], s["b"], s["bias"], right_transpose=s["rt"], out_scale=1.25)
        return amd.f8mm_launch(s["a"], s["b"], s["bias"], right_transpose=s["rt"], out_scales=s["scales"])
    return s["op"].inference(s["x"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------
def _a16_work(bits, M, K, N, g, in_bytes=2, out_bytes=2):
    G = K // g if g else 1
    return N * K * bits // 8 + N * G * 3 + M * K * in_bytes + M * N * out_bytes, 2 * M * K * N


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("a16", "dyn"):
        b, f = _a16_work(c["bits"], c["M"], c["K"], c["N"], c["g"])
    elif kind == "op":
        b, f = _a16_work(4, c["M"], c["K"], c["N"], c["g"], 4, 4)
    elif kind == "block":
        M, h, m, g = c["M"], c["hidden"], c["mlp"], c["g"]
        parts = [_a16_work(4, M, h, h, g)] * 4 + [_a16_work(4, M, h, m, g)] * 2 + [_a16_work(4, M, m, h, g)]
        b, f = sum(p[0] for p in parts) + 4 * M * h, sum(p[1] for p in parts)
    elif kind == "mlp":
        M, h, m = c["M"], c["hidden"], c["mlp"]
        b, f = 4 * M * h + 2 * h * m + 12 * (h + m) + M * h + 4 * M * h, 4 * M * h * m
    elif kind == "dyn2":
        b, f = 2 * (c["M"] * c["K"] + c["N"] * c["K"] + c["M"] * c["N"]), 2 * c["M"] * c["K"] * c["N"]
    else:  # i8, f8: operands and output one byte an element, 12 bytes of parameters a channel
        b, f = c["M"] * c["K"] + c["K"] * c["N"] + c["M"] * c["N"] + 12 * c["N"], 2 * c["M"] * c["K"] * c["N"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Integer results, and the dynamic integer flavours whose fp32 additions have a stated order, are exact.  The rest
    accumulate in fp32 in an order of the implementation's choosing before they round, so that a sum next to a rounding
    boundary moves by one step.  Seen against float64 sums rounded once: 16-bit outputs 4e-5 relative (one step, 0.0078
    of a value, on 5 outputs in 10000; a single step among 512 outputs is 1.7e-4), the block's chain of three matmuls
    4.6e-4, 8-bit-float codes 0.001 of the values; four times these are stated."""
    kind = case["kind"]
    if kind in ("i8", "mlp", "dyn2") or (kind == "dyn" and case["dq"] != "F8E4M3"):
        return "exact"
    if kind == "f8":
        return {"rel": 0.0, "differ": 0.004}
    return {"rel": 2e-3 if kind == "block" else 6e-4, "max": 0.03}
