"""Performance cases of the fully-connected path: what a model server or a model loader calls, through the public operators.

Every case is one call of one operator on tensors that are on the GPU already.  The sizes are those of the benchmark, of
the weight-compression and MLP demos and of the shape sweep of the tests, and in-between ones.
"""
import math

import torch

import mm_amx_amd as mx

DEV = "cuda"


def listed():
    return [
        # one small projection, fp32 result: the operator of the torch front end where launches count
        {"name": "linear_256", "kind": "linear", "M": 256, "K": 256, "N": 256},
        # a 7B feed-forward up-projection over a prompt of 1024 tokens, bias and GELU fused
        {"name": "ffn_up_1024", "kind": "fc", "M": 1024, "K": 4096, "N": 11008, "post": "bias_gelu", "out": "bf16"},
        # a classifier-like head on a ragged batch: no size is a multiple of a tile, rows of the result are not aligned
        {"name": "fc_ragged", "kind": "fc", "M": 391, "K": 1000, "N": 3001, "post": "bias", "out": "bf16"},
        # a quantised layer between two others: int8 in, per-channel dequantisation, bias, requantised int8 out
        {"name": "int8_requant_512", "kind": "int8", "M": 512, "K": 4096, "N": 4096, "post": "requant"},
        # prompt processing on int8-compressed weights (the published shape of the weight-compression demo)
        {"name": "w8_prefill_896", "kind": "w8", "M": 896, "K": 2560, "N": 10240},
        # the second operand is new at every call (constB left at its default): packed, then multiplied
        {"name": "fresh_b_32", "kind": "fresh", "M": 32, "K": 10240, "N": 10240, "trans": False},
        # loading a layer: a bf16 weight matrix compressed to int8 and packed
        {"name": "load_int8", "kind": "load", "to": "int8", "K": 4096, "N": 11008},
        # one token on int8-compressed weights
        {"name": "decode_w8_1", "kind": "w8", "M": 1, "K": 4096, "N": 11008},
        # a few sequences at once on int4-compressed weights
        {"name": "decode_w4_4", "kind": "w4", "M": 4, "K": 4096, "N": 11008},
        # the whole MLP of a 7B layer: a decode batch, and a long prompt
        {"name": "mlp_decode_16", "kind": "mlp", "M": 16, "K": 4096, "N": 11008},
        {"name": "mlp_prefill_2048", "kind": "mlp", "M": 2048, "K": 4096, "N": 11008},
        # one query vector against a key cache of 128 per head
        {"name": "qk_matvec", "kind": "matvec", "type": "bf16", "M": 131072, "K": 128},
    ]


def _size(rng, lo, hi, step=1):
    """A size from [lo, hi], even over the logarithm, a multiple of step."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "fc", "fc", "int8", "w8", "w8", "fresh", "load", "w4", "mlp", "mlp", "matvec"])
    if kind == "linear":  # the torch front end takes multiples of 32 only
        return {"kind": kind, "M": _size(rng, 1, 2048), "K": _size(rng, 256, 8192, 32), "N": _size(rng, 256, 8192, 32)}
    if kind == "fc":
        step = rng.choice([64, 64, 64, 8, 1])  # most layers are aligned, some are not
        return {"kind": kind, "M": _size(rng, 1, 2048), "K": _size(rng, 256, 8192, step), "N": _size(rng, 256, 11008, step),
                "post": rng.choice(["none", "bias", "bias_gelu"]), "out": rng.choice(["bf16", "f32"])}
    if kind == "int8":
        return {"kind": kind, "M": _size(rng, 1, 2048), "K": _size(rng, 256, 8192, 64), "N": _size(rng, 256, 11008, 32),
                "post": rng.choice(["requant", "bf16"])}
    if kind == "w8":
        return {"kind": kind, "M": _size(rng, 1, 32) if rng.random() < 0.5 else _size(rng, 33, 2048), "K": _size(rng, 1024, 11008, 64),
                "N": _size(rng, 1024, 16384, 32)}
    if kind == "fresh":
        return {"kind": kind, "M": _size(rng, 1, 1024), "K": _size(rng, 256, 8192, 32), "N": _size(rng, 256, 8192, 32), "trans": rng.random() < 0.5}
    if kind == "load":
        return {"kind": kind, "to": rng.choice(["bf16", "int8", "int8_scaled", "int4"]), "K": _size(rng, 512, 11008, 32), "N": _size(rng, 512, 11008, 32)}
    if kind == "w4":
        return {"kind": kind, "M": _size(rng, 1, 32), "K": _size(rng, 1024, 11008, 64), "N": _size(rng, 1024, 16384, 32)}
    if kind == "mlp":
        return {"kind": kind, "M": _size(rng, 1, 32) if rng.random() < 0.5 else _size(rng, 33, 2048), "K": _size(rng, 1024, 4096, 64),
                "N": _size(rng, 2048, 11008, 64)}
    return {"kind": kind, "type": rng.choice(["bf16", "int8"]), "M": _size(rng, 4096, 1 << 20), "K": rng.choice([64, 96, 128, 256])}


def _rand(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(shape, std=1.0, dtype=torch.bfloat16):
        return torch.randn(shape, device=DEV, generator=g, dtype=torch.float32).mul_(std).to(dtype)

    def int8(shape):
        return torch.randint(-127, 128, shape, device=DEV, generator=g, dtype=torch.int8)

    def uniform(n, lo, hi):
        return torch.rand(n, device=DEV, generator=g) * (hi - lo) + lo

    return normal, int8, uniform


_OUT = {"bf16": torch.bfloat16, "f32": torch.float32, "int8": torch.int8}


def prepare(case, seed):
    kind, K = case["kind"], case["K"]
    M, N = case.get("M", 0), case.get("N", 0)
    normal, int8, uniform = _rand(seed)
    S = mx.Steps
    if kind == "linear":
        lin = mx.LinearNxN()
        lin.set_weight(normal((N, K), 0.02))
        return {"kind": kind, "op": lin, "x": normal((M, K)), "y": torch.empty((M, N), device=DEV)}
    if kind == "load":
        s = {"kind": kind, "to": case["to"], "W": normal((N, K), 0.02) if case["to"] != "int8_scaled" else normal((K, N), 0.02)}
        s["scale"] = 127.0 / 0.1
        return s
    if kind == "matvec":
        new = normal if case["type"] == "bf16" else int8
        return {"kind": kind, "op": mx.MatmulVector(), "x": new((M, K)), "b": new((K,)),
                "y": torch.empty(M, device=DEV, dtype=torch.float32 if case["type"] == "bf16" else torch.int32)}
    if kind == "mlp":
        mlp = mx.MLP()
        mlp.setup(normal((N, K), 0.02), normal((N, K), 0.02), normal((K, N), 0.02))
        return {"kind": kind, "op": mlp, "x": normal((M, K)), "y": torch.empty((M, K), device=DEV, dtype=torch.bfloat16)}
    if kind == "w4":
        packed, deq = mx.quantize_pack_int4(normal((N, K), 0.02), transpose=True)
        y = torch.empty((M, N), device=DEV, dtype=torch.bfloat16)
        return {"kind": kind, "W": packed, "N": N, "x": normal((M, K)), "ep": mx.Epilogue(y, mx.PP_DEQUANT, deq_scale_per_oc=deq), "y": y}
    # what is left goes through Matmul, with the post-op and the result that the layer keeps
    if kind == "int8":
        requant = case["post"] == "requant"
        W, x = int8((K, N)), int8((M, K))
        y = torch.empty((M, N), device=DEV, dtype=torch.int8 if requant else torch.bfloat16)
        pp = mx.BiasGeluStore(y, S.DEQUANT | S.BIAS | (S.QUANT if requant else 0), normal((N,), 0.1, torch.float32))
        pp.set_deq_scale(uniform(N, 1e-3, 1e-2) * (0.02 / math.sqrt(K / 4096)))  # (the products of a longer row are larger)
        if requant:
            pp.set_q_scale(1.0)
        op = mx.Matmul(True, False)
    elif kind == "fc":
        W, x = normal((K, N), 0.02), normal((M, K))
        y = torch.empty((M, N), device=DEV, dtype=_OUT[case["out"]])
        steps = {"none": S.NONE, "bias": S.BIAS, "bias_gelu": S.BIAS_GELU}[case["post"]]
        pp = mx.BiasGeluStore(y, steps, normal((N,), 0.1, torch.float32) if steps else None)
        op = mx.Matmul(True, False)
    elif kind == "w8":
        W, x = normal((K, N), 0.02), normal((M, K))
        y = torch.empty((M, N), device=DEV)
        pp = mx.BiasGeluStore(y, S.DEQUANT)
        op = mx.Matmul(True, False, weight_int8=True)
    else:
        W, x = normal((N, K) if case["trans"] else (K, N), 0.02), normal((M, K))
        y = torch.empty((M, N), device=DEV)
        pp = mx.BiasGeluStore(y)
        op = mx.Matmul(False, case["trans"])
    if kind != "fresh":
        op(x[:1], W, ppkernel=pp)  # a constant second operand is packed at the first call
    return {"kind": kind, "op": op, "x": x, "W": W, "pp": pp, "y": y}


def run(state):
    s, kind = state, state["kind"]
    if kind == "linear":
        s["op"].forward(s["x"], s["y"])
        return s["y"]
    if kind == "load":
        if s["to"] == "int8":
            Wq, scales = mx.quantize_weights(s["W"])
            return mx.repack_b(Wq, transpose=True), scales
        if s["to"] == "int8_scaled":
            return mx.repackB_1xL(s["W"], torch.int8, 2, s["scale"])
        if s["to"] == "int4":
            return mx.quantize_pack_int4(s["W"], transpose=True)
        return mx.repack_b(s["W"], transpose=True)
    if kind == "matvec":
        return s["op"](s["x"], s["b"], s["y"])
    if kind == "mlp":
        return s["op"].run(s["x"], s["y"])
    if kind == "w4":
        mx.gemm(s["x"], s["W"], s["N"], s["ep"], b_dtype=mx.I4)
        return s["y"]
    s["op"](s["x"], s["W"], ppkernel=s["pp"])
    return s["y"]


def work(case):
    kind, K = case["kind"], case["K"]
    M, N = case.get("M", 0), case.get("N", 0)
    if kind == "load":
        out = {"bf16": 2 * K * N, "int8": K * N + 8, "int8_scaled": K * N, "int4": K * N // 2 + 4 * N}[case["to"]]
        return {"bytes": 2 * K * N + out, "flops": 0}
    if kind == "matvec":
        size = 2 if case["type"] == "bf16" else 1
        return {"bytes": (M * K + K) * size + 4 * M, "flops": 2 * M * K}
    if kind == "mlp":
        return {"bytes": 2 * (2 * M * K + 3 * K * N), "flops": 6 * M * K * N}
    x = M * K * (1 if kind == "int8" else 2)
    W = {"int8": K * N, "w8": K * N, "w4": K * N // 2}.get(kind, 2 * K * N)
    y = M * N * {"fc": 2 if case.get("out") == "bf16" else 4, "int8": 1 if case.get("post") == "requant" else 2, "w4": 2}.get(kind, 4)
    columns = 4 * N * {"fc": case.get("post", "none") != "none", "int8": 2, "w4": 1}.get(kind, 0)
    return {"bytes": x + W + y + int(columns), "flops": 2 * M * K * N}


def tolerance(case):
    """Four times what the operators differ from themselves by when K (and the MLP's N) is summed in another order."""
    kind = case["kind"]
    if kind in ("load", "int8") or case.get("type") == "int8":
        return "exact"  # whole numbers, and separately rounded fp32 steps on them
    if kind == "mlp":  # a bf16 intermediate that rounds the other way moves many results a little: 2e-4 .. 5e-4 seen
        return {"rel": 2e-3, "max": 3.2e-2}
    if kind == "w4" or case.get("out") == "bf16":  # single results round the other way (2^-7 of the value): 6e-5, in small results 1e-4
        return {"rel": 4e-4, "max": 3.2e-2}
    if case.get("post") == "bias_gelu":  # the deep negative tail of the GELU polynomial cancels: 5e-6 and 4e-4 seen
        return {"rel": 2.5e-5, "max": 2e-3}
    return {"rel": 1e-6, "max": 1e-5}  # 32-bit sums of up to 11008 products: 2.3e-7 and 1.5e-6 against 64-bit sums
