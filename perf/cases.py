"""The quantized-weight products that a server built on this library spends its time in, as cases to time.

Every case is one call sequence through ``oxydllm_amd.ops`` as an engine makes it: resident layers (AWQ / GPTQ,
GGUF, MXFP4 experts), the gated FFN over them, the stateless ops on checkpoint tensors, the FP8 experts, and a
decode step replayed from a graph.  Sizes are those of ``bench.py``'s configurations (4096 x 4096, 4096 x 14336,
5120 x 13824, experts of 2880 x 2880) and of the tests, with the row counts that decode (1 - 64) and prefill
(hundreds to thousands, seldom round) bring.  Weights are uniform codes with scales ~ U(0.002, 0.02) (GGUF block
scales ~ U(0.001, 0.02), E8M0 exponents in [118, 126]); activations and router logits are N(0, 1).
"""
import math

import torch

from oxydllm_amd import ops, synth

F32, F16, BF16 = "f32", "f16", "bf16"
DTYPES = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}
FORMATS = {"q4_0": synth.GGUF_Q4_0, "q8_0": synth.GGUF_Q8_0, "q4_k": synth.GGUF_Q4_K, "q6_k": synth.GGUF_Q6_K,
           "q4_1": synth.GGUF_Q4_1, "q5_0": synth.GGUF_Q5_0, "q5_1": synth.GGUF_Q5_1, "q2_k": synth.GGUF_Q2_K,
           "q3_k": synth.GGUF_Q3_K, "q5_k": synth.GGUF_Q5_K}
# the largest product a drawn case may hold, in multiply-adds of one weight matrix; the largest listed case has 7e11
MOST_MACS = 6e10


def listed():
    return [
        # one token of one sequence through an attention projection: the smallest call an engine makes
        dict(name="linear_awq4_f16_m1", kind="linear", pack="awq", bits=4, dtype=F16, m=1, k=4096, n=4096, group=128, bias=False),
        # an engine that only swaps the op functions and keeps the checkpoint tensors, four sequences at once
        dict(name="op_awq4_f16_m4", kind="op", pack="awq", bits=4, dtype=F16, m=4, k=4096, n=14336, group=128),
        # the same with an 8-bit GPTQ checkpoint at the largest batch of the decode ops
        dict(name="op_gptq8_f16_m8", kind="op", pack="gptq", bits=8, dtype=F16, m=8, k=5120, n=13824, group=128),
        # a GGUF projection in the 32-bit activations of a CPU-style pipeline
        dict(name="gguf_q4k_f32_m1", kind="gguf", fmt="q4_k", dtype=F32, m=1, k=4096, n=4096),
        # a GGUF down projection at a batch just above one decode tile
        dict(name="gguf_q6k_bf16_m33", kind="gguf", fmt="q6_k", dtype=BF16, m=33, k=14336, n=4096),
        # decoding eight sequences through a mixture-of-experts layer
        dict(name="moe_mxfp4_m8", kind="moe", m=8, hidden=2880, inter=2880, experts=32, top_k=4),
        # a prompt of ragged length through the same layer
        dict(name="moe_mxfp4_m515", kind="moe", m=515, hidden=2880, inter=2880, experts=32, top_k=4),
        # block-scaled FP8 expert weights streamed to a medium batch
        dict(name="f8_bf16_m96", kind="f8", m=96, k=2048, n=5632),
        # a prompt of ragged length through a GPTQ gate / up projection
        dict(name="linear_gptq4_bf16_m777", kind="linear", pack="gptq", bits=4, dtype=BF16, m=777, k=3584, n=18944, group=128, bias=True),
        # the gated FFN for 64 sequences decoding together
        dict(name="ffn_awq4_bf16_m64", kind="ffn", weights="awq4", dtype=BF16, m=64, k=4096, inter=14336),
        # the gated FFN over a long prompt: the largest call
        dict(name="ffn_awq4_bf16_m4096", kind="ffn", weights="awq4", dtype=BF16, m=4096, k=4096, inter=14336),
        # four decoder layers' projections for one token, captured once and replayed as a serving loop does
        dict(name="decode_graph_f16_m1", kind="decode_graph", dtype=F16, m=1, k=4096, qkv=6144, inter=14336, layers=4),
    ]


# ------------------------------------------------------------------ drawn cases
def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))
    return int(min(hi, max(lo, int(v / step) * step)))


def _rows(rng, k, n, most):
    """Rows over the whole range on a log scale, within the work that a drawn case may hold."""
    return _log_int(rng, 1, max(1, min(most, int(MOST_MACS / (k * n)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "op", "gguf", "gguf", "moe", "f8", "ffn", "decode_graph"])
    if kind in ("linear", "op"):
        group = rng.choice([128, 128, 128, 64, 32])
        k = _log_int(rng, 1024, 14336, max(group, 128) if rng.random() < 0.8 else group)
        # columns: whole strips of 64 mostly; a tensor-parallel shard or a padded vocabulary may end elsewhere
        n = _log_int(rng, 512, 28672, 64 if rng.random() < 0.8 else 8)
        c = dict(kind=kind, pack=rng.choice(["awq", "gptq"]), bits=rng.choice([4, 4, 8]), dtype=rng.choice([F16, BF16]),
                 m=_rows(rng, k, n, 4096), k=k, n=n, group=group)
        if kind == "linear":
            c["bias"] = rng.random() < 0.3
        return c
    if kind == "gguf":
        k = _log_int(rng, 1024, 14336, 256)
        n = _log_int(rng, 512, 28672, 64 if rng.random() < 0.8 else 8)
        f32 = rng.random() < 0.25
        return dict(kind=kind, fmt=rng.choice(sorted(FORMATS)), dtype=F32 if f32 else BF16,
                    m=rng.randint(1, 8) if f32 else _rows(rng, k, n, 4096), k=k, n=n)
    if kind == "moe":
        hidden, inter, top_k = _log_int(rng, 1024, 4096, 64), _log_int(rng, 512, 4096, 64), rng.choice([4, 8])
        return dict(kind=kind, m=_rows(rng, hidden * top_k, inter, 2048), hidden=hidden, inter=inter,
                    experts=rng.choice([32, 64, 128]), top_k=top_k)
    if kind == "f8":
        k, n = _log_int(rng, 512, 7168, 128), _log_int(rng, 512, 7168, 128)
        return dict(kind=kind, m=_log_int(rng, 1, 1024), k=k, n=n)
    if kind == "ffn":
        weights = rng.choice(["awq4", "awq4", "gptq4", "q4_k", "q6_k", "q8_0"])
        k, inter = _log_int(rng, 1024, 8192, 256), _log_int(rng, 2816, 14336, 256)
        dtype = rng.choice([F16, BF16]) if weights in ("awq4", "gptq4") else BF16
        return dict(kind=kind, weights=weights, dtype=dtype, m=_rows(rng, k, 2 * inter, 4096), k=k, inter=inter)
    k = _log_int(rng, 2048, 5120, 256)
    return dict(kind=kind, dtype=rng.choice([F16, BF16]), m=_log_int(rng, 1, 64), k=k, qkv=k + 128 * rng.choice([4, 8, 16]),
                inter=_log_int(rng, 5632, 14336, 256), layers=rng.randint(2, 4))


# ------------------------------------------------------------------ inputs
class _Maker:
    """Tensors of one seed, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, shape, dtype, scale=1.0):
        return (torch.randn(shape, device="cuda", generator=self.gen) * scale).to(dtype)

    def uniform(self, shape, lo, hi, dtype):
        return (torch.rand(shape, device="cuda", generator=self.gen) * (hi - lo) + lo).to(dtype)

    def words(self, shape):
        return torch.randint(-(1 << 31), 1 << 31, shape, device="cuda", dtype=torch.int32, generator=self.gen)

    def bytes_(self, n, lo=0, hi=256):
        return torch.randint(lo, hi, (n,), device="cuda", dtype=torch.uint8, generator=self.gen)

    def packed(self, pack, bits, k, n, group, dtype):
        """A uniform checkpoint triple: every code and every stored zero point is equally likely."""
        pf = 32 // bits
        qweight = self.words((k, n // pf) if pack == "awq" else (k // pf, n))
        return qweight, self.words((k // group, n // pf)), self.uniform((k // group, n), 0.002, 0.02, dtype)

    def gguf(self, fmt, k, n):
        elems, size = synth.GGUF_BLOCK_LAYOUT[fmt]
        blocks = self.bytes_(n * (k // elems) * size).view(-1, size)
        for off in synth.GGUF_F16_FIELDS[fmt]:
            d = self.uniform((blocks.shape[0], 1), 1e-3, 2e-2, torch.float16)
            blocks[:, off:off + 2] = d.view(torch.uint8)
        return blocks.reshape(-1)

    def packed_linear(self, pack, bits, k, n, group, dtype, bias=None, act=None):
        q, z, s = self.packed(pack, bits, k, n, group, dtype)
        return ops.PackedQuantLinear(bits, ops.PACK_OUT if pack == "awq" else ops.PACK_IN, q, z, s, bias, dtype,
                                     gate_up_act=act)


def _ffn(make, weights, dtype, k, inter):
    if weights in FORMATS:
        fmt = FORMATS[weights]
        up = ops.QLinear(fmt, make.gguf(fmt, k, 2 * inter), k, 2 * inter, None, dtype, gate_up_act=ops.ACT_GATED_SILU)
        down = ops.QLinear(fmt, make.gguf(fmt, inter, k), inter, k, None, dtype)
    else:
        pack = weights[:-1]
        up = make.packed_linear(pack, 4, k, 2 * inter, 128, dtype, act=ops.ACT_GATED_SILU)
        down = make.packed_linear(pack, 4, inter, k, 128, dtype)
    return ops.FeedForward(ops.GATE_UP_FUSED, up, None, down, inter)


def prepare(case, seed):
    make = _Maker(seed)
    kind, m = case["kind"], case["m"]
    s = {"case": case}
    if kind in ("linear", "op"):
        k, n, dtype = case["k"], case["n"], DTYPES[case["dtype"]]
        s["x"] = make.normal((m, k), dtype)
        if kind == "linear":
            bias = make.normal((n,), dtype) if case["bias"] else None
            s["layer"] = make.packed_linear(case["pack"], case["bits"], k, n, case["group"], dtype, bias)
        else:
            s["w"] = make.packed(case["pack"], case["bits"], k, n, case["group"], dtype)
    elif kind == "gguf":
        fmt, k, n, dtype = FORMATS[case["fmt"]], case["k"], case["n"], DTYPES[case["dtype"]]
        s["x"] = make.normal((m, k), dtype)
        s["layer"] = ops.QLinear(fmt, make.gguf(fmt, k, n), k, n, None, dtype)
    elif kind == "moe":
        h, i, e = case["hidden"], case["inter"], case["experts"]
        s["x"] = make.normal((m, h), torch.bfloat16)
        s["logits"] = make.normal((m, e), torch.float32)

        def experts(rows, cols):
            blocks, scales = make.bytes_(e * rows * cols // 2), make.bytes_(e * rows * cols // 32, 118, 127)
            return ops.Mxfp4Experts(blocks, scales, make.normal((e, rows), torch.bfloat16, 0.1), e, cols, rows)
        s["gate_up"], s["down"] = experts(2 * i, h), experts(h, i)
    elif kind == "f8":
        k, n = case["k"], case["n"]
        s["x"] = make.normal((m, k), torch.bfloat16)
        s["w"] = make.normal((n, k), torch.float32).to(torch.float8_e4m3fn).view(torch.uint8)
        s["scales"] = make.uniform((n // 128, k // 128), 0.002, 0.02, torch.float32)
    elif kind == "ffn":
        dtype = DTYPES[case["dtype"]]
        s["x"] = make.normal((m, case["k"]), dtype, 0.25)
        s["ffn"] = _ffn(make, case["weights"], dtype, case["k"], case["inter"])
    else:
        dtype, k = DTYPES[case["dtype"]], case["k"]
        s["layers"] = [(make.packed_linear("awq", 4, k, case["qkv"], 128, dtype), make.packed_linear("awq", 4, k, k, 128, dtype),
                        _ffn(make, "awq4", dtype, k, case["inter"])) for _ in range(case["layers"])]
        s["xs"] = [[make.normal((m, k), dtype, 0.25) for _ in range(3)] for _ in range(case["layers"])]

        def step():
            return [layer.forward(x) for trio, xs in zip(s["layers"], s["xs"]) for layer, x in zip(trio, xs)]
        step()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = step()
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("linear", "gguf"):
        return s["layer"].forward(s["x"])
    if kind == "op":
        x, (q, z, sc), bits = s["x"], s["w"], case["bits"]
        if case["m"] > 8:
            return ops.mpp_quant_matmul(x, q, z, sc, bits, ops.PACK_OUT if case["pack"] == "awq" else ops.PACK_IN)
        if case["pack"] == "gptq":
            return ops.gptq_matmul(x, q, z, sc, bits)
        return ops.w4a16_matmul(x, q, z, sc) if bits == 4 else ops.w8a16_matmul(x, q, z, sc)
    if kind == "moe":
        idx, vals, offsets, tokens, _, pos = ops.moe_route_group(s["logits"], case["top_k"], True)
        h = s["gate_up"].gate_up_swiglu(s["x"], offsets, tokens, 7.0)
        y = s["down"].matmul(h, offsets, None)
        return {"out": ops.moe_combine(y, pos, vals), "top_idx": idx, "top_vals": vals}
    if kind == "f8":
        return ops.f8_matmul(s["x"], s["w"], s["scales"])
    if kind == "ffn":
        return s["ffn"].forward(s["x"])
    s["graph"].replay()
    return s["out"]


# ------------------------------------------------------------------ what a pass cannot do without
def _packed_bytes(bits, k, n, group):
    return k * n * bits / 8 + (k / group) * n * (bits / 8 + 2)


def _weight_bytes(weights, k, n):
    if weights in FORMATS:
        elems, size = synth.GGUF_BLOCK_LAYOUT[FORMATS[weights]]
        return n * (k // elems) * size
    return _packed_bytes(4, k, n, 128)


def work(case):
    kind, m = case["kind"], case["m"]
    size = 4 if case.get("dtype") == F32 else 2
    if kind in ("linear", "op"):
        k, n = case["k"], case["n"]
        return {"bytes": _packed_bytes(case["bits"], k, n, case["group"]) + m * (k + n) * size + (n * size if case.get("bias") else 0),
                "flops": 2 * m * k * n}
    if kind == "gguf":
        k, n = case["k"], case["n"]
        return {"bytes": _weight_bytes(case["fmt"], k, n) + m * (k + n) * size, "flops": 2 * m * k * n}
    if kind == "moe":
        h, i, e, t = case["hidden"], case["inter"], case["experts"], case["top_k"]
        active = e * (1 - (1 - t / e) ** m)   # experts that a random routing of m tokens reaches
        expert = 3 * h * i * (0.5 + 1 / 32) + 2 * (2 * i + h)
        return {"bytes": active * expert + m * (2 * h * 2 + 4 * e + 8 * t), "flops": 2 * m * t * 3 * h * i}
    if kind == "f8":
        k, n = case["k"], case["n"]
        return {"bytes": n * k + n * k // 4096 + m * (k + n) * 2, "flops": 2 * m * k * n}
    if kind == "ffn":
        k, i = case["k"], case["inter"]
        return {"bytes": _weight_bytes(case["weights"], k, 2 * i) + _weight_bytes(case["weights"], i, k) + 2 * m * k * size,
                "flops": 6 * m * k * i}
    k, q, i, layers = case["k"], case["qkv"], case["inter"], case["layers"]
    weights = _packed_bytes(4, k, q, 128) + _packed_bytes(4, k, k, 128) + _packed_bytes(4, k, 2 * i, 128) + _packed_bytes(4, i, k, 128)
    return {"bytes": layers * (weights + m * (5 * k + q) * size), "flops": layers * 2 * m * (k * q + k * k + 3 * k * i)}


def tolerance(case):
    # f32 in and out: the order of f32 sums.  f16 / bf16: one rounding of the result and of the weights before the
    # matrix cores (prefill sizes), and in the FFN and the experts one more of the intermediate.
    return {"rel": {F32: 1e-5, F16: 2e-3}.get(case.get("dtype"), 1e-2)}
