"""Every tile of the prefill kernels' launches (pk4g_tile_of: squares of 8 row tiles x 8 column groups, a narrower last column of them,
the last row tiles by themselves) is some workgroup's: outputs that start as NaN come out whole."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests import test_gpu_pk4
from tests.helpers import assert_close, round_x, to_dev, tune
from tests.test_gpu_pk4 import dense, layer_of, make

pytestmark = pytest.mark.gpu
K = 256
# column groups of 512: one, one and a part, eight, nine; row tiles of 64: less than a band, one band, a band and three, two
NS, MS = (448, 1088, 4096, 4160), (300, 512, 700, 1024)


def check(forward, w, dt, n, kernel, bf16):
    x = np.random.default_rng(n).standard_normal((max(MS), K)).astype(np.float32)
    xd = to_dev(x, torch.bfloat16 if bf16 else torch.float16)
    ref = oracle.matmul_nt_f32(round_x(x, dt), w)
    for m in MS:
        print(f"[case] {kernel} N={n} m={m}", flush=True)
        y = forward(xd[:m].contiguous(), torch.full((m, n), float("nan"), device="cuda", dtype=xd.dtype))
        plan = ops.default_context().last_plan()
        assert kernel in plan["kernel"], plan
        assert_close(y, ref[:m], f"{plan['kernel']} N={n} m={m}", bf16_out=bf16)


@pytest.mark.parametrize("kind,dtn,strip16", [("awq", "f16", 0), ("gptq8", "bf16", 0), ("awq", "bf16", 2)])
@pytest.mark.parametrize("n", NS)
def test_uniform_layers(kind, dtn, strip16, n):
    test_gpu_pk4.ops = ops
    tune("OXQ_PK4_STRIP16", strip16)
    tune("OXQ_PK4_GEMM_ROWS", 64)
    dt = oracle.F16 if dtn == "f16" else oracle.BF16
    trip, pack_dim = make(kind, K, n, 128, seed=n)
    layer = layer_of(trip, pack_dim, dt, bits=8 if kind.endswith("8") else 4)
    w = oracle.round_through(dense(kind, trip, dt), dt)
    check(lambda x, out: layer.forward(x, out), w, dt, n, "_r64x8" + ("_n16" if strip16 else ""), dtn == "bf16")


@pytest.mark.parametrize("fmt", [synth.GGUF_Q4_K, synth.GGUF_Q6_K])
@pytest.mark.parametrize("n", NS)
def test_gguf_layers(fmt, n):
    tune("OXQ_GGUF_GEMM_MIN_M", 33)
    data = synth.gguf_weight(fmt, n, K, seed=n)
    layer = ops.QLinear(fmt, to_dev(data), K, n, None, torch.bfloat16)
    w = oracle.round_through(oracle.dequantize_gguf(fmt, data, n, K), oracle.BF16)
    check(lambda x, out: layer.forward(x, out), w, oracle.BF16, n, "_gemm_bf16_r64x8", True)


@pytest.mark.parametrize("n", NS)
def test_f8_weights(n):
    tune("OXQ_F8_FORM", 1)
    rng = np.random.default_rng(n)
    b = (rng.integers(0, 0x49, size=(n, K)) | (rng.integers(0, 2, size=(n, K)) << 7)).astype(np.uint8)
    sc = rng.uniform(0.05, 0.5, size=(n // 64, K // 128)).astype(np.float32)
    w = oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16)
    bd, sd = to_dev(b), to_dev(sc)
    check(lambda x, out: ops.f8_matmul(x, bd, sd, out=out), w, oracle.BF16, n, "f8_mul_mm_bf16_r64x8", True)
