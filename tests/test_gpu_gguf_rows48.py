"""Prefill rows of the GGUF copy's two-wave form: up to 48 rows run without the fourth row tile, to the same bits."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [synth.GGUF_Q4_0, synth.GGUF_Q8_0, synth.GGUF_Q4_K, synth.GGUF_Q6_K, synth.GGUF_Q4_1, synth.GGUF_Q5_0,
                                 synth.GGUF_Q5_1, synth.GGUF_Q5_K])
@pytest.mark.parametrize("N,K,slices", [(1088, 1024, 1), (1032, 2304, 3)])
def test_a_rows_bits_do_not_depend_on_the_row_tiles(fmt, N, K, slices):
    data = synth.gguf_weight(fmt, N, K, seed=N + K + fmt)
    layer = ops.QLinear(fmt, to_dev(data), K, N, None, torch.bfloat16)
    wr = oracle.round_through(oracle.dequantize_gguf(fmt, data, N, K), oracle.BF16)
    x = np.random.default_rng(K).standard_normal((64, K)).astype(np.float32)
    xd = to_dev(x, torch.bfloat16)
    if slices == 1:
        tune("OXQ_GGUF_GEMM_KS", 4)
    else:
        tune("OXQ_GGUF_GEMM_SLICES", slices)
    whole = layer.forward(xd)
    assert_close(whole, oracle.matmul_nt_f32(round_x(x, oracle.BF16), wr), synth.GGUF_NAMES[fmt], bf16_out=True)
    for m in (33, 47, 48, 49):
        print(f"[case] gguf {synth.GGUF_NAMES[fmt]} N={N} K={K} slices={slices} m={m}", flush=True)
        y = layer.forward(xd[:m].contiguous())
        plan = ops.default_context().last_plan()
        assert "_gemm_bf16_r64x2k4" in plan["kernel"] and plan["split_k"] == slices, plan
        assert np.array_equal(bits_of(y), bits_of(whole[:m])), plan
