"""Resident GGUF layers on the matrix cores: ggm_short_kernel (one chunk of K a wave, two) and ggm_kernel's loop, whose last round
requests nothing, with waves that have a chunk fewer, or none; 8 and 16 waves, one strip and four.

bf16: tolerance as in test_gpu_gguf_mfma.py.  f32: exact products, sums of K terms in f32, an error of at most sqrt(K) half ulps of
the sum of magnitudes at random signs: 1e-5 of the result's norm."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, round_x, to_dev, tune

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [2, 6, 8, 10, 16, 18, 24, 26, 32, 34, 40, 48, 50, 56])
@pytest.mark.parametrize("fmt", [synth.GGUF_Q8_0, synth.GGUF_Q4_K, synth.GGUF_Q6_K])
def test_chunks_of_a_wave(fmt, chunks):
    N, K = 128, 128 * chunks
    data = synth.gguf_weight(fmt, N, K, seed=chunks + fmt)
    w = oracle.dequantize_gguf(fmt, data, N, K)
    bf16, f32 = (ops.QLinear(fmt, to_dev(data), K, N, None, d) for d in (torch.bfloat16, torch.float32))
    x = np.random.default_rng(chunks).standard_normal((20, K)).astype(np.float32)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w)
    ref64 = x[:8].astype(np.float64) @ w.astype(np.float64).T
    for ns in (1, 4):
        tune("OXQ_GGUF_MFMA_NS", ns)
        for m in (1, 6, 16, 20):
            print(f"[case] gguf {synth.GGUF_NAMES[fmt]} chunks {chunks} strips {ns} rows {m}", flush=True)
            y = bf16.forward(to_dev(x, torch.bfloat16)[:m].contiguous())
            plan = ops.default_context().last_plan()
            assert f"_mfma_bf16_mt{2 if m > 16 else 1}" in plan["kernel"] and plan["kernel"].endswith("_n64") == (ns == 4), plan
            assert_close(y, ref[:m], f"{plan['kernel']} K={K} m={m}")
        for m in (1, 4, 8):
            print(f"[case] gguf {synth.GGUF_NAMES[fmt]} f32 chunks {chunks} strips {ns} rows {m}", flush=True)
            y = f32.forward(to_dev(x[:m], torch.float32)).cpu().numpy().astype(np.float64)
            assert np.linalg.norm(y - ref64[:m]) <= 1e-5 * np.linalg.norm(ref64[:m])
