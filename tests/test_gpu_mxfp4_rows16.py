"""The 16-row kernel of the resident MXFP4 experts, which long K at few pairs an expert keeps: each case asserts from the plan
that it ran (one layer of workgroups; mxfp4_wide_kernel takes two), at the edges of its chunks, rings, tiles and waves."""
import numpy as np
import pytest
import torch

import oracle
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
from tests.test_gpu_mxfp4_experts import _dense, _experts, _lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,N,K,counts", [
    (4, 16, 2048, [1, 0, 16, 17]),     # whole chunks; one live tile; a full row tile and one row more
    (3, 80, 2080, [3, 15, 0]),         # a last chunk of one block; a wave with one live tile of its four
    (2, 656, 2144, [5, 33]),           # of three blocks; two column groups, the second three waves wide
    (70, 64, 2176, [1] * 64 + [0, 2, 0, 31, 0, 4]),  # an odd number of chunks; idle experts
])
@pytest.mark.parametrize("gather", [True, False])
def test_few_pairs_an_expert_on_a_long_k(E, N, K, counts, gather):
    from oxydllm_amd import ops
    print(f"[case] experts in rows of 16 E={E} N={N} K={K} gather={gather}", flush=True)
    tune("OXQ_MXFP4_GEMM_MIN_PAIRS", 1)
    tune("OXQ_MXFP4_GEMM_ROWS", 16)
    blocks, scales, bias = _experts(E, N, K, seed=N + K)
    offsets, tokens, n_tok = _lists(counts)
    x = np.random.default_rng(K).standard_normal((n_tok, K)).astype(np.float32)
    xb, bb = round_x(x, oracle.BF16), round_x(bias, oracle.BF16)
    ref = np.concatenate([oracle.matmul_nt_f32(xb[tokens[lo:hi]], _dense(blocks, scales, e, N, K), bb[e])
                          for e, (lo, hi) in enumerate(zip(offsets, offsets[1:])) if hi > lo])
    ex = ops.Mxfp4Experts(to_dev(blocks), to_dev(scales), to_dev(bias, torch.bfloat16), E, K, N)
    xd, tok_d = (to_dev(x, torch.bfloat16), to_dev(tokens)) if gather else (to_dev(x[tokens], torch.bfloat16), None)
    off_d = to_dev(offsets)
    y = ex.matmul(xd, off_d, tok_d)
    plan = ops.default_context().last_plan()
    assert plan["kernel"] == "mxfp4_experts_gemm_bf16_r16x8" and plan["grid"][2] == 1, plan
    assert_close(y, ref, "experts in rows of 16")
    assert np.array_equal(bits_of(ex.matmul(xd, off_d, tok_d)), bits_of(y))
    two = ops.gated_activation(y, ops.ACT_GPT_OSS_SWIGLU, 7.0)
    assert np.array_equal(bits_of(ex.gate_up_swiglu(xd, off_d, tok_d, 7.0)), bits_of(two))
