"""mxfp4_wide_kernel: an expert's pairs in tiles of up to four units of 32 rows, all in one workgroup."""
import os

import numpy as np
import pytest

import oracle
from oxydllm_amd import _lib
from tests import gpu_code


def test_loads_into_lds_are_over_where_a_barrier_publishes_them(tmp_path):
    """Four stages of x, of which the two after the published one may be under way, at most two loads a wave each."""
    if not os.path.exists(gpu_code.LLVM + "llvm-objdump"):
        pytest.skip("no llvm-objdump")
    found = {}
    for co in gpu_code.code_objects(_lib.LIB_PATH, tmp_path):
        if b"mxfp4_wide_kernel" in co.read_bytes():
            found.update({n: c for n, c in gpu_code.kernels(co).items() if "mxfp4_wide_kernel" in n})
    assert len(found) == 1
    (code,) = found.values()
    at = list(gpu_code.loads_under_way_at_barriers(code).values())
    assert len(at) == 28 and max(at) == 4  # four tile heights: four rounds of the loop and three after it
    assert sorted(max(at[7 * i:7 * i + 7]) for i in range(4)) == [2, 2, 4, 4]


# pairs of the experts: every tile height, one pair more or less than it; several tiles, evenly and unevenly dealt; more
# experts than lanes; idle experts first and last
MANY = [0, 1, 31, 32, 33, 0, 64, 65, 96, 97, 128, 129, 160, 161, 257] + [0] * 50 + [5, 0, 40, 1, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("counts,N,K", [
    (MANY, 48, 96),                  # one unit and a half: the last block stands alone; a wave with one live tile
    ([130, 0, 70, 300], 272, 32),    # one block; two column groups, the second one wave wide
    ([40, 90], 512, 64 * 7),         # rounds after the loop
    ([33, 0, 100], 256, 64 * 8),     # none
])
def test_tiles_of_every_height(counts, N, K):
    from oxydllm_amd import ops
    from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
    from tests.test_gpu_mxfp4_experts import _dense, _experts, _lists
    import torch
    print(f"[case] wide experts E={len(counts)} N={N} K={K}", flush=True)
    tune("OXQ_MXFP4_GEMM_MIN_PAIRS", 1)
    E = len(counts)
    blocks, scales, bias = _experts(E, N, K, seed=N + K)
    offsets, tokens, n_tok = _lists(counts)
    x = np.random.default_rng(K).standard_normal((n_tok, K)).astype(np.float32)
    xb, bb = round_x(x, oracle.BF16), round_x(bias, oracle.BF16)
    ref = np.concatenate([oracle.matmul_nt_f32(xb[tokens[lo:hi]], _dense(blocks, scales, e, N, K), bb[e])
                          for e, (lo, hi) in enumerate(zip(offsets, offsets[1:])) if hi > lo])
    ex = ops.Mxfp4Experts(to_dev(blocks), to_dev(scales), to_dev(bias, torch.bfloat16), E, K, N)
    xd, off_d, tok_d = to_dev(x, torch.bfloat16), to_dev(offsets), to_dev(tokens)
    for rows in (16, 32, 128):
        tune("OXQ_MXFP4_GEMM_ROWS", rows)
        y = ex.matmul(xd, off_d, tok_d)
        plan = ops.default_context().last_plan()
        assert plan["kernel"] == f"mxfp4_experts_gemm_bf16_r{rows}x8" and plan["grid"][2] == 2, plan
        assert_close(y, ref, f"wide experts, grid for {rows} rows")
        two = ops.gated_activation(y, ops.ACT_GPT_OSS_SWIGLU, 7.0)
        assert np.array_equal(bits_of(ex.gate_up_swiglu(xd, off_d, tok_d, 7.0)), bits_of(two))
