"""mxfp4_wide12_kernel: the tiles of mxfp4_wide_kernel by twelve waves, where workgroups of 384 columns fit one round of CUs."""
import os

import numpy as np
import pytest

import oracle
from oxydllm_amd import _lib
from tests import gpu_code
from tests.test_mxfp4_wide import MANY


def test_loads_into_lds_are_over_where_a_barrier_publishes_them(tmp_path):
    """Four stages of x, of which the two after the published one may be under way: a load a wave each, two with 128 rows."""
    if not os.path.exists(gpu_code.LLVM + "llvm-objdump"):
        pytest.skip("no llvm-objdump")
    found = {}
    for co in gpu_code.code_objects(_lib.LIB_PATH, tmp_path):
        if b"mxfp4_wide12_kernel" in co.read_bytes():
            found.update({n: c for n, c in gpu_code.kernels(co).items() if "mxfp4_wide12_kernel" in n})
    (code,) = found.values()
    at = list(gpu_code.loads_under_way_at_barriers(code).values())
    assert len(at) == 28
    assert sorted(max(at[7 * i:7 * i + 7]) for i in range(4)) == [2, 2, 2, 4]


@pytest.mark.gpu
@pytest.mark.parametrize("counts,N,K", [
    (MANY, 784, 96),                                          # one unit and a half; the third group one live tile wide
    (MANY, 1152, 64 * 7),                                     # whole groups; rounds after the loop
    ([0, 33, 64, 96, 97, 128, 129] * 14 + [5, 0], 528, 32),   # one block
    ([1, 0, 31, 32, 65] * 26, 272, 64 * 8),                   # one group, not filled; no rounds after the loop
])
def test_the_bits_of_eight_waves(counts, N, K):
    from oxydllm_amd import ops
    from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
    from tests.test_gpu_mxfp4_experts import _dense, _experts, _lists
    import torch
    E = len(counts)
    print(f"[case] twelve waves E={E} N={N} K={K}", flush=True)
    blocks, scales, bias = _experts(E, N, K, seed=N + K)
    offsets, tokens, n_tok = _lists(counts)
    x = np.random.default_rng(K).standard_normal((n_tok, K)).astype(np.float32)
    xb, bb = round_x(x, oracle.BF16), round_x(bias, oracle.BF16)
    ref = np.concatenate([oracle.matmul_nt_f32(xb[tokens[lo:hi]], _dense(blocks, scales, e, N, K), bb[e])
                          for e, (lo, hi) in enumerate(zip(offsets, offsets[1:])) if hi > lo])
    ex = ops.Mxfp4Experts(to_dev(blocks), to_dev(scales), to_dev(bias, torch.bfloat16), E, K, N)
    args = to_dev(x, torch.bfloat16), to_dev(offsets), to_dev(tokens)
    got = []
    for rows, waves in ((None, 12), (128, 8)):
        tune("OXQ_MXFP4_GEMM_ROWS", rows)
        y = ex.matmul(*args)
        plan = ops.default_context().last_plan()
        assert plan["kernel"].endswith(f"x{waves}") and plan["block"][0] == 64 * (12 if waves == 12 else 8), plan
        got.append((bits_of(y), bits_of(ex.gate_up_swiglu(*args, 7.0))))
        assert_close(y, ref, f"{waves} waves")
    assert all(np.array_equal(a, b) for a, b in zip(*got))
