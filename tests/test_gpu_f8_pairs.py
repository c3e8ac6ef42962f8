"""Block-scaled F8E4M3 in tiles of 32 columns (f8_mm.hip): 32 and 48 rows a workgroup, at the edges of rows, columns and K.

Tolerance and bounds as for the other forms (test_gpu_f8_direct.py): 2e-3 relative, 1e-2 absolute, the half ulp of a bf16 result."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops
from tests.helpers import assert_close, bits_of, round_x, to_dev

pytestmark = pytest.mark.gpu

TILE32X32, TILE48X32 = 5, 6  # OXQ_F8_FORM


# N: half a pair of strips, a ragged last pair, whole pairs; K: fewer chunks than waves, one wave with a chunk more
@pytest.mark.parametrize("N,K,block_r,block_c", [(16, 128, 16, 128), (80, 384, 16, 128), (192, 1152, 48, 128), (640, 2176, 128, 128)])
def test_tiles_of_two_strips(N, K, block_r, block_c):
    print(f"[case] f8 tiles of 32 columns {N}x{K}", flush=True)
    rng = np.random.default_rng(N + K)
    b = (rng.integers(0, 0x49, size=(N, K)) | (rng.integers(0, 2, size=(N, K)) << 7)).astype(np.uint8)
    sc = rng.uniform(0.05, 0.5, size=(N // block_r, K // block_c)).astype(np.float32)
    w = oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16)
    bd, sd = to_dev(b), to_dev(sc)
    ctx = ops.default_context()
    try:
        for form, rows, mt in ((TILE32X32, (17, 32, 33, 65), 2), (TILE48X32, (17, 48, 49, 97), 3)):
            ctx.set_tuning("OXQ_F8_FORM", form)
            for m in rows:
                x = rng.standard_normal((m, K)).astype(np.float32)
                xd = to_dev(x, torch.bfloat16)
                y = ops.f8_matmul(xd, bd, sd)
                plan = ctx.last_plan()
                assert plan["kernel"] == f"f8_mul_mm_bf16_mt{mt}_n32" and plan["grid"] == ((N + 31) // 32, 1, -(-m // (16 * mt))), plan
                assert_close(y, oracle.matmul_nt_f32(round_x(x, oracle.BF16), w), f"f8 {plan['kernel']} m{m} {N}x{K}")
                np.testing.assert_array_equal(bits_of(ops.f8_matmul(xd, bd, sd)), bits_of(y))
    finally:
        ctx.set_tuning("OXQ_F8_FORM", None)
