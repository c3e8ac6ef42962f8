"""Block-scaled F8E4M3 straight from the tensor to the matrix cores (f8_mm.hip): every form at the edges of its tiles.

Tolerance as in the other parity tests (2e-3 relative / 1e-2 absolute, bf16 outputs plus their half ulp) of the
f32-accumulated x . dequant(W)^T.  Bytes stay below 4.5 and scales below 0.5, so a sum of K = 2176 products of unit
normals holds at most about 2000 in absolute terms and its f32 rounding stays under 2000 x 2^-24 x log2(K) = 1.3e-3."""
import sys

import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops
from tests.helpers import assert_close, bits_of, round_x, to_dev

pytestmark = pytest.mark.gpu

TILE16, GEMM_WIDE, TILE64, TILE48, GEMM_K4 = 0, 1, 2, 3, 4  # OXQ_F8_FORM


def case(N, K, s_r, s_c, seed):
    rng = np.random.default_rng(seed)
    b = (rng.integers(0, 0x49, size=(N, K)) | (rng.integers(0, 2, size=(N, K)) << 7)).astype(np.uint8)
    return b, rng.uniform(0.05, 0.5, size=(s_r, s_c)).astype(np.float32), rng


# N: part of a strip group, of a 128- and of a 512-column workgroup; K: fewer chunks than waves, a ragged last round
@pytest.mark.parametrize("N,K,block_r,block_c", [(16, 128, 16, 128), (80, 384, 16, 128), (192, 1152, 48, 128),
                                                 (640, 2176, 128, 128), (1088, 1024, 64, 256)])
def test_forms_at_their_edges(N, K, block_r, block_c):
    print(f"[case] f8 direct {N}x{K} blocks {block_r}x{block_c}", flush=True)
    sys.stdout.flush()
    b, sc, rng = case(N, K, N // block_r, K // block_c, N + K)
    w = oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16)
    bd, sd = to_dev(b), to_dev(sc)
    ctx = ops.default_context()
    try:
        for form, rows, slices in ((TILE16, (3, 4, 5, 8, 9, 16, 17, 33, 80), (0,)), (TILE64, (17, 32, 33, 65), (0,)),
                                   (TILE48, (33, 48, 49, 97), (0,)),
                                   (GEMM_K4, (33, 64, 65, 130), (1, 2, 3, 5)), (GEMM_WIDE, (33, 64, 65, 700), (0,))):
            for m in rows:
                x = rng.standard_normal((m, K)).astype(np.float32)
                ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w)
                xd = to_dev(x, torch.bfloat16)
                for s in slices:
                    ctx.set_tuning("OXQ_F8_FORM", form)
                    ctx.set_tuning("OXQ_F8_SLICES", s)
                    y = ops.f8_matmul(xd, bd, sd)
                    assert_close(y, ref, f"f8 {ctx.last_plan()['kernel']} m{m} {N}x{K} slices {s}")
                    np.testing.assert_array_equal(bits_of(ops.f8_matmul(xd, bd, sd)), bits_of(y))
    finally:
        ctx.set_tuning("OXQ_F8_FORM", None)
        ctx.set_tuning("OXQ_F8_SLICES", None)


@pytest.mark.parametrize("m", [1, 2])
def test_one_and_two_rows_of_a_large_matrix(m):
    N, K = 2048, 2048  # 2^22 weights: tiles from one row
    b, sc, rng = case(N, K, 16, 16, m)
    x = rng.standard_normal((m, K)).astype(np.float32)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16))
    xd, bd, sd = to_dev(x, torch.bfloat16), to_dev(b), to_dev(sc)
    for y in (ops.f8_matmul(xd, bd, sd), ops.f8_gemv(xd, bd, sd)):
        assert ops.default_context().last_plan()["kernel"] == "f8_mul_mm_bf16_mt1"
        assert_close(y, ref, f"f8 tiles m{m}")
