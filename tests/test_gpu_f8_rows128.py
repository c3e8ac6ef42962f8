"""The F8 product in workgroups of 128 rows at the edges of their tiles; sums stored in groups of four columns.

Tolerance and inputs as for the other forms (tests/test_gpu_f8_direct.py)."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
from tests.test_gpu_f8_direct import GEMM_WIDE, case

pytestmark = pytest.mark.gpu
WIDE128, PAIRS128 = 9, 10  # OXQ_F8_FORM: 256 columns; 128 columns, K over two waves


# N: half a strip pair of a wave, part of either workgroup, one wave of a second one; K: one chunk, an odd last round,
# slices of an odd number of rounds
@pytest.mark.parametrize("N,K,block_r,block_c", [(16, 128, 16, 128), (144, 384, 48, 128), (272, 1152, 16, 128), (640, 2176, 128, 128),
                                                 (1088, 1024, 64, 256)])
def test_forms_at_their_edges(N, K, block_r, block_c):
    b, sc, rng = case(N, K, N // block_r, K // block_c, N + K)
    w = oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16)
    bd, sd = to_dev(b), to_dev(sc)
    x = rng.standard_normal((700, K)).astype(np.float32)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w)
    xd = to_dev(x, torch.bfloat16)
    tune("OXQ_F8_FORM", GEMM_WIDE)
    wide64 = bits_of(ops.f8_matmul(xd, bd, sd))
    for form, slices in ((WIDE128, 0), (PAIRS128, 1), (PAIRS128, 2), (PAIRS128, 3), (PAIRS128, 8)):
        tune("OXQ_F8_FORM", form)
        tune("OXQ_F8_SLICES", slices or None)
        for m in (33, 127, 128, 129, 700):
            print(f"[case] f8 128 rows {N}x{K} blocks {block_r}x{block_c} m={m} form={form} slices={slices}", flush=True)
            y = ops.f8_matmul(xd[:m], bd, sd)
            plan = ops.default_context().last_plan()
            if not plan["kernel"].startswith("f8_mul_mm_bf16_r128x"):
                assert slices > 1, plan  # more slices than rounds: no such form
                continue
            assert_close(y, ref[:m], f"{plan['kernel']} m{m} {N}x{K} slices {plan['split_k']}")
            np.testing.assert_array_equal(bits_of(ops.f8_matmul(xd[:m], bd, sd)), bits_of(y))
            if form == WIDE128:  # K in the same order as in the form of 64 rows
                np.testing.assert_array_equal(bits_of(y), wide64[:m])


@pytest.mark.parametrize("form", [GEMM_WIDE, 4, WIDE128, PAIRS128])
def test_outputs_that_are_not_8_byte_aligned(form):
    """Such an output is stored a value at a time: the same bits."""
    N, K, m = 144, 512, 70
    b, sc, rng = case(N, K, N // 16, K // 128, 5)
    xd = to_dev(rng.standard_normal((m, K)).astype(np.float32), torch.bfloat16)
    bd, sd = to_dev(b), to_dev(sc)
    tune("OXQ_F8_FORM", form)
    tune("OXQ_F8_SLICES", 1)
    y = ops.f8_matmul(xd, bd, sd)
    room = torch.full((m * N + 3,), 7.0, dtype=torch.bfloat16, device="cuda")
    out = room[1:1 + m * N].view(m, N)
    ops.f8_matmul(xd, bd, sd, out=out)
    np.testing.assert_array_equal(bits_of(out), bits_of(y))
    assert room[0].item() == 7.0 and (room[1 + m * N:] == 7.0).all()
