"""f8_tile_kernel: bodies by the most chunks of K a wave has (one, two, three, a loop), with waves that have one fewer, or none.

Every form adds a wave's chunks in order and then the waves, so all give the same bits; tolerance as in test_gpu_f8_direct.py."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops
from tests.helpers import assert_close, bits_of, round_x, to_dev

pytestmark = pytest.mark.gpu

FORMS = {0: "", 2: "_n64", 3: "_n64", 5: "_n32", 6: "_n32"}  # OXQ_F8_FORM


@pytest.mark.parametrize("chunks", [1, 7, 8, 9, 15, 16, 17, 23, 24, 25, 33])
def test_chunks_of_a_wave(chunks):
    N, K = 80, 128 * chunks
    rng = np.random.default_rng(chunks)
    b = (rng.integers(0, 0x49, size=(N, K)) | (rng.integers(0, 2, size=(N, K)) << 7)).astype(np.uint8)
    sc = rng.uniform(0.05, 0.5, size=(N // 16, K // 128)).astype(np.float32)
    w = oracle.widen_to_f32(oracle.f8_block_dequant_bf16(b, sc), oracle.BF16)
    bd, sd = to_dev(b), to_dev(sc)
    x = rng.standard_normal((50, K)).astype(np.float32)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w)
    ctx = ops.default_context()
    bits = None
    try:
        for form, name in FORMS.items():
            ctx.set_tuning("OXQ_F8_FORM", form)
            for m in (50, 17) if form else (50, 17, 16, 8, 3):
                print(f"[case] f8 chunks {chunks} form {form} rows {m}", flush=True)
                xd = to_dev(x, torch.bfloat16)[:m].contiguous()
                y = ops.f8_matmul(xd, bd, sd)
                plan = ctx.last_plan()
                mt = 3 if form in (3, 6) else 2 if m > 16 else 1
                assert plan["kernel"] == f"f8_mul_mm_bf16_mt{mt}{name}", plan
                assert_close(y, ref[:m], f"f8 {plan['kernel']} m{m} K{K}")
                got = bits_of(y)
                bits = got if bits is None else bits
                np.testing.assert_array_equal(got, bits[:m])
    finally:
        ctx.set_tuning("OXQ_F8_FORM", None)
