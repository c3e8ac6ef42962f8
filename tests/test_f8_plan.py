"""Which F8 form a call takes, asked of a plan-only ctx: workgroups of 128 rows with K in slices against the forms without."""
import ctypes as C

import pytest

from oxydllm_amd import _lib, ops
from tests.helpers import fake


@pytest.mark.parametrize("K,N,m,kernel,split", [  # us: 128 rows in slices / this form
    (7296, 640, 218, "f8_mul_mm_bf16_mt2_n32", 1),      # 18.9 / 13.6
    (7936, 1792, 157, "f8_mul_mm_bf16_mt3_n32", 1),     # 21.9 / 17.2
    (2176, 2048, 453, "f8_mul_mm_bf16_mt2_n64", 1),     # 21.4 / 16.9
    (5632, 5632, 128, "f8_mul_mm_bf16_r128x4k2", 5),    # 24 / 32
    (5632, 5632, 400, "f8_mul_mm_bf16_r128x4k2", 1), (5632, 5632, 1024, "f8_mul_mm_bf16_r128x8", 1)])
def test_form(K, N, m, kernel, split):
    lib, ctx = _lib.load(), ops.Context(plan_only=True)
    assert lib.oxq_f8_matmul(ctx.handle, None, C.byref(fake((m, K), _lib.BF16)), C.byref(fake((N, K), _lib.U8)),
                             C.byref(fake((N // 128, K // 128), _lib.F32)), C.byref(fake((m, N), _lib.BF16))) == 0
    plan = ctx.last_plan()
    assert (plan["kernel"], plan["split_k"]) == (kernel, split)
