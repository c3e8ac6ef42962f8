"""A fused GGUF gate|up layer in the prefill kernel: the plain layer's form, with slices of K as without, asked of a plan-only ctx."""
import ctypes as C

import pytest

from oxydllm_amd import _lib, ops, synth
from tests.helpers import fake

ROWS = (40, 74, 98, 144, 200, 300, 400, 512, 640, 777, 1100, 2048, 4096)


@pytest.mark.parametrize("fmt", [synth.GGUF_Q4_K, synth.GGUF_Q8_0, synth.GGUF_Q6_K])
def test_same_form_as_the_plain_layer(fmt):
    lib, plan = _lib.load(), ops.Context(plan_only=True)
    elems, size = synth.GGUF_BLOCK_LAYOUT[fmt]
    sliced = 0
    for K in (1024, 2048, 4096, 6144, 6400, 8192):
        for N in (1024, 2048, 4096, 7168, 9216, 10752, 14336, 28672):
            w, plain, fused = fake((N * (K // elems) * size,), _lib.U8), C.c_void_p(), C.c_void_p()
            assert lib.oxq_qlinear_new(plan.handle, fmt, C.byref(w), K, N, None, _lib.BF16, C.byref(plain)) == 0
            assert lib.oxq_qlinear_new_gate_up(plan.handle, fmt, C.byref(w), K, N, None, ops.ACT_GATED_SILU, _lib.BF16, C.byref(fused)) == 0
            for m in ROWS:
                x, seen = fake((m, K), _lib.BF16), []
                for layer, cols in ((plain, N), (fused, N // 2)):
                    assert lib.oxq_qlinear_forward(layer, None, C.byref(x), C.byref(fake((m, cols), _lib.BF16))) == 0
                    p = plan.last_plan()
                    seen.append((p["kernel"], tuple(p["grid"]), p["split_k"], p["workspace_bytes"]))
                (kernel, *form), got = seen
                if "_gemm_" not in kernel or ("_r128x" not in kernel and form[1] > 1):  # slices of 64 rows: row tiles of the integer kernel
                    assert "_gemm_" not in got[0], (K, N, m, seen)
                    continue
                assert got == (kernel + "_silu", *form), (K, N, m, seen)
                sliced += form[1] > 1
            lib.oxq_qlinear_free(plain)
            lib.oxq_qlinear_free(fused)
    assert sliced >= 5
