"""The two-strip kernel with K split inside the workgroup (pk4_mid_kernel) at 33 (f16: 49) to 64 rows of wide layers, and the widening
of nibbles through f8 codes in the bf16 tile forms.

Tolerance as in the other parity tests (tests/helpers.py: 2e-3 relative, 1e-2 absolute, bf16 outputs plus half an ulp)."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, resident_rounds_weights, round_x, to_dev, tune

pytestmark = pytest.mark.gpu


def build(kind, bits, K, N, dt, tdt, seed, bias=None):
    gptq = kind == "gptq"
    qw, qz, sc = (synth.gptq_checkpoint if gptq else synth.awq_checkpoint)(K, N, 128, bits, seed=seed)[:3]
    s_r = oracle.round_through(sc, dt)
    if gptq:
        w = oracle.dequantize_gptq(qw, qz, s_r, bits)
    else:
        w = oracle.dequantize_awq(qw, qz, s_r) if bits == 4 else oracle.dequantize_awq8(qw, qz, s_r)
    layer = ops.PackedQuantLinear(bits, ops.PACK_IN if gptq else ops.PACK_OUT, to_dev(qw), to_dev(qz), to_dev(sc, tdt),
                                  None if bias is None else to_dev(bias, tdt), tdt)
    return layer, w


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K", [128, 640, 1152])  # one block, a ragged second round, an odd count of rounds
def test_wide_layers_at_33_to_64_rows(K, bits, dtn):
    """257 strips of 64 columns: a second round of one-strip workgroups, one round of two-strip ones, the last of them
    with one live strip."""
    N = 257 * 64
    dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
    rng = np.random.default_rng(K + bits)
    bias = (np.arange(N, dtype=np.float32) % 13 - 6) * np.float32(0.125)
    layer, w = build("awq", bits, K, N, dt, tdt, K + bits, bias)
    x = rng.standard_normal((65, K)).astype(np.float32)
    xd = to_dev(x, tdt)
    tile = oracle.matmul_nt_f32(round_x(x, dt), oracle.round_through(w, dt), bias)
    tune("OXQ_PK4_GEMM_KS", 4)
    first = bits_of(layer.forward(xd))  # the same kernel at 65 rows, two row tiles
    tune("OXQ_PK4_GEMM_KS", None)
    for m in (33, 48, 49, 63, 64) if dtn == "bf16" else (49, 63, 64):
        print(f"[case] mid {bits}-bit {dtn} K={K} m={m}", flush=True)
        y = layer.forward(xd[:m])
        plan = ops.default_context().last_plan()
        assert plan["kernel"] == f"pk{bits}_gemm_{dtn}_r64x2k4" and plan["launches"] == 1 and plan["grid"][0] == 129, plan
        assert_close(y, tile[:m], f"mid m{m}")
        np.testing.assert_array_equal(bits_of(y), first[:m])  # a row's bits do not depend on m
    layer.forward(xd[:32 if dtn == "bf16" else 48])  # f16 weights stay unrounded up to 48 rows
    assert "_gemm_" not in ops.default_context().last_plan()["kernel"]


@pytest.mark.parametrize("kind", ["awq", "gptq"])
@pytest.mark.parametrize("strip16", [0, 2])
def test_nibbles_through_f8_codes_are_exact(kind, strip16):
    """Rows of the identity as x: y is the dequantized weight itself, bit for bit, in every bf16 form that widens nibbles
    through f8 codes (two to four row tiles, two strips with K split, eight strips of 64 and 128 rows)."""
    K, N = 256, 1024
    tune("OXQ_PK4_STRIP16", strip16)
    layer, w = build(kind, 4, K, N, oracle.BF16, torch.bfloat16, 5)
    want = bits_of(layer.dequantize())
    np.testing.assert_array_equal(want, oracle.transpose_convert(w, oracle.BF16))
    eye = torch.eye(K, dtype=torch.bfloat16, device="cuda")
    seen = set()
    for rows, ks, step in ((None, None, 17), (None, None, 33), (None, None, 64), (None, 4, 128), (64, None, 128), (128, None, 256)):
        tune("OXQ_PK4_GEMM_ROWS", rows)
        tune("OXQ_PK4_GEMM_KS", ks)
        for r in range(0, K - step + 1, step):
            y = layer.forward(eye[r:r + step].contiguous())
            kernel = ops.default_context().last_plan()["kernel"]
            if resident_rounds_weights(step, oracle.BF16, kind == "gptq"):
                np.testing.assert_array_equal(bits_of(y), want[r:r + step], err_msg=kernel)
        seen.add(kernel)
    assert len(seen) == 6, seen
