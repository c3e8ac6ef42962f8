"""Resident 4-bit layers in workgroups of 128 rows and two strips, K over four waves.

Weights, order of K and of the partial tiles are those of the 64-row form, which the oracle holds (tests/test_gpu_pk4.py): the
same bits."""
import numpy as np
import pytest
import torch

from oxydllm_amd import ops, synth
from tests.helpers import bits_of, to_dev, tune

pytestmark = pytest.mark.gpu


# K: fewer blocks than waves, whole rounds and ragged ones, one to eight rounds.  N: one strip, a last workgroup of one
# strip.  Rows: both halves of a tile ragged, one row in the lower half, a second tile of one row
@pytest.mark.parametrize("pack", ["awq", "gptq"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("strip16", [0, 2])
@pytest.mark.parametrize("K,N,g", [(128, 64, 128), (384, 192, 128), (512, 320, 256), (1280, 576, 128), (4096, 128, 128)])
def test_same_bits_as_rows_of_64(pack, dt, K, N, g, strip16):
    make = synth.awq_checkpoint if pack == "awq" else synth.gptq_checkpoint
    q, z, s = make(K, N, g, 4, seed=K + N)
    args = (4, ops.PACK_OUT if pack == "awq" else ops.PACK_IN, to_dev(q), to_dev(z), to_dev(s, dt))
    rng = np.random.default_rng(K * N)
    bias = to_dev(rng.standard_normal(N).astype(np.float32), dt)
    x = to_dev(rng.standard_normal((330, K)).astype(np.float32), dt)
    x[3, 5], x[200, 0] = float("inf"), float("nan")
    tune("OXQ_PK4_STRIP16", strip16)
    tune("OXQ_PK4_GEMM_KS", 4)
    acts = (None, ops.ACT_GATED_SILU, ops.ACT_GATED_GELU_TANH) if N > 64 and not strip16 else (None,)
    for act in acts:
        layer = ops.PackedQuantLinear(*args, None if act is None and K == 512 else bias, dt, gate_up_act=act)
        for m in (65, 100, 128, 129, 193, 330):
            print(f"[case] pk4 128 rows x two strips {pack} {dt} {K}x{N} g={g} strips={strip16} act={act} m={m}", flush=True)
            tune("OXQ_PK4_GEMM_ROWS", 64)
            want = layer.forward(x[:m])
            tune("OXQ_PK4_GEMM_ROWS", 128)
            got = layer.forward(x[:m])
            plan = layer.ctx.last_plan()
            assert "_r128x2k4" + ("_n16" if strip16 else "") in plan["kernel"] and plan["grid"][0] == -(-m // 128) * -(-N // 128), plan
            np.testing.assert_array_equal(bits_of(got), bits_of(want))


# K that ends in a block's first and second half and inside them
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", [(1216, 320, 64), (2176, 264, 64), (1184, 328, 32), (1376, 192, 32), (4256, 64, 32)])
def test_groups_inside_a_block(dt, K, N, g):
    q, z, s = synth.awq_checkpoint(K, N, g, 4, seed=K + N)
    rng = np.random.default_rng(K * N)
    bias = to_dev(rng.standard_normal(N).astype(np.float32), dt)
    x = to_dev(rng.standard_normal((330, K)).astype(np.float32), dt)
    x[3, K - 1], x[200, 0] = float("inf"), float("nan")
    tune("OXQ_PK4_GEMM_KS", 4)
    layer = ops.PackedQuantLinear(4, ops.PACK_OUT, to_dev(q), to_dev(z), to_dev(s, dt), bias, dt)
    for m in (65, 128, 129, 330):
        print(f"[case] pk4 128 rows x two strips awq {dt} {K}x{N} g={g} m={m}", flush=True)
        tune("OXQ_PK4_GEMM_ROWS", 64)
        want = layer.forward(x[:m])
        tune("OXQ_PK4_GEMM_ROWS", 128)
        got = layer.forward(x[:m])
        plan = layer.ctx.last_plan()
        assert plan["kernel"].endswith("_r128x2k4") and plan["grid"][0] == -(-m // 128) * -(-N // 128), plan
        np.testing.assert_array_equal(bits_of(got), bits_of(want))
