"""Prefill rows of resident layers: up to 32 rows behind whole tiles of 128 run as a tile of 32 in the same launch."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import _lib, ops
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
from tests import test_gpu_pk4
from tests.test_gpu_pk4 import DT, TORCH_DT, bits_of_kind, dense, layer_of, make
from tests.test_pk4_plan import kernels


def test_last_rows_take_idle_compute_units():
    """Where the whole tiles leave compute units idle or a padded one would start a round; not where 64-row tiles are ahead."""
    names = lambda k, n, rows: [kern for kern, _ in kernels(ops.PACK_IN, 4, k, n, 128, _lib.BF16, rows)]
    assert names(3584, 18944, (768, 777, 800, 801, 1040)) == ["pk4_gemm_bf16_r128x8"] + ["pk4_gemm_bf16_r128x8r32"] * 2 + ["pk4_gemm_bf16_r64x8"] * 2
    assert names(4096, 11008, (641, 1300)) == ["pk4_gemm_bf16_r64x8", "pk4_gemm_bf16_r128x8r32"] and names(2048, 8192, (905,)) == ["pk4_gemm_bf16_r64x8"]


# the last group: seven strips of eight, two of eight; K of two and five blocks; whole bands of eight row tiles and a last one
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["awq", "gptq", "awq8", "gptq8"])
@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("K,N", [(256, 448), (640, 1152)])
def test_rows_behind_the_whole_tiles(kind, dtn, K, N):
    test_gpu_pk4.ops = ops
    tune("OXQ_PK4_STRIP16", 0)
    dt, bits = DT[dtn], bits_of_kind(kind)
    trip, pack_dim = make(kind, K, N, 128, seed=K + N)
    bias = (np.arange(N, dtype=np.float32) % 9 - 4) * np.float32(0.25)
    tdt = TORCH_DT[dt]
    layers = [layer_of(trip, pack_dim, dt, bias, bits=bits)]
    if N % 128 == 0:
        layers.append(ops.PackedQuantLinear(bits, pack_dim, to_dev(trip[0]), to_dev(trip[1]), to_dev(trip[2], tdt), to_dev(bias, tdt),
                                            tdt, gate_up_act=ops.ACT_GATED_SILU))
    x = np.random.default_rng(K).standard_normal((1056, K)).astype(np.float32)
    xd = to_dev(x, tdt)
    ref = oracle.matmul_nt_f32(round_x(x, dt), oracle.round_through(dense(kind, trip, dt), dt), bias)
    for i, layer in enumerate(layers):
        for m in (129, 145, 160, 257, 288, 1025, 1056):
            print(f"[case] pk4 last rows {kind} {dtn} K={K} N={N} m={m} act={i}", flush=True)
            tune("OXQ_PK4_GEMM_ROWS", 128)
            whole = layer.forward(xd[:m].contiguous())
            tune("OXQ_PK4_GEMM_ROWS", 32)
            y = layer.forward(xd[:m].contiguous())
            plan = ops.default_context().last_plan()
            assert plan["kernel"].startswith(f"pk{bits}_gemm_{dtn}_r128x8r32") and plan["launches"] == 1, plan
            np.testing.assert_array_equal(bits_of(y), bits_of(whole))
            if i == 0:
                assert_close(y, ref[:m], f"{plan['kernel']} m={m}", bf16_out=dtn == "bf16")
