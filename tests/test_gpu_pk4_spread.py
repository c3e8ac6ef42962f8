"""Resident layers of few column strips: the row tiles go to workgroups of their own, with the same bits."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import _lib, ops
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
from tests import test_gpu_pk4
from tests.test_gpu_pk4 import DT, TORCH_DT, bits_of_kind, dense, layer_of, make
from tests.test_pk4_plan import kernels


def test_workgroups_fit_one_round():
    """No compute unit is handed a second workgroup for it, and layers that fill the chip keep their row tiles."""
    rows = (17, 33, 49, 64)
    assert kernels(ops.PACK_OUT, 4, 2304, 3328, 128, _lib.BF16, rows) == [
        ("pk4_mfma_bf16_mt2_n16x4_by1", 2), ("pk4_mfma_bf16_mt3_n16x4_by1", 3)] + [("pk4_mfma_bf16_mt4_n16x4_by1", 4)] * 2
    assert kernels(ops.PACK_OUT, 4, 4096, 6144, 128, _lib.F16, (20, 40, 64)) == [
        ("pk4_mfma_f16_mt2_gs_n16x4_by1", 2), ("pk4_mfma_f16_mt3_n16x4_by2", 2), ("pk4_mfma_f16_mt4_n16x4_by2", 2)]
    assert kernels(ops.PACK_OUT, 4, 4096, 4096, 128, _lib.BF16, (20, 64)) == [("pk4_mfma_bf16_mt2_n16x4", 1), ("pk4_mfma_bf16_mt4_n16x4_by1", 4)]
    for k, n in [(4096, 14336), (14336, 4096)]:
        assert not any("_by" in kern for kern, _ in kernels(ops.PACK_OUT, 4, k, n, 128, _lib.BF16, (17, 33, 64)))


@pytest.mark.gpu
@pytest.mark.parametrize("kind,K,N,g", [("awq", 2048, 2048, 128), ("awq", 640, 448, 128), ("gptq", 640, 448, 64), ("awq", 1024, 448, 32),
                                        ("gptq", 1152, 448, 128), ("awq8", 640, 448, 128), ("gptq8", 512, 448, 128), ("awq8", 640, 448, 64)])
@pytest.mark.parametrize("dtn", ["f16", "bf16"])
def test_row_tiles_of_their_own(kind, K, N, g, dtn):
    test_gpu_pk4.ops = ops
    dt = DT[dtn]
    trip, pack_dim = make(kind, K, N, g, seed=K + N)
    bias = (np.arange(N, dtype=np.float32) % 9 - 4) * np.float32(0.25)
    layer = layer_of(trip, pack_dim, dt, bias, bits=bits_of_kind(kind))
    w0 = dense(kind, trip, dt)
    rng = np.random.default_rng(K)
    seen = set()
    for m in (17, 32, 33, 48, 49, 64, 65, 100, 600):
        print(f"[case] pk4 spread {kind} {dtn} K={K} g={g} m={m}", flush=True)
        x = rng.standard_normal((m, K)).astype(np.float32)
        xd = to_dev(x, TORCH_DT[dt])
        y = layer.forward(xd)
        plan = ops.default_context().last_plan()
        seen.add(plan["kernel"].rsplit("_", 1)[1] if "_by" in plan["kernel"] else "")
        w = w0 if "_gs" in plan["kernel"] else oracle.round_through(w0, dt)
        assert_close(y, oracle.matmul_nt_f32(round_x(x, dt), w, bias), f"pk4 spread {kind} {dtn} m{m} {plan['kernel']}")
        if plan["kernel"].startswith(("pk4_mfma", "pk8_mfma")):
            tune("OXQ_PK4_KS", plan["split_k"])  # a workgroup with all the row tiles
            tune("OXQ_PK4_GEMM_MIN_M", 0)
            assert np.array_equal(bits_of(layer.forward(xd)), bits_of(y)), plan
            assert "_by" not in ops.default_context().last_plan()["kernel"]
            tune("OXQ_PK4_KS", None)
            tune("OXQ_PK4_GEMM_MIN_M", None)
    assert "by1" in seen
