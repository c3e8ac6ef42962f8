"""Resident 4-bit AWQ layers whose columns end inside a strip, at the rows and lengths of K of the one-tile kernel: the last strip
was not launched, its columns kept what the output held before."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, resident_rounds_weights, round_x, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("K,N", [(4096, 328), (5120, 1096)])
def test_columns_that_end_inside_a_strip(dtn, K, N):
    dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
    q, z, s = synth.awq_checkpoint(K, N, 128, 4, seed=K + N)
    w = oracle.round_through(oracle.dequantize_awq(q, z, oracle.round_through(s, dt)), dt)
    layer = ops.PackedQuantLinear(4, ops.PACK_OUT, to_dev(q), to_dev(z), to_dev(s, tdt), None, tdt)
    x = np.random.default_rng(N).standard_normal((64, K)).astype(np.float32)
    for m in (49, 57, 64):
        print(f"[case] ragged {dtn} {K}x{N} m={m}", flush=True)
        assert resident_rounds_weights(m, dt, False)
        y = torch.full((m, N), float("nan"), dtype=tdt, device="cuda")
        layer.forward(to_dev(x[:m], tdt), out=y)
        assert_close(y, oracle.matmul_nt_f32(round_x(x[:m], dt), w), f"{ops.default_context().last_plan()['kernel']} m{m}")
