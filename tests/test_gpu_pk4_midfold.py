"""Layers of unrounded weights in workgroups of 64 rows and two strips, K over four waves, against the oracle's unrounded product
with the tolerance of the other forms."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune
from tests.test_gpu_pk4_fine import build

pytestmark = pytest.mark.gpu


# fewer blocks than waves, K that ends in a block's first and second half and between, a ragged round; one strip, a last workgroup of
# one strip, columns that end inside a strip
@pytest.mark.parametrize("kind,bits", [("gptq", 4), ("gptq", 8), ("awq", 8)])
@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("K,N,g", [(128, 2056, 128), (64, 4096, 64), (1216, 328, 64), (96, 2760, 32), (1376, 192, 32), (4256, 64, 32),
                                   (1280, 328, 128)])
def test_against_the_unrounded_product(kind, bits, dtn, K, N, g):
    dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
    rng = np.random.default_rng(K + N + g)
    bias = (np.arange(N, dtype=np.float32) % 9 - 4) * np.float32(0.25)
    layer, args, w = build(kind, bits, K, N, g, dt, tdt, K + bits, bias)
    assert layer.prepacked
    x = rng.standard_normal((200, K)).astype(np.float32)
    xd = to_dev(x, tdt)
    ref = oracle.matmul_nt_f32(round_x(x, dt), w, bias)
    tune("OXQ_PK4_GEMM_KS", 4)
    first = None
    for m in (200, 65, 127, 129):
        print(f"[case] unrounded two strips {kind}{bits} {dtn} {K}x{N} g={g} m={m}", flush=True)
        y = layer.forward(xd[:m])
        plan = ops.default_context().last_plan()
        assert plan["kernel"].endswith("_r64x2k4_gs") and plan["grid"][0] == -(-m // 64) * -(-N // 128), plan
        assert_close(y, ref[:m], f"{plan['kernel']} m{m}")
        first = bits_of(y) if first is None else first
        np.testing.assert_array_equal(bits_of(y), first[:m])
