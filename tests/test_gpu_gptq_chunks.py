"""gptq_tile_kernel by the blocks of K a wave has: straight-line code for one to five, waves with fewer or none, the loops for even and
odd numbers; K slices whose last one is shorter; more than one round of workgroups.

Up to 32 rows the weights are unrounded, above rounded to x's type: the oracle of either, at the tolerances of the other GPTQ tests."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, round_x, to_dev, tune

pytestmark = pytest.mark.gpu
DT = {"f16": (oracle.F16, torch.float16), "bf16": (oracle.BF16, torch.bfloat16)}


def check(K, N, bits, dtn, rows, slices):
    dt, tdt = DT[dtn]
    q, z, s = synth.gptq_checkpoint(K, N, 128, bits, seed=K + N + bits)
    w = oracle.dequantize_gptq(q, z, oracle.round_through(s, dt), bits)
    wr = oracle.round_through(w, dt)
    args = to_dev(q), to_dev(z), to_dev(s, tdt)
    x = np.random.default_rng(K + bits).standard_normal((max(rows), K)).astype(np.float32)
    xr, xd = round_x(x, dt), to_dev(x, tdt)
    tune("OXQ_GPTQ_TILE", 2)
    for ks in slices:
        tune("OXQ_GPTQ_TILE_KS", ks)
        for m in rows:
            print(f"[case] gptq {bits} {dtn} {K}x{N} rows {m} slices {ks}", flush=True)
            y = ops.gptq_matmul(xd[:m], *args, bits) if m <= 8 else ops.mpp_quant_matmul(xd[:m], *args, bits, ops.PACK_IN)
            plan = ops.default_context().last_plan()
            assert f"gptq{bits}_tile_{dtn}_mt{1 if m <= 16 else 2 if m <= 32 else 4}" == plan["kernel"] and plan["split_k"] == ks, plan
            assert_close(y, oracle.matmul_nt_f32(xr[:m], w if m <= 32 else wr), f"{plan['kernel']} K={K} m={m} slices {ks}")


@pytest.mark.parametrize("blocks", [1, 2, 7, 8, 9, 15, 16, 17, 24, 25, 28, 32, 33, 36, 40, 41, 48, 50, 56, 57])
@pytest.mark.parametrize("bits,dtn", [(4, "f16"), (4, "bf16"), (8, "f16"), (8, "bf16")])
def test_blocks_of_a_wave(blocks, bits, dtn):
    check(128 * blocks, 128, bits, dtn, (3, 16, 20, 40), (1,) if blocks < 24 else (1, 3))


@pytest.mark.parametrize("blocks", [8, 16, 18, 26, 34])  # one, two, three, four and five blocks a wave; 257 strips
@pytest.mark.parametrize("bits,dtn", [(4, "f16"), (8, "bf16")])
def test_more_than_a_round_of_workgroups(blocks, bits, dtn):
    check(128 * blocks, 64 * 257, bits, dtn, (2, 24, 40), (1,))
