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


@pytest.mark.parametrize("K,N,slices", [(1024, 512, 1), (2048, 192, 1), (3072, 64, 3), (3712, 256, 3), (8192, 128, 8)])
@pytest.mark.parametrize("bits,dtn", [(4, "f16"), (4, "bf16"), (8, "f16"), (8, "bf16")])
def test_one_row_beside_the_dot_product_kernel(K, N, slices, bits, dtn):
    """The kernel that one row has by default beside the one it had: the same infinities and NaN, no further from 64 bits (the
    outputs of both are rounded to 16 bits: 2^-12 / 2^-9 of the 2-norm at the most, which the sums' own order moves by 2 % of it)."""
    dt, tdt = DT[dtn]
    q, z, s = synth.gptq_checkpoint(K, N, 128, bits, seed=K + N + bits)
    w = torch.from_numpy(oracle.dequantize_gptq(q, z, oracle.round_through(s, dt), bits)).cuda().double()  # [N, K]
    args = to_dev(q), to_dev(z), to_dev(s, tdt)
    former = ops.Context()
    tune("OXQ_GPTQ_TILE", 0, former)
    x = to_dev(np.random.default_rng(K).standard_normal((1, K)).astype(np.float32), tdt)
    print(f"[case] gptq {bits} {dtn} {K}x{N} one row", flush=True)
    y, o = ops.gptq_matmul(x, *args, bits), ops.gptq_matmul(x, *args, bits, ctx=former)
    plan = ops.default_context().last_plan()
    assert ("tile" in plan["kernel"]) == (bits == 4 or K != 3072 and K != 3712) and "gemv_fast" in former.last_plan()["kernel"], plan
    assert "tile" not in plan["kernel"] or plan["split_k"] == slices, plan
    ref = x.double() @ w.T
    e, f = (((v.double() - ref).norm() / ref.norm()).item() for v in (y, o))
    assert e <= max(1.02 * f, 2.0 ** (-12 if dtn == "f16" else -9)), (e, f)
    for value in ("inf", "-inf", "nan"):
        xi = x.clone()
        xi[0, K - 51] = float(value)
        y, o = ops.gptq_matmul(xi, *args, bits), ops.gptq_matmul(xi, *args, bits, ctx=former)
        assert torch.equal(y.isnan(), o.isnan()) and torch.equal(y.isinf(), o.isinf()), (K, N, value)
