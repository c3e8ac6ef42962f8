"""The ops on checkpoint tensors where their kernel changes: AWQ, one row of ragged columns and bf16 at 9 - 16 rows; AWQ and GPTQ, the rows
from which the tile op builds the tile-major copy for its call."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, resident_rounds_weights, round_x, to_dev

pytestmark = pytest.mark.gpu
DT = {"f16": (oracle.F16, torch.float16), "bf16": (oracle.BF16, torch.bfloat16)}


def tensors(K, N, g, bits, dt, tdt):
    q, z, s = synth.awq_checkpoint(K, N, g, bits, seed=K + N + bits)
    s_r = oracle.round_through(s, dt)
    w = oracle.dequantize_awq(q, z, s_r) if bits == 4 else oracle.dequantize_awq8(q, z, s_r)
    return (to_dev(q), to_dev(z), to_dev(s, tdt)), w


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K,N,g", [(1024, 264, 128), (4096, 1096, 64), (2080, 520, 32), (1280, 8200, 128), (960, 1096, 64), (1024, 1096, 64)])
def test_one_row_of_ragged_columns(dtn, bits, K, N, g):
    """Weights stay unrounded: outputs are the 64-bit product rounded once, but for those next to a boundary."""
    dt, tdt = DT[dtn]
    args, w = tensors(K, N, g, bits, dt, tdt)
    x = np.random.default_rng(K).standard_normal((1, K)).astype(np.float32)
    y = (ops.w4a16_matmul if bits == 4 else ops.w8a16_matmul)(to_dev(x, tdt), *args)
    short = bits == 8 and g == 64 and K < 1024  # the generic kernel
    assert ("_slab" in ops.default_context().last_plan()["kernel"]) != short
    ref = round_x(x, dt).astype(np.float64) @ w.astype(np.float64).T
    assert (y.cpu() == torch.from_numpy(ref).to(tdt)).double().mean().item() > 0.97


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("K,N,g,rows", [(1024, 2048, 128, {"f16": 49, "bf16": 17}), (1088, 2056, 64, {"f16": 49, "bf16": 17}),
                                        (4096, 4104, 128, {"f16": 64, "bf16": 17}), (8224, 2048, 32, {"f16": 65, "bf16": 17}),
                                        (4608, 512, 128, {"f16": 65, "bf16": 17}), (6144, 1032, 128, {"f16": 129, "bf16": 17}),
                                        (9280, 520, 64, {"f16": 129, "bf16": 17}), (7680, 520, 128, {"f16": 193, "bf16": 17})])
def test_rows_at_the_lines_of_the_rule(dtn, K, N, g, rows):
    dt, tdt = DT[dtn]
    args, w = tensors(K, N, g, 4, dt, tdt)
    x = np.random.default_rng(K).standard_normal((200, K)).astype(np.float32)
    xd, wr = to_dev(x, tdt), oracle.round_through(w, dt)
    for m in (9, 16, 17, rows[dtn] - 1, rows[dtn], 200):
        y = ops.mpp_quant_matmul(xd[:m], *args, 4, ops.PACK_OUT)
        plan = ops.default_context().last_plan()
        print(f"[case] awq op {dtn} {K}x{N} g={g} m={m} {plan['kernel']}", flush=True)
        resident = m >= rows[dtn]
        slab = "_slab" in plan["kernel"]
        assert slab == (m <= 16 and dtn == "bf16") and plan["kernel"].startswith("pk4_") == resident, plan
        unrounded = slab or resident and not resident_rounds_weights(m, dt, False)
        assert_close(y, oracle.matmul_nt_f32(round_x(x[:m], dt), w if unrounded else wr), f"m{m} {plan['kernel']}")


# (rows that stay on the tile kernel, rows of a copy): one round of the tile kernel's workgroups, and the row tiles the rule asks for
@pytest.mark.parametrize("bits,dtn,K,N,edges", [
    (4, "f16", 3072, 4096, ((320, 321),)), (4, "f16", 8192, 2048, ((448, 513), (512, 513))), (4, "f16", 4096, 8192, ((320, 321),)),
    (4, "bf16", 4096, 8192, ((192, 193),)), (4, "bf16", 3072, 4032, ((639, 640),)), (8, "f16", 8192, 3072, ((384, 385), (577, 640))),
    (8, "f16", 3072, 4160, ((384, 385), (449, 577))), (8, "bf16", 1920, 6592, ((384, 385),))])
def test_rows_at_the_lines_of_the_gptq_rule(bits, dtn, K, N, edges):
    dt, tdt = DT[dtn]
    q, z, s = synth.gptq_checkpoint(K, N, 128, bits, seed=K + N + bits)
    s_r = oracle.round_through(s, dt)
    w = oracle.round_through(oracle.dequantize_gptq(q, z, s_r, bits), dt)
    x = np.random.default_rng(K).standard_normal((max(m for pair in edges for m in pair), K)).astype(np.float32)
    xd, args = to_dev(x, tdt), (to_dev(q), to_dev(z), to_dev(s, tdt))
    ref = oracle.matmul_nt_f32(round_x(x, dt), w)
    for pair in edges:
        for m, copied in zip(pair, (False, True)):
            y = ops.mpp_quant_matmul(xd[:m], *args, bits, ops.PACK_IN)
            plan = ops.default_context().last_plan()
            print(f"[case] gptq op {bits} {dtn} {K}x{N} m={m} {plan['kernel']}", flush=True)
            assert plan["kernel"].startswith(f"pk{bits}_" if copied else f"gptq{bits}_tile_"), plan
            assert_close(y, ref[:m], f"m{m} {plan['kernel']}")


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("K,N", [(2048, 1032), (1024, 2048)])
def test_an_infinite_row_keeps_its_signs(dtn, K, N):
    """One infinite value of x: infinity times a weight, or NaN where the weight is zero, whichever kernel takes the rows."""
    dt, tdt = DT[dtn]
    args, w = tensors(K, N, 128, 4, dt, tdt)
    col = np.argmin((w == 0).sum(axis=0))
    with np.errstate(invalid="ignore"):
        want = np.where(w[:, col] == 0, np.nan, np.sign(w[:, col]) * np.inf).astype(np.float32)
    for m in (9, 16, 17, 48, 49):
        x = np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)
        x[m - 1, col] = np.inf
        y = ops.mpp_quant_matmul(to_dev(x, tdt), *args, 4, ops.PACK_OUT)
        print(f"[case] infinite row {dtn} {K}x{N} m={m} {ops.default_context().last_plan()['kernel']}", flush=True)
        np.testing.assert_array_equal(y[m - 1].float().cpu().numpy(), want)
        assert bool(torch.isfinite(y[:m - 1]).all())


def test_a_plan_only_context_reports_what_runs():
    """Calls that build a copy of their tensors and calls next to them."""
    plans = ops.Context(plan_only=True)

    def same(name, call, bits_out):
        seen = []
        for ctx in (plans, ops.default_context()):
            call(ctx)
            seen.append({k: v for k, v in ctx.last_plan().items()})
        print(f"[case] plan only {name} {seen[1]['kernel']}", flush=True)
        assert seen[0] == seen[1], name
        assert seen[0]["kernel"].startswith(bits_out), seen[0]

    K, N = 2048, 1024
    for dtn, (dt, tdt) in DT.items():
        args, _ = tensors(K, N, 128, 4, dt, tdt)
        q, z, s = synth.gptq_checkpoint(K, N, 128, 8, seed=1)
        gargs = (to_dev(q), to_dev(z), to_dev(s, tdt))
        for m in (16, 17, 49, 64, 640):
            x = torch.zeros(m, K, dtype=tdt, device="cuda")
            same(f"awq {dtn} {m}", lambda c: ops.mpp_quant_matmul(x, *args, 4, ops.PACK_OUT, ctx=c), ("awq4", "pk4"))
            same(f"gptq {dtn} {m}", lambda c: ops.mpp_quant_matmul(x, *gargs, 8, ops.PACK_IN, ctx=c), ("gptq8", "pk8"))
    wd = to_dev(synth.gguf_weight(synth.GGUF_Q4_K, N, K, seed=2))
    for m in (1023, 1024):
        x = torch.zeros(m, K, dtype=torch.bfloat16, device="cuda")
        same(f"gguf {m}", lambda c: ops.gguf_quant_mul_mm(x, wd, K, N, synth.GGUF_Q4_K, ctx=c), "gguf_q4k_")
