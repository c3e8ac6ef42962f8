"""The prefill kernel's workgroups of 128 rows (two strips a wave) at the edges of their tiles."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune

pytestmark = pytest.mark.gpu

WIDE, PAIRS = 8, 2  # OXQ_GGUF_GEMM_KS: 256 columns; 128 columns, K over two waves
NAME = {WIDE: "_r128x8", PAIRS: "_r128x4k2"}
FMTS = [synth.GGUF_Q4_K, synth.GGUF_Q8_0, synth.GGUF_Q5_1, synth.GGUF_Q6_K, synth.GGUF_Q2_K, synth.GGUF_Q3_K]


# columns: part of a workgroup's, one live wave of its last, a last strip of eight; chunks of 128 of K: fewer than waves that
# share them, both ring halves, an odd round at the end; rows: one, a tile less and more one, whole bands of row tiles
@pytest.mark.parametrize("fmt,N,K", [(f, n, k) for f in FMTS[:4] for n, k in ((64, 256), (288, 768), (1032, 1280))] +
                         [(f, 1040, 1280) for f in FMTS[4:]] + [(f, 4176, 256) for f in FMTS[4:]])  # (smaller ones of these have no such copy)
def test_rows_at_the_edges(fmt, N, K):
    name = synth.GGUF_NAMES[fmt]
    data = synth.gguf_weight(fmt, N, K, seed=N + K + fmt)
    bias = ((np.arange(N, dtype=np.float32) % 13) - 6) * np.float32(0.25)
    layer = ops.QLinear(fmt, to_dev(data), K, N, to_dev(bias, torch.bfloat16), torch.bfloat16)
    w = oracle.round_through(oracle.dequantize_gguf(fmt, data, N, K), oracle.BF16)
    x = np.random.default_rng(K + N).standard_normal((1100, K)).astype(np.float32)
    xd = to_dev(x, torch.bfloat16)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w, round_x(bias, oracle.BF16))
    for form in (WIDE, PAIRS):
        tune("OXQ_GGUF_GEMM_KS", form)
        first = None
        for m in (1100, 33, 127, 128, 129, 300):
            print(f"[case] gguf 128 rows {name} N={N} K={K} m={m} form={form}", flush=True)
            y = layer.forward(xd[:m])
            plan = ops.default_context().last_plan()
            assert plan["kernel"].endswith(NAME[form]) and plan["launches"] == 1, plan
            assert_close(y, ref[:m], f"gguf 128 rows {name} m={m}", bf16_out=True)
            if first is None:
                first = bits_of(y)
            np.testing.assert_array_equal(bits_of(y), first[:m])


@pytest.mark.parametrize("fmt", FMTS[:4])
@pytest.mark.parametrize("form", [WIDE, PAIRS])
def test_fused_activation(fmt, form):
    """The same bits as the plain layer in the same form, then the activation; 160 gate columns leave two live waves."""
    K, I = 1024, 160
    wd = to_dev(synth.gguf_weight(fmt, 2 * I, K, seed=I + fmt))
    bias = to_dev(((np.arange(2 * I, dtype=np.float32) % 9) - 4) * np.float32(0.5), torch.bfloat16)
    xd = to_dev(np.random.default_rng(5).standard_normal((150, K)).astype(np.float32), torch.bfloat16)
    tune("OXQ_GGUF_GEMM_KS", form)
    plain = ops.QLinear(fmt, wd, K, 2 * I, bias, torch.bfloat16)
    fused = ops.QLinear(fmt, wd, K, 2 * I, bias, torch.bfloat16, gate_up_act=ops.ACT_GATED_SILU)
    for m in (40, 150):
        y = fused.forward(xd[:m])
        assert ops.default_context().last_plan()["kernel"].endswith(NAME[form] + "_silu")
        np.testing.assert_array_equal(bits_of(y), bits_of(ops.gated_activation(plain.forward(xd[:m]), ops.ACT_GATED_SILU)))


def test_slices():
    """A down projection of few columns: 128 rows and columns, K in slices of workgroups that a second launch adds."""
    fmt, N, K, m = synth.GGUF_Q6_K, 520, 8192, 520
    data = synth.gguf_weight(fmt, N, K, seed=3)
    layer = ops.QLinear(fmt, to_dev(data), K, N, None, torch.bfloat16)
    x = np.random.default_rng(4).standard_normal((m, K)).astype(np.float32)
    y = layer.forward(to_dev(x, torch.bfloat16))
    plan = ops.default_context().last_plan()
    print(f"[case] gguf 128 rows in slices {plan['kernel']}", flush=True)
    ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), oracle.round_through(oracle.dequantize_gguf(fmt, data, N, K), oracle.BF16))
    assert_close(y, ref, plan["kernel"], bf16_out=True)
    assert f"{NAME[PAIRS]}_s" in plan["kernel"] and plan["split_k"] > 1 and plan["launches"] == 2, plan


@pytest.mark.parametrize("fmt,K,I,m,act,biased", [(synth.GGUF_Q4_K, 8192, 2048, 300, ops.ACT_GATED_SILU, True), (synth.GGUF_Q4_K, 8192, 1024, 777, ops.ACT_GATED_GELU_TANH, False),
                                                  (synth.GGUF_Q8_0, 8192, 1056, 333, ops.ACT_GATED_SILU, True), (synth.GGUF_Q4_K, 6144, 5376, 74, ops.ACT_GATED_SILU, False)])
def test_fused_activation_where_the_plain_layer_takes_slices(fmt, K, I, m, act, biased):
    """No form forced: fused layer and FeedForward give the plain layer's bits and the activation's."""
    wd = to_dev(synth.gguf_weight(fmt, 2 * I, K, seed=I + fmt))
    bias = to_dev(((np.arange(2 * I, dtype=np.float32) % 9) - 4) * np.float32(0.5), torch.bfloat16) if biased else None
    xd = to_dev(np.random.default_rng(7).standard_normal((m, K)).astype(np.float32), torch.bfloat16)
    plain = ops.QLinear(fmt, wd, K, 2 * I, bias, torch.bfloat16)
    fused = ops.QLinear(fmt, wd, K, 2 * I, bias, torch.bfloat16, gate_up_act=act)
    both = plain.forward(xd)
    plan = ops.default_context().last_plan()
    print(f"[case] gguf fused slices {plan['kernel']} m={m}", flush=True)
    assert "_gemm_bf16" in plan["kernel"] and plan["split_k"] > 1, plan
    want = ops.gated_activation(both, act)
    room = torch.full((m * I + 5,), 7.0, dtype=torch.bfloat16, device="cuda")
    for out in (None, room[1:1 + m * I].view(m, I)):  # (the second one begins off 8 bytes)
        y = fused.forward(xd, out=out)
        got = ops.default_context().last_plan()
        assert got["split_k"] == plan["split_k"] and got["launches"] == 2 and got["grid"] == plan["grid"], got
        np.testing.assert_array_equal(bits_of(y), bits_of(want))
    assert room[0].item() == 7.0 and (room[1 + m * I:] == 7.0).all()
    if I % 256 == 0:
        down = ops.QLinear(fmt, to_dev(synth.gguf_weight(fmt, 512, I, seed=3)), I, 512, None, torch.bfloat16)
        ffn = ops.FeedForward(ops.GATE_UP_FUSED, fused, None, down, I, act)
        np.testing.assert_array_equal(bits_of(ffn.forward(xd)), bits_of(down.forward(want)))


def test_op_keeps_whole_sums():
    """The op's copy lies in the workspace, where the partial sums of slices would go: such a call takes whole sums, where the
    layer, whose copy is its own, takes slices."""
    fmt, N, K, m = synth.GGUF_Q4_K, 1056, 8192, 1100
    data = synth.gguf_weight(fmt, N, K, seed=8)
    wd, xd = to_dev(data), to_dev(np.random.default_rng(9).standard_normal((m, K)).astype(np.float32), torch.bfloat16)
    layer = ops.QLinear(fmt, wd, K, N, None, torch.bfloat16)
    y = layer.forward(xd)
    assert ops.default_context().last_plan()["split_k"] > 1
    z = ops.gguf_quant_mul_mm(xd, wd, K, N, fmt)
    plan = ops.default_context().last_plan()
    print(f"[case] op {plan}", flush=True)
    assert plan["split_k"] == 1 and "gemm_bf16" in plan["kernel"], plan
    w = oracle.round_through(oracle.dequantize_gguf(fmt, data, N, K), oracle.BF16)
    ref = oracle.matmul_nt_f32(round_x(xd.float().cpu().numpy(), oracle.BF16), w)
    for out in (y, z):
        assert_close(out, ref, "op and layer", bf16_out=True)


# these forms store groups of four columns where rows of y begin on 8 bytes
@pytest.mark.parametrize("form", [WIDE, PAIRS])
@pytest.mark.parametrize("act", [None, ops.ACT_GATED_SILU])
def test_outputs_off_the_8_byte_grid(form, act):
    """Columns that are no multiple of four, an output that begins 2 bytes later: a value at a time, the same bits."""
    fmt, N, K, m = synth.GGUF_Q4_K, 1152, 1024, 70
    data = synth.gguf_weight(fmt, N, K, seed=11)
    xd = to_dev(np.random.default_rng(12).standard_normal((m, K)).astype(np.float32), torch.bfloat16)
    bias = to_dev(((np.arange(N, dtype=np.float32) % 7) - 3) * np.float32(0.5), torch.bfloat16)
    tune("OXQ_GGUF_GEMM_KS", form)
    y = ops.QLinear(fmt, to_dev(data), K, N, bias, torch.bfloat16, gate_up_act=act).forward(xd)
    cols = y.shape[1]
    room = torch.full((m * cols + 5,), 7.0, dtype=torch.bfloat16, device="cuda")
    out = room[1:1 + m * cols].view(m, cols)
    ops.QLinear(fmt, to_dev(data), K, N, bias, torch.bfloat16, gate_up_act=act).forward(xd, out=out)
    assert "_gemm_bf16" in ops.default_context().last_plan()["kernel"]
    np.testing.assert_array_equal(bits_of(out), bits_of(y))
    assert room[0].item() == 7.0 and (room[1 + m * cols:] == 7.0).all()
    if act is None:
        less = data.reshape(N, -1)[:N - 6].reshape(-1)
        z = ops.QLinear(fmt, to_dev(less.copy()), K, N - 6, bias[:N - 6].contiguous(), torch.bfloat16).forward(xd)
        np.testing.assert_array_equal(bits_of(z), bits_of(y)[:, :N - 6])
