"""Resident layers with quantization groups of 32 or 64 rows, K that ends inside a block of 128 rows and N that ends
inside a strip of 64 columns: dense dequant bit for bit, products against the oracle.

Tolerance as in the other parity tests, 2e-3 relative / 1e-2 absolute on the f32-accumulated product (bf16 outputs
plus their own half ulp).  The reference rounds the weights of 4-bit AWQ layers where the resident layers do (test helper);
those of GPTQ and 8-bit AWQ layers of these shapes are never rounded."""
import sys

import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, resident_rounds_weights, round_x, to_dev

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def build(kind, bits, K, N, g, dt, tdt, seed, bias=None):
    gptq = kind == "gptq"
    qw, qz, sc = (synth.gptq_checkpoint if gptq else synth.awq_checkpoint)(K, N, g, bits, seed=seed)[:3]
    s_r = oracle.round_through(sc, dt)
    if gptq:
        w = oracle.dequantize_gptq(qw, qz, s_r, bits)
    else:
        w = oracle.dequantize_awq(qw, qz, s_r) if bits == 4 else oracle.dequantize_awq8(qw, qz, s_r)
    args = (to_dev(qw), to_dev(qz), to_dev(sc, tdt))
    layer = ops.PackedQuantLinear(bits, ops.PACK_IN if gptq else ops.PACK_OUT, *args,
                                  None if bias is None else to_dev(bias, tdt), tdt)
    return layer, args, w


def rounds(kind, bits, m, dt):
    return (kind, bits) == ("awq", 4) and resident_rounds_weights(m, dt, False)


def correctly_rounded_share(y, x, w, dt, tdt, bias=None):
    """Share of outputs that are the 64-bit product rounded once to the output type.  The f32 sums of unrounded weights
    move one over a rounding boundary in 0.1 - 3 % of the cases (bias of the folded integers against the result's ulp);
    weights rounded to the type miss it in 40 %."""
    ref = round_x(x, dt).astype(np.float64) @ w.astype(np.float64).T
    if bias is not None:
        ref = ref + round_x(bias, dt)
    return (y.cpu() == torch.from_numpy(ref).to(tdt)).double().mean().item()


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("kind,bits", [("awq", 8), ("gptq", 4), ("gptq", 8)])
@pytest.mark.parametrize("K,N,g", [(1024, 256, 32), (1088, 328, 64), (1024, 328, 128), (672, 1096, 32), (2048, 264, 256)])
def test_weights_stay_unrounded(kind, bits, K, N, g, dtn):
    """GPTQ and 8-bit AWQ layers of these shapes and the stateless tile op on their tensors, in every form: one and two
    row tiles of the ring kernel, the prefill kernel at whole and ragged tiles of 64 rows, an unfilled group of strips."""
    dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
    rng = np.random.default_rng(K + N + g + bits)
    layer, args, w = build(kind, bits, K, N, g, dt, tdt, K + bits)
    assert layer.prepacked
    for m in (16, 17, 32, 33, 48, 49, 64, 65, 128, 200, 700):
        x = rng.standard_normal((m, K)).astype(np.float32)
        y = layer.forward(to_dev(x, tdt))
        kernel = ops.default_context().last_plan()["kernel"]
        say(f"unrounded {kind}{bits} {dtn} {K}x{N} g={g} m={m} {kernel}")
        share = correctly_rounded_share(y, x, w, dt, tdt)
        assert share > 0.9, f"{kernel}: {share:.3f} of the outputs correctly rounded"
        if m in (17, 200):
            y = ops.mpp_quant_matmul(to_dev(x, tdt), *args, bits, ops.PACK_IN if kind == "gptq" else ops.PACK_OUT)
            share = correctly_rounded_share(y, x, w, dt, tdt)
            assert share > 0.9, f"stateless, {ops.default_context().last_plan()['kernel']}: {share:.3f}"


@pytest.mark.parametrize("kind", ["awq", "gptq"])
def test_fused_activation_is_that_of_the_plain_layer(kind):
    """The gate|up epilogue of the folded prefill form and of the ring kernel: the plain layer's bits."""
    K, N, m_all, tdt = 1088, 1152, (17, 64, 65, 130), torch.bfloat16
    _, args, _ = build(kind, 8, K, N, 64, oracle.BF16, tdt, 11)
    pack = ops.PACK_IN if kind == "gptq" else ops.PACK_OUT
    fused = ops.PackedQuantLinear(8, pack, *args, None, tdt, gate_up_act=ops.ACT_GATED_SILU)
    plain = ops.PackedQuantLinear(8, pack, *args, None, tdt)
    for m in m_all:
        say(f"fused activation {kind}8 m={m}")
        x = to_dev(np.random.default_rng(m).standard_normal((m, K)).astype(np.float32) * 0.25, tdt)
        np.testing.assert_array_equal(bits_of(fused.forward(x)), bits_of(ops.gated_activation(plain.forward(x), ops.ACT_GATED_SILU)))


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("kind,bits", [("awq", 4), ("awq", 8), ("gptq", 4), ("gptq", 8)])
@pytest.mark.parametrize("K,N,g", [(1024, 256, 32), (1024, 264, 64), (672, 520, 32), (1088, 328, 64), (1024, 328, 128)])
def test_fine_groups_and_ragged_edges(kind, bits, K, N, g, dtn):
    dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
    say(f"fine {kind}{bits} {dtn} {K}x{N} g={g}")
    rng = np.random.default_rng(K + N + g)
    bias = (np.arange(N, dtype=np.float32) % 9 - 4) * np.float32(0.25)
    layer, args, w = build(kind, bits, K, N, g, dt, tdt, K + bits, bias)
    assert layer.prepacked
    want = oracle.transpose_convert(w, dt)
    np.testing.assert_array_equal(bits_of(layer.dequantize()), want)
    # row tiles 1 - 4 and their edges, then both prefill forms (two strips with K split, eight strips of 64 / 128 rows)
    for m in (1, 4, 5, 9, 16, 17, 33, 49, 64, 65, 130, 700):
        x = rng.standard_normal((m, K)).astype(np.float32)
        xd = to_dev(x, tdt)
        wr = oracle.round_through(w, dt) if rounds(kind, bits, m, dt) else w
        ref = oracle.matmul_nt_f32(round_x(x, dt), wr, bias)
        y = layer.forward(xd)
        kernel = ops.default_context().last_plan()["kernel"]
        assert_close(y, ref, f"{kind}{bits} m{m} {K}x{N} g{g} {kernel}")
        if m in (1, 65):  # rows at an address that is no multiple of 16
            off = torch.empty(m * K + 1, dtype=tdt, device="cuda")
            off[1:] = xd.reshape(-1)
            out = torch.full((m * N + 1,), float("nan"), dtype=tdt, device="cuda")
            layer.forward(off[1:].view(m, K), out=out[1:].view(m, N))
            assert_close(out[1:].view(m, N), ref, f"staged {kind}{bits} m{m} {K}x{N} g{g}")
            assert torch.isnan(out[0])


@pytest.mark.parametrize("tune_rows", [64, 128])
def test_fine_prefill_forms(tune_rows):
    """The eight-strip forms, forced: an unfilled last group of strips, K inside a block, every row-tile remainder class."""
    from tests.helpers import tune
    for dtn, bits, K, N, g in [("f16", 4, 672, 1096, 32), ("bf16", 4, 1088, 584, 64)]:
        dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
        layer, _, w = build("awq", bits, K, N, g, dt, tdt, 7)
        tune("OXQ_PK4_GEMM_ROWS", tune_rows)
        for m in (65, 127, 129):
            say(f"fine prefill {dtn} pk{bits} m={m} rows={tune_rows}")
            x = np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)
            y = layer.forward(to_dev(x, tdt))
            assert f"_r{tune_rows}x8" in ops.default_context().last_plan()["kernel"]
            assert_close(y, oracle.matmul_nt_f32(round_x(x, dt), oracle.round_through(w, dt)), f"m{m}")


@pytest.mark.parametrize("kind,bits,K,N,g", [("awq", 8, 1024, 264, 32), ("gptq", 4, 672, 520, 32), ("gptq", 8, 1088, 328, 64)])
def test_stateless_op_on_fine_groups(kind, bits, K, N, g):
    """The tile op builds the tile-major copy in the workspace for shapes without a checkpoint-layout tile kernel."""
    for dtn, m in (("f16", 9), ("bf16", 70)):
        dt, tdt = (oracle.F16, torch.float16) if dtn == "f16" else (oracle.BF16, torch.bfloat16)
        say(f"stateless {kind}{bits} {dtn} m={m} {K}x{N} g={g}")
        _, args, w = build(kind, bits, K, N, g, dt, tdt, 3)
        x = np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)
        y = ops.mpp_quant_matmul(to_dev(x, tdt), *args, bits, ops.PACK_IN if kind == "gptq" else ops.PACK_OUT)
        wr = oracle.round_through(w, dt) if rounds(kind, bits, m, dt) else w
        assert_close(y, oracle.matmul_nt_f32(round_x(x, dt), wr), f"{kind}{bits} m{m}")


def test_rows_beyond_32_bit_offsets():
    """x of more than 2 GiB on an unrounded layer: only the prefill form addresses it, whatever the cost rule says."""
    K, N, g, tdt = 4096, 136, 64, torch.float16
    m = (1 << 31) // (2 * K) + 65
    layer, _, w = build("gptq", 4, K, N, g, oracle.F16, tdt, 5)
    say(f"unrounded, {m} rows")
    x = torch.randn((1024, K), device="cuda").to(tdt).repeat((m + 1023) // 1024, 1)[:m]
    y = layer.forward(x)
    assert "_gemm_f16_r64x8_gs" in ops.default_context().last_plan()["kernel"]
    assert torch.equal(y[1024:2048], y[:1024]) and torch.equal(y[m - 65:], y[(m - 65) % 1024:][:65])
    ref = x[:64].cpu().numpy().astype(np.float64) @ w.astype(np.float64).T
    assert (y[:64].cpu() == torch.from_numpy(ref).to(tdt)).double().mean().item() > 0.9
