"""Resident layers with quantization groups of 32 or 64 rows, K that ends inside a block of 128 rows and N that ends
inside a strip of 64 columns: dense dequant bit for bit, products against the oracle.

Tolerance as in the other parity tests, 2e-3 relative / 1e-2 absolute on the f32-accumulated product (bf16 outputs
plus their own half ulp); the reference rounds the weights where the resident layers do (test helper)."""
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
        wr = oracle.round_through(w, dt) if resident_rounds_weights(m, dt, kind == "gptq") else w
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
    for dtn, bits, K, N, g in [("f16", 4, 672, 1096, 32), ("bf16", 8, 1088, 584, 64)]:
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
        wr = oracle.round_through(w, dt) if resident_rounds_weights(m, dt, kind == "gptq") else w
        assert_close(y, oracle.matmul_nt_f32(round_x(x, dt), wr), f"{kind}{bits} m{m}")
