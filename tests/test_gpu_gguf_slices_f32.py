"""The matrix-core copy of GGUF layers beyond bf16 decode: f32 activations (three bf16 pieces a value), prefill rows of
layers of few columns (K slices over workgroups, added by a second launch) and rows that end inside a strip of 16.

f32: against the product in float64.  A value, a weight's integer and their product are exact; what rounds is f32
addition: per output a chain of at most 32 products, 4 - 8 steps a chunk, 14 chunks a wave and 8 waves (K = 14336), each
rounding by at most 2^-24 of sums that the operand's bias makes up to four times as large as the result.  As a random walk
that is about 4 x 2^-24 x sqrt(2) = 3.4e-7 of the 2-norm at the worst, and never more than the vector kernels' own error.
bf16: 2e-3 relative / 1e-2 absolute against the oracle with the weights rounded as the prefill tiles round them."""
import sys

import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune

pytestmark = pytest.mark.gpu
FMTS = [synth.GGUF_Q4_0, synth.GGUF_Q8_0, synth.GGUF_Q4_K, synth.GGUF_Q6_K, synth.GGUF_Q4_1, synth.GGUF_Q5_0,
        synth.GGUF_Q5_1, synth.GGUF_Q5_K]


def say(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N,K", [(1024, 1024), (1032, 2304), (144, 8192), (12296, 256), (12352, 256)])  # 12352: four strips a workgroup
def test_f32_rows_on_the_matrix_core_copy(fmt, N, K):
    data = synth.gguf_weight(fmt, N, K, seed=N + K + fmt)
    w = oracle.dequantize_gguf(fmt, data, N, K)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    layer = ops.QLinear(fmt, to_dev(data), K, N, to_dev(bias), torch.float32)
    assert layer.resident
    assert np.array_equal(layer.dequantize().cpu().numpy().view(np.uint32), w.view(np.uint32)), "repack changed a weight"
    for m in (1, 3, 4, 5, 8, 9, 21):
        say(f"gguf f32 matrix cores {synth.GGUF_NAMES[fmt]} N={N} K={K} m={m}")
        x = np.random.default_rng(K + m).standard_normal((m, K)).astype(np.float32)
        y = layer.forward(to_dev(x))
        kernel = ops.default_context().last_plan()["kernel"]
        assert ("_mfma_f32" if m >= 3 or N % 16 else "_f32") in kernel and kernel.endswith("_n64") == (N == 12352), kernel
        ref = x.astype(np.float64) @ w.astype(np.float64).T + bias
        err = np.linalg.norm(y.cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err < 4e-7, f"{synth.GGUF_NAMES[fmt]} m={m}: {err:.2e}"
        assert np.array_equal(bits_of(layer.forward(to_dev(x))), bits_of(y)), "run to run"


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N,K", [(1024, 14336), (1032, 4096), (1024, 1024)])
def test_f32_rows_are_no_further_from_64_bits_than_the_vector_kernels(fmt, N, K):
    """Against the layer without the matrix-core copy (rotated copy up to 8 rows, the file layout above): the 2-norm error over
    3 N outputs and more (ratios measured over six draws: 0.3 - 0.93; one draw scatters by a few per cent)."""
    data = to_dev(synth.gguf_weight(fmt, N, K, seed=N + K + fmt))
    plain = ops.Context()
    tune("OXQ_GGUF_MFMA", 0, plain)
    layer, former = ops.QLinear(fmt, data, K, N, None, torch.float32), ops.QLinear(fmt, data, K, N, None, torch.float32, ctx=plain)
    w = layer.dequantize().double()
    for m in (3, 8, 9, 21):
        say(f"gguf f32 error {synth.GGUF_NAMES[fmt]} N={N} K={K} m={m}")
        x = to_dev(np.random.default_rng(K + m).standard_normal((m, K)).astype(np.float32))
        ref = x.double() @ w.T
        err, was = [((y.double() - ref).norm() / ref.norm()).item() for y in (layer.forward(x), former.forward(x))]
        assert "_mfma_f32" in layer.ctx.last_plan()["kernel"] and "mfma" not in plain.last_plan()["kernel"]
        assert err <= 1.04 * was, f"{synth.GGUF_NAMES[fmt]} m={m}: {err:.3e}, vector kernel {was:.3e}"


def test_f32_rows_beyond_one_grid():
    """More rows than 65535 row tiles of eight: two launches."""
    fmt, N, K, m = synth.GGUF_Q4_0, 1040, 1024, 65535 * 8 + 9
    layer = ops.QLinear(fmt, to_dev(synth.gguf_weight(fmt, N, K, seed=3)), K, N, None, torch.float32)
    say(f"gguf f32 {m} rows")
    x = torch.randn((4096, K), device="cuda").repeat((m + 4095) // 4096, 1)[:m]
    y = layer.forward(x)
    plan = layer.ctx.last_plan()
    assert "_mfma_f32" in plan["kernel"] and plan["launches"] == 2
    assert torch.equal(y[65536:131072], y[:65536])  # 65536 = 16 x 4096 rows on, the same rows of x in tiles of their own
    tail = torch.arange(m - 9 - 16, m, device="cuda")
    assert torch.equal(y[tail], y[tail % 4096])
    ref = x[:64].double() @ layer.dequantize().double().T
    assert ((y[:64].double() - ref).norm() / ref.norm()).item() < 4e-7


def test_f32_layer_with_one_copy():
    """OXQ_GGUF_MFMA = 2: the matrix-core copy alone, at every row count, and the memory of one copy less."""
    fmt, N, K = synth.GGUF_Q8_0, 4096, 4096
    data = to_dev(synth.gguf_weight(fmt, N, K, seed=9))
    x = to_dev(np.random.default_rng(9).standard_normal((8, K)).astype(np.float32))
    ctx, taken, layers = ops.Context(), [], []
    for value in (2, None):
        tune("OXQ_GGUF_MFMA", value, ctx)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        layers.append(ops.QLinear(fmt, data, K, N, None, torch.float32, ctx=ctx))
        taken.append(before - torch.cuda.mem_get_info()[0])
    copy = 4096 * (4096 // 32) * 34
    assert copy <= taken[0] < 1.3 * copy and 2 * copy <= taken[1] < 2.3 * copy, taken
    for m in (1, 2, 8):
        say(f"gguf f32 one copy m={m}")
        y = layers[0].forward(x[:m])
        assert "_mfma_f32" in ctx.last_plan()["kernel"]
        want = layers[1].forward(x[:m])
        assert ("_mfma_f32" in ctx.last_plan()["kernel"]) == (m > 2)
        assert ((y - want).norm() / want.norm()).item() < 8e-7  # two forms, each within 4e-7 of the 64-bit product


@pytest.mark.parametrize("fmt", FMTS)
def test_small_f32_rows_keep_their_bits(fmt):
    """Rows whose values lie near 1e-36 (one row: 1e-30 beside them): all three pieces of a value count, up to one row."""
    N, K = 1032, 2048  # ragged: the matrix cores take every row count
    layer = ops.QLinear(fmt, to_dev(synth.gguf_weight(fmt, N, K, seed=fmt)), K, N, None, torch.float32)
    w = layer.dequantize().double()
    for m in (1, 3, 8):
        say(f"gguf f32 small values {synth.GGUF_NAMES[fmt]} m={m}")
        x = to_dev(np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)) * 1e-36
        if m > 1:
            x[1] *= 1e6
        ref = x.double() @ w.T
        y = layer.forward(x)
        assert "_mfma_f32" in layer.ctx.last_plan()["kernel"]
        for r in range(m):
            err = ((y[r].double() - ref[r]).norm() / ref[r].norm()).item()
            assert err < 4e-7, f"{synth.GGUF_NAMES[fmt]} m={m} row {r}: {err:.2e}"


@pytest.mark.parametrize("fmt", FMTS)
def test_infinite_and_nan_rows_of_f32(fmt):
    """An infinity, and a NaN whose payload lies in the bits that the first piece drops, give what the vector kernels give and
    stay in their row."""
    N, K = 1024, 2048
    data = to_dev(synth.gguf_weight(fmt, N, K, seed=fmt))
    plain = ops.Context()
    tune("OXQ_GGUF_MFMA", 0, plain)
    layer, former = ops.QLinear(fmt, data, K, N, None, torch.float32), ops.QLinear(fmt, data, K, N, None, torch.float32, ctx=plain)
    for m in (3, 8, 9):
        x = to_dev(np.random.default_rng(m).standard_normal((m, K)).astype(np.float32))
        x[0, 77], x[1, 1500] = float("inf"), -float("inf")
        x.view(torch.int32)[2, 5] = 0x7F800001
        say(f"gguf f32 infinities {synth.GGUF_NAMES[fmt]} m={m}")
        got, want = layer.forward(x), former.forward(x)
        assert "_mfma_f32" in layer.ctx.last_plan()["kernel"]
        assert torch.equal(torch.nan_to_num(got[:3], 0.0, 1.0, -1.0), torch.nan_to_num(want[:3], 0.0, 1.0, -1.0))
        assert bool(got[2].isnan().all()) and bool(got[3:].isfinite().all())
        if fmt in (synth.GGUF_Q4_1, synth.GGUF_Q5_1):
            assert got[0].isinf().sum() > N // 2 and got[1].isinf().sum() > N // 2


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N,K", [(256, 4096), (1032, 2304), (640, 14336), (4100, 1024)])
def test_prefill_rows_of_few_columns(fmt, N, K):
    data = synth.gguf_weight(fmt, N, K, seed=N + K + fmt)
    bias = ((np.arange(N, dtype=np.float32) % 13) - 6) * np.float32(0.25)
    layer = ops.QLinear(fmt, to_dev(data), K, N, to_dev(bias, torch.bfloat16), torch.bfloat16)
    assert layer.resident
    w = oracle.dequantize_gguf(fmt, data, N, K)
    wr = oracle.round_through(w, oracle.BF16)
    for m, slices in ((33, None), (64, 2), (65, None), (200, 3), (300, None)):
        tune("OXQ_GGUF_GEMM_SLICES", slices)
        x = np.random.default_rng(K + m).standard_normal((m, K)).astype(np.float32)
        y = layer.forward(to_dev(x, torch.bfloat16))
        plan = ops.default_context().last_plan()
        say(f"gguf slices {synth.GGUF_NAMES[fmt]} N={N} K={K} m={m} {plan['kernel']} x {plan['split_k']}")
        whole = "_mfma_bf16_mt2" in plan["kernel"]  # row tiles of the integer kernel: the weights unrounded
        assert plan["launches"] == (2 if plan["split_k"] > 1 else 1) and (slices is None or plan["split_k"] > 1), plan
        assert whole or "_gemm_bf16_r" in plan["kernel"], plan
        ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w if whole else wr, round_x(bias, oracle.BF16))
        assert_close(y, ref, f"{synth.GGUF_NAMES[fmt]} m={m}", bf16_out=True)
    for m in (1, 17, 32):  # the integer kernel on a ragged last strip
        x = np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)
        ref = oracle.matmul_nt_f32(round_x(x, oracle.BF16), w, round_x(bias, oracle.BF16))
        assert_close(layer.forward(to_dev(x, torch.bfloat16)), ref, f"m={m}", bf16_out=True)


@pytest.mark.parametrize("fmt", [synth.GGUF_Q4_K, synth.GGUF_Q6_K])
@pytest.mark.parametrize("slices", [2, None])
def test_ffn_without_room_for_the_fused_activation(fmt, slices):
    """A gate|up layer of few columns: the projection runs in K slices on the interleaved copy, its columns put back in
    the file's order, and the activation by itself - the plain layer's bits.  Unforced: row tiles of the integer kernel,
    the activation in its epilogue, again the plain layer's bits."""
    tune("OXQ_GGUF_GEMM_SLICES", slices)
    K, inter, m = 2048, 512, 40
    say(f"gguf ffn slices {synth.GGUF_NAMES[fmt]}")
    gu, dn = synth.gguf_weight(fmt, 2 * inter, K, seed=1), synth.gguf_weight(fmt, K, inter, seed=2)
    fused = ops.QLinear(fmt, to_dev(gu), K, 2 * inter, None, torch.bfloat16, gate_up_act=ops.ACT_GATED_SILU)
    plain = ops.QLinear(fmt, to_dev(gu), K, 2 * inter, None, torch.bfloat16)
    down = ops.QLinear(fmt, to_dev(dn), inter, K, None, torch.bfloat16)
    x = to_dev(np.random.default_rng(3).standard_normal((m, K)).astype(np.float32) * 0.25, torch.bfloat16)
    want = down.forward(ops.gated_activation(plain.forward(x), ops.ACT_GATED_SILU))
    got = ops.FeedForward(ops.GATE_UP_FUSED, fused, None, down, inter).forward(x)
    np.testing.assert_array_equal(bits_of(got), bits_of(want))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N,K,rows", [(1024, 1024, (1, 2)), (592, 1792, (1, 2)), (512, 2048, (2,)), (256, 5376, (1,)), (4112, 3072, (1, 2))])
def test_one_and_two_f32_rows_where_the_matrix_cores_take_them(fmt, N, K, rows):
    """Beside the layer without the matrix-core copy: both within 4e-7 of 64 bits, and not further from it; the same infinities."""
    data = to_dev(synth.gguf_weight(fmt, N, K, seed=N + K + fmt))
    plain = ops.Context()
    tune("OXQ_GGUF_MFMA", 0, plain)
    layer, former = ops.QLinear(fmt, data, K, N, None, torch.float32), ops.QLinear(fmt, data, K, N, None, torch.float32, ctx=plain)
    w = layer.dequantize().double()
    try:
        for m in rows:
            err = []
            for ly, ctx, name in ((layer, ops.default_context(), "_mfma_f32_mt1"), (former, plain, "_res_gemv_f32")):
                x = torch.from_numpy(np.random.default_rng(K + m).standard_normal((m, K)).astype(np.float32)).cuda()
                say(f"gguf f32 {synth.GGUF_NAMES[fmt]} N={N} K={K} m={m} {name}")
                y = ly.forward(x)
                assert name in ctx.last_plan()["kernel"], ctx.last_plan()
                ref = x.double() @ w.T
                err.append(((y.double() - ref).norm() / ref.norm()).item())
            assert err[0] < 4e-7 and err[0] <= 1.1 * err[1], (m, err)  # (a draw of a few hundred outputs scatters by a few per cent)
            x = torch.from_numpy(np.random.default_rng(m).standard_normal((m, K)).astype(np.float32)).cuda()
            x[0, 77], x[m - 1, K - 3] = float("inf"), -float("inf") if m == 2 else 1.0
            got, want = layer.forward(x), former.forward(x)
            assert torch.equal(torch.nan_to_num(got, 0.0, 1.0, -1.0), torch.nan_to_num(want, 0.0, 1.0, -1.0)), "infinities"
    finally:
        plain.close()
