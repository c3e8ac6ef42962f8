"""The checkpoint layouts at few rows on the matrix cores (wna16_slab_kernel): against the oracle's unrounded weights."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import TORCH_DT, assert_close, bits_of, round_x, to_dev, tune

pytestmark = pytest.mark.gpu
DT = {"f16": oracle.F16, "bf16": oracle.BF16}


def call(x, d, bits, m):
    if m > 8:
        return ops.mpp_quant_matmul(x, *d, bits, ops.PACK_OUT)
    return ops.w4a16_matmul(x, *d) if bits == 4 else ops.w8a16_matmul(x, *d)


@pytest.mark.parametrize("bits,K,N,g,ms", [
    (4, 1152, 3080, 128, (2, 3, 8)),      # 64-row runs; the last workgroup 8 columns wide
    (4, 1120, 1032, 32, (1, 4, 5, 8)),    # K ends inside a run; groups inside a run
    (4, 1216, 264, 64, (2, 7)),
    (4, 4096, 6144, 128, (2, 8)),         # 128-row runs
    (4, 5120, 13824, 128, (2,)),          # two runs a wave
    (4, 4064, 8200, 32, (1, 6)),          # K ends inside a run
    (8, 576, 1032, 64, (2, 5, 8)),
    (8, 1120, 1000, 32, (1, 3, 8, 9, 16)),
    (8, 8192, 14336, 128, (2, 16)),       # several runs a wave
])
@pytest.mark.parametrize("dtn", ["f16", "bf16"])
def test_awq_against_the_oracle(bits, K, N, g, ms, dtn):
    dt = DT[dtn]
    qw, qz, sc = synth.awq_checkpoint(K, N, g, bits, seed=K + N)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, TORCH_DT[dt]))
    s = oracle.round_through(sc, dt)
    w = oracle.dequantize_awq(qw, qz, s) if bits == 4 else oracle.dequantize_awq8(qw, qz, s)
    rng = np.random.default_rng(K)
    for m in ms:
        print(f"[case] awq slab {bits} {dtn} K={K} N={N} g={g} m={m}", flush=True)
        x = rng.standard_normal((m, K)).astype(np.float32)
        xd = to_dev(x, TORCH_DT[dt])
        y = call(xd, d, bits, m)
        assert "_slab" in ops.default_context().last_plan()["kernel"], ops.default_context().last_plan()
        assert_close(y, oracle.matmul_nt_f32(round_x(x, dt), w), f"awq slab {bits} {dtn} m{m}")
        assert np.array_equal(bits_of(call(xd, d, bits, m)), bits_of(y))


@pytest.mark.parametrize("bits,K,N,g,ms", [
    (4, 1120, 1032, 32, (3, 8, 9, 16)),   # K ends inside a run; the last workgroup 8 columns wide
    (4, 4096, 4096, 64, (1, 2, 7, 16)),
    (4, 5120, 13832, 128, (2, 16)),       # 128-row runs, two a wave
    (8, 1216, 1000, 64, (3, 8, 16)),
    (8, 1120, 1032, 32, (5, 12)),
    (8, 4096, 4104, 128, (2, 9, 40)),     # 40 rows: the copy in the workspace
])
@pytest.mark.parametrize("dtn", ["f16", "bf16"])
def test_gptq_against_the_oracle(bits, K, N, g, ms, dtn):
    dt = DT[dtn]
    qw, qz, sc = synth.gptq_checkpoint(K, N, g, bits, seed=K + N)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, TORCH_DT[dt]))
    w = oracle.dequantize_gptq(qw, qz, oracle.round_through(sc, dt), bits)
    rng = np.random.default_rng(K)
    for m in ms:
        print(f"[case] gptq slab {bits} {dtn} K={K} N={N} g={g} m={m}", flush=True)
        x = rng.standard_normal((m, K)).astype(np.float32)
        xd = to_dev(x, TORCH_DT[dt])
        y = ops.gptq_matmul(xd, *d, bits) if m <= 8 else ops.mpp_quant_matmul(xd, *d, bits, ops.PACK_IN)
        assert ("_slab" in ops.default_context().last_plan()["kernel"]) == (m <= 16), ops.default_context().last_plan()
        ref = oracle.matmul_nt_f32(round_x(x, dt), w)
        assert_close(y, ref, f"gptq slab {bits} {dtn} m{m}")
        if m > 16:  # passes of 16 rows
            tune("OXQ_TRANSIENT_REPACK", 0)
            y = ops.mpp_quant_matmul(xd, *d, bits, ops.PACK_IN)
            assert "_slab" in ops.default_context().last_plan()["kernel"]
            assert_close(y, ref, f"gptq slab passes {bits} {dtn} m{m}")
            tune("OXQ_TRANSIENT_REPACK", None)


@pytest.mark.parametrize("dtn", ["f16", "bf16"])
@pytest.mark.parametrize("method,bits", [("gptq", 4), ("gptq", 8), ("awq", 4), ("awq", 8)])
def test_infinite_rows_give_what_the_generic_kernel_gives(method, bits, dtn):
    K, N, g, dt = 4096, 2048, 32, DT[dtn]
    qw, qz, sc = (synth.gptq_checkpoint if method == "gptq" else synth.awq_checkpoint)(K, N, g, bits, seed=3)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, TORCH_DT[dt]))
    x = np.random.default_rng(1).standard_normal((4, K)).astype(np.float32)
    x[1, 37], x[2, 900], x[3, 5], x[3, 6] = np.inf, -np.inf, np.nan, np.inf
    xd = to_dev(x, TORCH_DT[dt])

    def op():
        if method == "gptq":
            return ops.gptq_matmul(xd, *d, bits)
        return ops.w4a16_matmul(xd, *d) if bits == 4 else ops.w8a16_matmul(xd, *d)
    y = op()
    assert "_slab" in ops.default_context().last_plan()["kernel"]
    tune("OXQ_FORCE_GENERIC", 1)
    old = op()
    assert "generic" in ops.default_context().last_plan()["kernel"]
    tune("OXQ_FORCE_GENERIC", None)
    for r in (1, 2, 3):
        assert torch.equal(torch.isnan(y[r]), torch.isnan(old[r])) and torch.equal(torch.nan_to_num(y[r]), torch.nan_to_num(old[r]))
    assert bool(torch.isposinf(y[1]).any()) and bool(torch.isneginf(y[1]).any())


def test_an_infinite_f16_row_keeps_its_signs():
    """Where the weight is not zero, infinity times it; the other rows as without it.  The rows-of-16 kernel that such calls ran
    on gives the same."""
    K, N = 1024, 1024
    qw, qz, sc = synth.awq_checkpoint(K, N, 128, 4, seed=9)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, torch.float16))
    x = np.random.default_rng(1).standard_normal((4, K)).astype(np.float32)
    clean = to_dev(x, torch.float16)
    x[1, 37], x[2, 900], x[3, 5], x[3, 6] = np.inf, -np.inf, np.nan, np.inf
    xd = to_dev(x, torch.float16)
    tune("OXQ_GEMV_TILE", None)
    big = [torch.cat([t, t], 1).contiguous() for t in d]   # 2048 columns: enough workgroups for the kernel
    big = [torch.cat([t] * 4, 1).contiguous() for t in big]
    y = ops.w4a16_matmul(xd, *big)
    assert "_slab" in ops.default_context().last_plan()["kernel"]
    tune("OXQ_GEMV_TILE", 0)
    old = ops.mpp_quant_matmul(torch.cat([xd] * 3), *big, 4, ops.PACK_OUT)[:4]
    assert "awq4_mfma" in ops.default_context().last_plan()["kernel"]
    tune("OXQ_GEMV_TILE", None)
    for r in (1, 2, 3):
        a, b = y[r].float(), old[r].float()
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    assert bool(torch.isposinf(y[1]).any()) and bool(torch.isneginf(y[1]).any())
    assert torch.equal(y[0], ops.w4a16_matmul(clean, *big)[0]) or bool(((y[0] - ops.w4a16_matmul(clean, *big)[0]).abs() <= 2e-3 * y[0].abs() + 1e-2).all())


def at_address(t, off):
    """The same words ``off`` elements behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + 16, device="cuda", dtype=t.dtype)
    v = buf[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 16 == off * t.element_size()
    return v


@pytest.mark.parametrize("bits,g", [(4, 64), (4, 128), (8, 128)])
@pytest.mark.parametrize("which", ["qweight", "qzeros", "neither"])
def test_infinite_bf16_rows_where_the_dot_product_kernel_does_not_take_the_address(bits, g, which):
    """AWQ tensors off a 16-byte boundary ran the generic kernel, which keeps the sign of an infinity; on one, the
    dot-product kernel, where such a row is NaN."""
    K, N = 1024, 2048
    print(f"[case] awq slab {bits} g={g} {which} off a boundary", flush=True)
    qw, qz, sc = synth.awq_checkpoint(K, N, g, bits, seed=5)
    d = [to_dev(qw), to_dev(qz), to_dev(sc, torch.bfloat16)]
    if which != "neither":
        i = ["qweight", "qzeros"].index(which)
        d[i] = at_address(d[i], 1)
    x = np.random.default_rng(1).standard_normal((4, K)).astype(np.float32)
    x[1, 37], x[2, 900], x[3, 5], x[3, 6] = np.inf, -np.inf, np.nan, np.inf
    xd = to_dev(x, torch.bfloat16)
    op = ops.w4a16_matmul if bits == 4 else ops.w8a16_matmul
    y = op(xd, *d)
    assert "_slab" in ops.default_context().last_plan()["kernel"]
    tune("OXQ_GEMV_TILE", 0)
    old = op(xd, *d)
    assert ("generic" in ops.default_context().last_plan()["kernel"]) == (which != "neither")
    tune("OXQ_GEMV_TILE", None)
    for r in (1, 2, 3):
        assert torch.equal(torch.isnan(y[r]), torch.isnan(old[r])) and torch.equal(torch.nan_to_num(y[r]), torch.nan_to_num(old[r]))
    assert bool(torch.isposinf(y[1]).any()) == (which != "neither")


@pytest.mark.parametrize("method,bits,g", [("gptq", 4, 32), ("gptq", 4, 64), ("gptq", 8, 64), ("awq", 4, 32), ("awq", 8, 32)])
def test_large_finite_bf16_rows_do_not_overflow(method, bits, g):
    """Rows whose products with bias + q overflow f32 while those with q - z do not.  A result is one bf16 rounding and the
    f32 sums off (2^-8 and 2^-20 of the sum of the terms' magnitudes)."""
    K, N = 1024, 4096
    print(f"[case] slab large finite rows {method} {bits} g={g}", flush=True)
    make = synth.gptq_checkpoint if method == "gptq" else synth.awq_checkpoint
    qw, qz, sc = make(K, N, g, bits, seed=7)
    s = oracle.round_through(sc, oracle.BF16)
    w = oracle.dequantize_gptq(qw, qz, s, bits) if method == "gptq" else (oracle.dequantize_awq if bits == 4 else oracle.dequantize_awq8)(qw, qz, s)
    x = np.random.default_rng(2).standard_normal((4, K)).astype(np.float32)
    x[1] = np.abs(x[1]) * (1e36 if bits == 4 else 1.2e35)   # 32 products with 128 + q, with q of 8 bits: beyond 3.4e38
    x[2, 5], x[3, 5], x[3, 6] = 3e38 if bits == 4 else 2e37, 3e36, -3e36   # one weight without its scale
    xr = round_x(x, oracle.BF16)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, torch.bfloat16))
    xd = to_dev(x, torch.bfloat16)
    if method == "gptq":
        y = ops.gptq_matmul(xd, *d, bits)
    else:
        y = (ops.w4a16_matmul if bits == 4 else ops.w8a16_matmul)(xd, *d)
    assert "_slab" in ops.default_context().last_plan()["kernel"]
    y = y.double().cpu().numpy()
    x64, w64 = xr.astype(np.float64), w.reshape(N, K).astype(np.float64)
    ref, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64.T)
    assert np.isfinite(y).all()
    assert (np.abs(y - ref) <= 2.0 ** -8 * np.abs(ref) + 2.0 ** -20 * mag).all()


@pytest.mark.parametrize("method,bits,K,N,g,m", [("gptq", 4, 4096, 4096, 32, 4), ("gptq", 4, 4096, 4096, 64, 4),
                                                 ("gptq", 8, 4096, 4096, 32, 4), ("awq", 4, 4096, 8192, 32, 1), ("awq", 4, 4096, 4104, 64, 1),
                                                 ("awq", 8, 4096, 4096, 32, 4)])
def test_f16_sums_are_as_exact_as_with_every_weight_by_itself(method, bits, K, N, g, m):
    """Beyond the result's own rounding, errors of small outputs stay within the generic kernel's f32 sums: K products whose
    partial sums lie near sqrt(K) of them, 2^-22 of the sum of the terms' magnitudes in all (a bias of 1024: up to 2^-20.5)."""
    print(f"[case] slab f16 sums {method} {bits} K={K} g={g} m={m}", flush=True)
    make = synth.gptq_checkpoint if method == "gptq" else synth.awq_checkpoint
    qw, qz, sc = make(K, N, g, bits, seed=11)
    s = oracle.round_through(sc, oracle.F16)
    w = oracle.dequantize_gptq(qw, qz, s, bits) if method == "gptq" else (oracle.dequantize_awq if bits == 4 else oracle.dequantize_awq8)(qw, qz, s)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, torch.float16))
    for mean in (0.0, 8.0):
        x = (np.random.default_rng(5).standard_normal((m, K)) + mean).astype(np.float32)
        xd = to_dev(x, torch.float16)
        y = (ops.gptq_matmul(xd, *d, bits) if method == "gptq" else (ops.w4a16_matmul if bits == 4 else ops.w8a16_matmul)(xd, *d))
        assert "_slab" in ops.default_context().last_plan()["kernel"]
        x64, w64 = round_x(x, oracle.F16).astype(np.float64), w.reshape(N, K).astype(np.float64)
        ref, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64.T)
        over = np.abs(y.double().cpu().numpy() - ref) - 2.0 ** -11 * np.abs(ref)
        assert (over <= 2.0 ** -22 * mag).all(), (over / mag).max()


# A f32 error of e moves the rounding of a share 2 e / ulp of the results.  Beside a bias of at most the codes' own range (16 in
# bf16, 64 / 256 in f16) a result's sums are off by a few 2^-24 of it: 2^-13 to 2^-12 of the results in bf16, eight times that
# share in f16; beside 128, or 1024, four times as many and more.
@pytest.mark.parametrize("dtn,method,bits,K,N,g,m,most", [
    ("bf16", "awq", 4, 4096, 14336, 128, 4, 4e-4), ("bf16", "awq", 4, 4096, 4096, 32, 8, 4e-4), ("bf16", "gptq", 4, 4096, 4096, 64, 16, 4e-4),
    ("f16", "awq", 8, 4096, 4096, 32, 4, 3e-3), ("f16", "gptq", 8, 4096, 4096, 64, 8, 3e-3), ("f16", "awq", 4, 4096, 4096, 128, 1, 8e-3)])
def test_nearly_all_results_are_the_nearest(dtn, method, bits, K, N, g, m, most):
    print(f"[case] slab nearest {dtn} {method} {bits} K={K} N={N} g={g} m={m}", flush=True)
    dt = DT[dtn]
    qw, qz, sc = (synth.gptq_checkpoint if method == "gptq" else synth.awq_checkpoint)(K, N, g, bits, seed=11)
    s = oracle.round_through(sc, dt)
    w = oracle.dequantize_gptq(qw, qz, s, bits) if method == "gptq" else (oracle.dequantize_awq if bits == 4 else oracle.dequantize_awq8)(qw, qz, s)
    d = (to_dev(qw), to_dev(qz), to_dev(sc, TORCH_DT[dt]))
    w64 = torch.from_numpy(w.reshape(N, K)).cuda().double()
    for mean in (0.0, 4.0):
        xd = to_dev((np.random.default_rng(5).standard_normal((m, K)) + mean).astype(np.float32), TORCH_DT[dt])
        if m > 8:
            y = ops.mpp_quant_matmul(xd, *d, bits, ops.PACK_IN if method == "gptq" else ops.PACK_OUT)
        else:
            y = ops.gptq_matmul(xd, *d, bits) if method == "gptq" else (ops.w4a16_matmul if bits == 4 else ops.w8a16_matmul)(xd, *d)
        assert "_slab" in ops.default_context().last_plan()["kernel"], ops.default_context().last_plan()
        off = (y != (xd.double() @ w64.T.contiguous()).to(y.dtype)).double().mean().item()
        assert off <= most, (mean, off)
