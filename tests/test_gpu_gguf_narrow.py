"""Q2_K and Q3_K layers from 2^20 weights: 3 - 8 rows and prefill rows on the matrix-core copy.

Tolerances as for the other formats of that copy: the GEMV's, against unrounded weights up to 8 rows and against weights
rounded to bf16 beyond (the tile arithmetic)."""
import numpy as np
import pytest
import torch

import oracle
from oxydllm_amd import ops, synth
from tests.helpers import assert_close, bits_of, round_x, to_dev, tune

pytestmark = pytest.mark.gpu
TAG = {synth.GGUF_Q2_K: "q2k", synth.GGUF_Q3_K: "q3k"}


# a ragged last group of 64 columns and one chunk a wave; three and two chunks a wave (nine blocks); four strips a workgroup;
# large enough that prefill rows are on the copy by themselves
@pytest.mark.parametrize("fmt", list(TAG))
@pytest.mark.parametrize("N,K", [(1040, 1024), (528, 2304), (12352, 256), (2624, 3328)])
def test_rows_on_the_matrix_core_copy(fmt, N, K):
    data = synth.gguf_weight(fmt, N, K, seed=N + K + fmt)
    w = oracle.dequantize_gguf(fmt, data, N, K)
    wr = oracle.round_through(w, oracle.BF16)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    x = np.random.default_rng(K).standard_normal((130, K)).astype(np.float32)
    wd = to_dev(data)
    for tdt, rows in ((torch.float32, (3, 4, 5, 8)), (torch.bfloat16, (3, 4, 5, 8) + ((33, 130) if N * K >= 1 << 23 else ()))):
        f32 = tdt == torch.float32
        layer = ops.QLinear(fmt, wd, K, N, to_dev(bias, tdt), tdt)
        xr, br, xd = (x, bias, to_dev(x)) if f32 else (round_x(x, oracle.BF16), round_x(bias, oracle.BF16), to_dev(x, tdt))
        assert np.array_equal(layer.dequantize().cpu().numpy().view(np.uint32), w.view(np.uint32))
        for m in rows:
            print(f"[case] gguf {TAG[fmt]} N={N} K={K} m={m} {tdt}", flush=True)
            y = layer.forward(xd[:m].contiguous())
            kernel = ops.default_context().last_plan()["kernel"]
            exact = m <= 8
            assert kernel.startswith(f"gguf_{TAG[fmt]}_" + ("mfma_f32" if f32 else "mfma_bf16" if exact else "gemm_bf16")), kernel
            assert_close(y, oracle.matmul_nt_f32(xr[:m], w if exact else wr, br), f"{kernel} m={m}", bf16_out=not f32)
            assert np.array_equal(bits_of(layer.forward(xd[:m].contiguous())), bits_of(y)), "run to run"
    # the forms of the prefill kernel, its K slices, and a row's bits through the row tiles of 16, 32, 48 and 64
    for ks, slices in ((1, 0), (4, 0), (0, 1), (0, 2)):
        if (slices == 2 and K < 1024) or (ks and N % 64):
            continue
        tune("OXQ_GGUF_GEMM_MIN_M", 9 if ks else None)
        tune("OXQ_GGUF_GEMM_KS", ks or None)
        tune("OXQ_GGUF_GEMM_SLICES", slices or None)
        whole = layer.forward(xd)
        assert_close(whole, oracle.matmul_nt_f32(xr, wr, br), f"ks {ks} slices {slices}", bf16_out=True)
        for m in (9, 16, 17, 32, 33, 48, 49, 65):
            print(f"[case] gguf {TAG[fmt]} N={N} K={K} m={m} ks {ks} slices {slices}", flush=True)
            y = layer.forward(xd[:m].contiguous())
            plan = ops.default_context().last_plan()
            assert "_gemm_bf16" in plan["kernel"] and plan["split_k"] == max(1, slices), plan
            assert np.array_equal(bits_of(y), bits_of(whole[:m])), plan


@pytest.mark.parametrize("fmt", list(TAG))
def test_infinities_follow_the_kernels_of_fewer_and_more_rows(fmt):
    """An infinite activation: what the vector GEMV gives up to 4 rows, what the tile matmul on the file layout gives beyond."""
    N, K = 2624, 3328
    wd = to_dev(synth.gguf_weight(fmt, N, K, seed=fmt))
    new = ops.QLinear(fmt, wd, K, N, None, torch.bfloat16)
    tune("OXQ_GGUF_MFMA", 0)
    old = ops.QLinear(fmt, wd, K, N, None, torch.bfloat16)
    tune("OXQ_GGUF_MFMA", None)
    x = torch.randn((40, K), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    x[1, 5], x[2, 700], x[3, 9] = float("inf"), float("-inf"), float("nan")
    for m in (4, 40):
        a, b = new.forward(x[:m].cuda()).float().cpu().numpy(), old.forward(x[:m].cuda()).float().cpu().numpy()
        for f in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(f(a), f(b), err_msg=f"m={m}")


@pytest.mark.parametrize("fmt", list(TAG))
@pytest.mark.parametrize("N,K,m", [(1040, 1024, 5), (2624, 3328, 8), (12352, 256, 7), (528, 2304, 8)])  # 8 and 16 waves; four strips a workgroup
def test_infinite_and_large_rows_from_five_on(fmt, N, K, m):
    """5 - 8 rows ran on the tile matmul with unrounded weights before: an infinity times a weight keeps its sign, and large rows have
    finite sums where the result is one, though those with the integers alone are not."""
    data = synth.gguf_weight(fmt, N, K, seed=fmt + K)
    w = oracle.dequantize_gguf(fmt, data, N, K)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    layer = ops.QLinear(fmt, to_dev(data), K, N, to_dev(bias, torch.bfloat16), torch.bfloat16)
    x = np.random.default_rng(K + m).standard_normal((m, K)).astype(np.float32)
    plain = layer.forward(to_dev(x, torch.bfloat16))
    x[0, 5], x[1, K - 1], x[2, 9] = np.inf, -np.inf, np.nan
    x[3] *= 3e39 / float((np.abs(x[3]) @ np.abs(w).T).max())
    x[m - 1] = 0.0
    x[m - 1, 17] = 3e38 / max(1.0, float(np.abs(w[:, 17]).max()))
    print(f"[case] gguf {TAG[fmt]} infinite and large rows N={N} K={K} m={m}", flush=True)
    y = layer.forward(to_dev(x, torch.bfloat16))
    assert ops.default_context().last_plan()["kernel"].startswith(f"gguf_{TAG[fmt]}_mfma_bf16")
    got = y.float().cpu().numpy()
    for r, k, sign in ((0, 5, 1.0), (1, K - 1, -1.0)):
        np.testing.assert_array_equal(got[r], np.where(w[:, k] == 0, np.nan, sign * np.sign(w[:, k]) * np.inf).astype(np.float32))
    assert np.isnan(got[2]).all()
    x64 = round_x(x, oracle.BF16).astype(np.float64)
    for r in (3, m - 1):
        ref, mag = x64[r] @ w.T.astype(np.float64), np.abs(x64[r]) @ np.abs(w.T.astype(np.float64))
        fits = np.abs(ref) < 3.3e38
        assert fits.any() and np.isfinite(got[r][fits]).all()
        # one bf16 rounding, f32 sums, the bias
        assert (np.abs(got[r] - ref)[fits] <= (2.0 ** -8 * np.abs(ref) + 2.0 ** -18 * mag + 8)[fits]).all()
        big = np.abs(ref) > 3.5e38
        np.testing.assert_array_equal(got[r][big], (np.sign(ref) * np.inf)[big].astype(np.float32))
    for r in range(4, m - 1):
        assert torch.equal(y[r], plain[r])
