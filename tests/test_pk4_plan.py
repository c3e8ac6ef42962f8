"""Which kernel a resident packed layer runs, asked of a plan-only ctx: no GPU needed."""
import ctypes as C

import pytest

from oxydllm_amd import _lib, ops
from tests.helpers import fake


def kernels(pack, bits, K, N, g, dt, rows):
    lib, plan = _lib.load(), ops.Context(plan_only=True)
    pf = 32 // bits
    qw = fake((K, N // pf) if pack == ops.PACK_OUT else (K // pf, N), _lib.I32)
    h = C.c_void_p()
    rc = lib.oxq_packed_quant_linear_new(plan.handle, bits, pack, C.byref(qw), C.byref(fake((K // g, N // pf), _lib.I32)),
                                         C.byref(fake((K // g, N), dt)), None, dt, C.byref(h))
    assert rc == 0, lib.oxq_last_error().decode()
    out = []
    for m in rows:
        assert lib.oxq_packed_quant_linear_forward(h, None, C.byref(fake((m, K), dt)), C.byref(fake((m, N), dt))) == 0
        out.append((plan.last_plan()["kernel"], plan.last_plan()["grid"][2]))
    lib.oxq_packed_quant_linear_free(h)
    return out


def test_fused_layer_with_a_bias_at_any_address():
    """A bias that is no multiple of eight bytes: the fused layer is built as before, and every row count runs on the tiles
    that read it column by column."""
    lib, plan = _lib.load(), ops.Context(plan_only=True)
    K, N, dt = 4096, 28672, _lib.BF16
    bias = fake((N,), dt)
    bias.data = 0x1002
    h = C.c_void_p()
    rc = lib.oxq_packed_quant_linear_new_gate_up(plan.handle, 4, ops.PACK_OUT, C.byref(fake((K, N // 8), _lib.I32)),
                                                 C.byref(fake((K // 128, N // 8), _lib.I32)), C.byref(fake((K // 128, N), dt)),
                                                 C.byref(bias), ops.ACT_GATED_SILU, dt, C.byref(h))
    assert rc == 0, lib.oxq_last_error().decode()
    for m in (1, 33, 64, 65, 1000):
        assert lib.oxq_packed_quant_linear_forward(h, None, C.byref(fake((m, K), dt)), C.byref(fake((m, N // 2), dt))) == 0
        assert plan.last_plan()["kernel"].startswith("pk4_mfma_") and plan.last_plan()["launches"] == 1
    lib.oxq_packed_quant_linear_free(h)


def test_no_three_tiles_of_folded_sums_beside_two_sets_of_pairs():
    """f16, groups of 64, 33 - 48 rows: that form spills; the rows run as two tiles of 32, still folded."""
    rows = (33, 40, 48)
    assert kernels(ops.PACK_OUT, 4, 4096, 11008, 64, _lib.F16, rows) == [("pk4_mfma_f16_mt2_gs_g64", 2)] * 3
    assert kernels(ops.PACK_OUT, 4, 4096, 11008, 32, _lib.F16, rows) == [("pk4_mfma_f16_mt3_gs_g32", 1)] * 3
    assert kernels(ops.PACK_OUT, 4, 4096, 11008, 64, _lib.BF16, rows) == [("pk4_mfma_bf16_mt3_g64", 1)] * 3
    assert kernels(ops.PACK_OUT, 4, 4096, 11008, 64, _lib.F16, (32, 49)) == [("pk4_mfma_f16_mt2_gs_g64", 1), ("pk4_mfma_f16_mt4_g64", 1)]


@pytest.mark.parametrize("pack,bits,K,N,g", [(ops.PACK_IN, 4, 4096, 11008, 64), (ops.PACK_IN, 8, 4096, 4096, 32),
                                             (ops.PACK_OUT, 8, 4096, 11000, 128), (ops.PACK_IN, 4, 4128, 4096, 32)])
@pytest.mark.parametrize("dt", [_lib.F16, _lib.BF16])
def test_unrounded_layers_run_folded_forms_only(pack, bits, K, N, g, dt):
    rows = (1, 16, 17, 32, 33, 48, 49, 64, 65, 128, 200, 512, 1024, 2048, 4096, 1 << 20)
    for m, (kernel, _) in zip(rows, kernels(pack, bits, K, N, g, dt, rows)):
        assert "_gs" in kernel and "_mt4" not in kernel, (m, kernel)


def test_narrow_layers_keep_the_tiles_that_fit_one_round():
    """64-column strips x row tiles of 64 up to the compute units run as one round of split-K tiles, also where the strips are no
    multiple of eight: 14 x 18, 12 x 17, 9 x 19 (8-bit: 10 x 20, 19 x 13).  One more round goes to the two-strip form."""
    for bits, k, n, m, dt in [(4, 1408, 896, 1099, _lib.BF16), (4, 1664, 768, 1053, _lib.F16), (8, 1024, 576, 1170, _lib.BF16),
                              (8, 5120, 640, 1257, _lib.F16), (4, 3840, 1216, 817, _lib.BF16)]:
        (kernel, _), = kernels(ops.PACK_OUT, bits, k, n, 128, dt, (m,))
        assert "_mfma_" in kernel, (k, n, m, kernel)
    (kernel, _), = kernels(ops.PACK_OUT, 4, 1408, 896, 128, _lib.BF16, (1153,))  # 14 x 19
    assert "_gemm_" in kernel, kernel


def k_slices(pack, bits, K, N, g, dt, m):
    lib, plan = _lib.load(), ops.Context(plan_only=True)
    pf = 32 // bits
    h = C.c_void_p()
    assert lib.oxq_packed_quant_linear_new(plan.handle, bits, pack, C.byref(fake((K, N // pf) if pack == ops.PACK_OUT else (K // pf, N), _lib.I32)),
                                           C.byref(fake((K // g, N // pf), _lib.I32)), C.byref(fake((K // g, N), dt)), None, dt, C.byref(h)) == 0
    assert lib.oxq_packed_quant_linear_forward(h, None, C.byref(fake((m, K), dt)), C.byref(fake((m, N), dt))) == 0
    lib.oxq_packed_quant_linear_free(h)
    return plan.last_plan()["kernel"], plan.last_plan()["split_k"]


def test_k_slices_stay_where_a_whole_k_a_workgroup_takes_longer():
    """K = 4096, row tiles of few strips: up to 1.45 x the time in 8-bit layers and groups of 32 without their slices."""
    for bits, n, g, m, dt in [(8, 3072, 32, 30, _lib.F16), (8, 1536, 64, 30, _lib.F16), (8, 768, 128, 30, _lib.BF16), (4, 1152, 32, 60, _lib.BF16),
                              (8, 704, 128, 164, _lib.BF16), (4, 4096, 128, 20, _lib.BF16)]:
        kernel, ks = k_slices(ops.PACK_OUT, bits, 4096, n, g, dt, m)
        assert ks >= 2, (bits, n, g, m, kernel)
    for bits, n, g, m, dt in [(4, 1792, 128, 67, _lib.F16), (4, 2816, 64, 74, _lib.BF16), (8, 3072, 128, 66, _lib.F16), (4, 4096, 128, 64, _lib.F16)]:
        kernel, ks = k_slices(ops.PACK_OUT, bits, 4096, n, g, dt, m)
        assert ks == 1 and "_by" in kernel, (bits, n, g, m, kernel)


def test_row_tiles_stay_together_on_long_chains():
    """Two or three row tiles a workgroup in the place of four: not where a workgroup's K is long and a strip's workgroups stand on
    all XCDs."""
    for k, n, m, dt in [(13568, 1472, 383, _lib.F16), (8704, 1984, 343, _lib.F16), (8064, 832, 564, _lib.F16), (10880, 3712, 192, _lib.F16),
                        (12544, 2624, 256, _lib.BF16), (7680, 2824, 197, _lib.F16), (4096, 5512, 42, _lib.BF16)]:
        (kernel, _), = kernels(ops.PACK_OUT, 4, k, n, 128, dt, (m,))
        assert "_by" not in kernel, (k, n, m, kernel)
    for k, n, m, dt in [(9216, 2048, 340, _lib.F16), (1664, 960, 615, _lib.F16), (3200, 1024, 677, _lib.F16), (9600, 2768, 185, _lib.BF16), (2304, 3328, 128, _lib.BF16)]:
        (kernel, _), = kernels(ops.PACK_OUT, 4, k, n, 128, dt, (m,))
        assert "_by" in kernel, (k, n, m, kernel)
