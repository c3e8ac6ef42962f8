// Prefill of resident layers whose weights are not rounded to the activation type (pk4_unrounded): the folded form of
// pk4_gemm_kernel, 64 rows x eight strips a workgroup.
//
// What bounds it: a group's sums need registers of their own (64 more, 188 - 256 in all: one workgroup a CU, where the rounded
// 4-bit form has two), a row-sum MFMA joins every four, and a group costs 128 multiply-adds in f32.  GPTQ 4-bit, groups of 64,
// 4096 x 11008: 2048 rows f16 265 us, 0.70 PFLOP/s (rounded weights 181); passes of the dot-product kernel over the
// checkpoint layout took 31 ms.  64-bit relative error, f16 / bf16: 2.07e-4 / 1.66e-3, that of the dot-product kernel;
// rounded weights 2.9e-4 / 2.3e-3.
#include "pk4_gemm.hpp"

namespace oxq {

template <typename TT, int BITS>
static int fold_by_sets(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    switch (pk4_sets(p.w.group_shift)) {
    case 1: return pk4_gemm_wide_go<TT, 4, BITS, 1, true>(s, grid, p, NG, RT);
    case 2: return pk4_gemm_wide_go<TT, 4, BITS, 2, true>(s, grid, p, NG, RT);
    default: return pk4_gemm_wide_go<TT, 4, BITS, 4, true>(s, grid, p, NG, RT);
    }
}

template <typename TT> static int fold_by_bits(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    return p.w.bits == 4 ? fold_by_sets<TT, 4>(s, grid, p, NG, RT) : fold_by_sets<TT, 8>(s, grid, p, NG, RT);
}

int launch_pk4_gemm_fold(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    return p.w.dtype == OXQ_F16 ? fold_by_bits<F16Traits>(s, grid, p, NG, RT) : fold_by_bits<BF16Traits>(s, grid, p, NG, RT);
}

}  // namespace oxq
