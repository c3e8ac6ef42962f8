// Resident layers whose quantization groups are shorter than a block of 128 rows: 64 or 32 rows (AWQ and GPTQ
// checkpoints with group_size 64 or 32, compressed-tensors int4 with its default of 32).
//
// The layout, the kernels and the rules are those of pk4.hip and pk4_gemm.hip with two or four sets of zero/scale
// pairs in a block.  Group of 64: two MFMA steps share a set.  Group of 32: a step's 32 rows are one group, so the rows
// go to the lane groups in order (pk4_kk) and the folded form can take a group's sum out of one MFMA.  K is a multiple
// of the group only; a last block that is not full holds zero weights with zero scales, and the kernels mask x there.
//
// Before, such layers ran on the checkpoint layout: 4-bit AWQ on the split-K tiles, everything else as one pass of
// the dot-product kernel per 8 rows of x (GPTQ 4-bit 8000 x 12704, groups of 64, bf16, 12 rows: 447 -> 17.1 us; AWQ
// 8-bit 3456 x 704, groups of 64, 472 rows: 665 -> 16.6 us; AWQ 8-bit 6144 x 3520, groups of 32, 7 rows: 52.6 -> 10.1 us).
#include "pk4_gemm.hpp"
#include "pk4_mfma.hpp"

namespace oxq {

template <typename TT, int BITS, int SETS>
static int fine_by_mt(oxq_ctx *ctx, hipStream_t s, dim3 grid, const Pk4Problem &p, int bslice, int mt, bool fold) {
    constexpr int WD = 4;
    switch (mt) {
    case 1:
        if (!fold) return pk4_mfma_go<TT, BITS, 1, false, WD, 4, false, 0, SETS>(ctx, s, grid, p, bslice);
        if (p.M <= 4) return pk4_mfma_go<TT, BITS, 1, true, WD, 1, false, 0, SETS>(ctx, s, grid, p, bslice);
        if (p.M <= 8) return pk4_mfma_go<TT, BITS, 1, true, WD, 2, false, 0, SETS>(ctx, s, grid, p, bslice);
        return pk4_mfma_go<TT, BITS, 1, true, WD, 4, false, 0, SETS>(ctx, s, grid, p, bslice);
    case 2:
        return fold ? pk4_mfma_go<TT, BITS, 2, true, WD, 8, false, 0, SETS>(ctx, s, grid, p, bslice)
                    : pk4_mfma_go<TT, BITS, 2, false, WD, 8, false, 0, SETS>(ctx, s, grid, p, bslice);
    case 3:
        if constexpr (TT::DTYPE == F16Traits::DTYPE && SETS == 4)  // (two sets: pk4_row_tiles)
            if (fold) return pk4_mfma_go<TT, BITS, 3, true, WD, 12, false, 0, SETS>(ctx, s, grid, p, bslice);
        return pk4_mfma_go<TT, BITS, 3, false, WD, 12, false, 0, SETS>(ctx, s, grid, p, bslice);
    default: return pk4_mfma_go<TT, BITS, 4, false, WD, 16, false, 0, SETS>(ctx, s, grid, p, bslice);
    }
}

template <typename TT>
static int fine_go(oxq_ctx *ctx, hipStream_t s, dim3 grid, const Pk4Problem &p, int bslice, int mt, bool fold) {
    const bool g64 = pk4_sets(p.w.group_shift) == 2;
    if (p.w.bits == 4) return g64 ? fine_by_mt<TT, 4, 2>(ctx, s, grid, p, bslice, mt, fold) : fine_by_mt<TT, 4, 4>(ctx, s, grid, p, bslice, mt, fold);
    return g64 ? fine_by_mt<TT, 8, 2>(ctx, s, grid, p, bslice, mt, fold) : fine_by_mt<TT, 8, 4>(ctx, s, grid, p, bslice, mt, fold);
}

int launch_pk4_fine(oxq_ctx *ctx, hipStream_t s, dim3 grid, const Pk4Problem &p, int bslice, int mt, bool fold) {
    return p.w.dtype == OXQ_F16 ? fine_go<F16Traits>(ctx, s, grid, p, bslice, mt, fold)
                                : fine_go<BF16Traits>(ctx, s, grid, p, bslice, mt, fold);
}

template <typename TT, int MT>
static int fine_gemm(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    const bool g64 = pk4_sets(p.w.group_shift) == 2;
    if (p.w.bits == 4)
        return g64 ? pk4_gemm_wide_go<TT, MT, 4, 2>(s, grid, p, NG, RT) : pk4_gemm_wide_go<TT, MT, 4, 4>(s, grid, p, NG, RT);
    return g64 ? pk4_gemm_wide_go<TT, MT, 8, 2>(s, grid, p, NG, RT) : pk4_gemm_wide_go<TT, MT, 8, 4>(s, grid, p, NG, RT);
}

int launch_pk4_gemm_fine(hipStream_t s, dim3 grid, const Pk4Problem &p, int rows, int NG, int RT) {
    const bool f16 = p.w.dtype == OXQ_F16;
    if (rows == 128) return f16 ? fine_gemm<F16Traits, 8>(s, grid, p, NG, RT) : fine_gemm<BF16Traits, 8>(s, grid, p, NG, RT);
    return f16 ? fine_gemm<F16Traits, 4>(s, grid, p, NG, RT) : fine_gemm<BF16Traits, 4>(s, grid, p, NG, RT);
}

}  // namespace oxq
