// Instances and launches of pk4_mid_kernel (pk4_mid.hpp).
#include "pk4_mid.hpp"

namespace oxq {

template <typename TT, int BITS, int SETS, bool NARROW>
static int mid_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)PK4M_STAGES * PK4M_KS * 16 * PK4M_MT * 128;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4_mid_kernel<TT, BITS, SETS, NARROW>, lds));
    hipLaunchKernelGGL((pk4_mid_kernel<TT, BITS, SETS, NARROW>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw,
                       (const uint16_t *)p.bias, (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

template <typename TT>
static int mid_layout(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    if (p.w.strip == 16) return mid_go<TT, 4, 1, true>(s, grid, p, NG);
    const bool b4 = p.w.bits == 4;
    switch (pk4_sets(p.w.group_shift)) {
    case 1: return b4 ? mid_go<TT, 4, 1, false>(s, grid, p, NG) : mid_go<TT, 8, 1, false>(s, grid, p, NG);
    case 2: return b4 ? mid_go<TT, 4, 2, false>(s, grid, p, NG) : mid_go<TT, 8, 2, false>(s, grid, p, NG);
    default: return b4 ? mid_go<TT, 4, 4, false>(s, grid, p, NG) : mid_go<TT, 8, 4, false>(s, grid, p, NG);
    }
}

int launch_pk4_mid(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    return p.w.dtype == OXQ_F16 ? mid_layout<F16Traits>(s, grid, p, NG) : mid_layout<BF16Traits>(s, grid, p, NG);
}

}  // namespace oxq
