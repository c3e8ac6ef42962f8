// pk4_midfold_kernel: resident layers whose weights are not rounded to the activation type (pk4_unrounded), between few rows
// and the folded prefill form: 64 rows x two groups of 64 columns a workgroup, K over four waves, as pk4_mid_kernel
// (pk4_mid.hpp), with the arithmetic of pk4_gemm_kernel's folded form (pk4_gemm.hpp).
//
// Row tiles of 32 of pk4_mfma_kernel, one strip a workgroup, read a layer's weights once per 32 rows and fold a group's sums
// for two row tiles at a time; the prefill form needs 512 columns a workgroup to fill the chip.  A group's sums take as many
// registers as the accumulators (64 each, 16 for the row sums), so x comes in half blocks through five stages of LDS with
// one step's fragments in registers, and weights one block ahead, as in pk4_mid128_kernel.  What bounds it: the issue of the fold's
// multiply-adds beside the MFMAs.  f16 therefore multiplies q - z, an exact packed subtraction a pair of weights: no row sums of
// x (a fifth of the MFMAs) and one multiply-add a sum and group instead of two.  bf16 has no packed arithmetic and keeps them.
#include "pk4_gemm.hpp"
#include "pk4_mid.hpp"

namespace oxq {

constexpr int PK4MF_STAGES = 5;

template <typename TT, int BITS, int SETS>
__global__ __launch_bounds__(512) void pk4_midfold_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                          const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                          int M, int K, int N, int NG, int act) {
    typedef MfmaOps<TT> Ops;
    constexpr int MT = PK4M_MT, KS = PK4M_KS, SPW = PK4M_GROUPS, ROWS = 16 * MT, NS = PK4MF_STAGES;
    constexpr int WL = BITS / 4, BB = pk4_block_words(BITS, SETS) * 4;
    constexpr int TILE = ROWS * 128, STAGE = KS * TILE;  // bytes of x: a wave's half block, a stage
    constexpr int SPS = 4 / SETS;                        // steps that share a set of pairs
    constexpr int OOB = 0x7FFFFF00;
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE, MINUS_ZERO = !BF;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws_ = wave % SPW, kq = wave / SPW;  // the wave's column group of the workgroup, and its share of K
    const int rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;  // (as in pk4_mid_kernel)
    const int j = g * SPW + ws_;
    const bool live = j < ((N + 63) >> 6);  // wave-uniform: the last workgroup of a layer may have one column group
    const int m0 = rt * ROWS;
    const int NB = SETS > 1 ? (K + 127) >> 7 : K >> 7, NR = (NB + KS - 1) / KS;  // blocks; rounds of KS blocks

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl = make_rsrc(pw + (size_t)(live ? j : 0) * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)min(M - m0, ROWS) * (uint32_t)K * 2u);
    // offsets made where they are used: as in pk4_mid128_kernel
    auto lane_again = [] {
        uint32_t ones = ~0u;
        asm volatile("" : "+s"(ones));
        return (int)__builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u));
    };

    // a half block's loads: pk4_mid_kernel's, where load q + 2 lies 16 rows on (rows past M: beyond the descriptor by the lane's offset)
    int xo[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int r = 8 * (ws_ * MT + q) + (lane >> 3);
        xo[q] = r * K * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    // the lanes whose piece of 8 elements lies in the upper half of a half block: of even loads, odd ones the others
    const bool upper = (lane >> 2) & 1;
    auto dma = [&](int i, int hf, int slot, int q) {  // load q of a half of block i
        // K may end inside the last block, at groups of 32 inside the half: zeros for the pieces past it, not the next row
        const int left = K - i * 128 - hf * 64;
        const __amdgpu_buffer_rsrc_t rs = left > 0 ? rs_x : rs_none;
        int rows16 = 32 * K;
        asm volatile("" : "+s"(rows16));
        int off = q < 2 ? xo[q] : xo[q & 1] + rows16;
        if constexpr (SETS == 4) off = left < 64 && upper == !(q & 1) ? OOB : off;
        pk4g_load_lds16(rs, pk4_lds + slot * STAGE + kq * TILE + ws_ * (MT * 1024) + q * 1024, off, i * 256 + hf * 128);
    };
    // fragment of a half block's first step, row tile mt (+ 2048 mt): row ni; the second step's is a bit of the piece away
    constexpr int STEP = SETS == 4 ? 64 : 16;
    const int a_rd = kq * TILE + ni * 128 + (((pk4_x_chunk<SETS>(0, kb) & 7) ^ ((ni >> 1) & 7)) << 4);

    u32x4_t wring[4][WL];
    uint32_t zring[SETS];
    auto load_w = [&](int i, int st) {
#pragma unroll
        for (int h = 0; h < WL; ++h)
            wring[st][h] = __builtin_amdgcn_raw_buffer_load_b128(i < NB ? rs_w : rs_none, lane_again() * 16, i * BB + (st * WL + h) * 1024, 0);
    };
    auto load_z = [&](int i, int set) {
        const int l = lane_again();
        zring[set] = __builtin_amdgcn_raw_buffer_load_b32(i < NB ? rs_w : rs_none, 4096 * WL + ((l & 15) * 4 + (l >> 4)) * 4, i * BB + set * 256, 0);
    };

    // The compiler orders nothing against the loads into LDS: the waits for them count the younger loads, whose order
    // the barriers of the scheduler keep.
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int q = 0; q < MT; ++q) dma(KS * (u >> 1) + kq, u & 1, u, q);
    __builtin_amdgcn_sched_barrier(0);
    // (behind the third half block: the first wait in the loop, for that one, counts as many ring loads as the others)
#pragma unroll
    for (int st = 0; st < 4; ++st) load_w(kq, st);
#pragma unroll
    for (int u = 0; u < SETS; ++u) load_z(kq, u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < MT; ++q) dma(KS + kq, 1, 3, q);
    __builtin_amdgcn_sched_barrier(0);
    // one constant of v_and_or_b32 may come from a scalar register: the mask is a vector register's
    constexpr int AT = Pk4Fold<TT, BITS>::AT;
    uint32_t nibbles = (0xFu << AT) * 0x10001u;
    asm volatile("" : "+v"(nibbles));
    auto integers = [&](uint32_t word, int f) {  // Pk4Fold::pair
        if constexpr (BITS == 4) {
            const int left = AT - 4 * f;
            return ((left >= 0 ? word << left : word >> -left) & nibbles) | (BF ? 0x41804180u : 0x4C004C00u);
        } else {
            return Pk4Fold<TT, BITS>::pair(word, f);
        }
    };
    const float4_t zero4 = float4_t{0.f, 0.f, 0.f, 0.f};
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = zero4;
    // Raw barriers, as in pk4_mid_kernel: a wave's own reads of LDS are over before it arrives.
    auto meet = [&](auto younger) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(younger)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    u32x4_t a[2][MT];  // fragments of x: the two steps
    auto read_x = [&](int slot, int s) {
        const unsigned char *from = pk4_lds + ((slot * STAGE + a_rd) ^ (s ? STEP : 0));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[s][mt] = *(const u32x4_t *)(from + mt * 2048);
    };
    // The first two half blocks, counting as younger only the loads into LDS (the compiler may issue the ring loads behind this wait).
    meet(std::integral_constant<int, 2 * MT>{});
    read_x(0, 0);
    __builtin_amdgcn_sched_barrier(0);

    float4_t tmp[MT][4], tmps[MINUS_ZERO ? 1 : MT];  // a group's sums, and those of x
    float sf[4], nz[4];  // a group's scales and -(BIAS + z); f16 has the latter in nzp, twice in a register
    uint32_t nzp[4];
    auto constants = [&](int set) {
        uint32_t zv[4];
        pk4_pair_words(zring[set], zv);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            sf[f] = TT::to_f32((uint16_t)(zv[f] >> 16));
            asm volatile("" : "+v"(sf[f]));  // a conversion here, not a slower multiply-add of mixed types sixteen times
            if constexpr (MINUS_ZERO) {
                const uint16_t lack = TT::from_f32(Pk4Fold<TT, BITS>::offset(f));
                nzp[f] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, perm_b32(zv[f], zv[f], 0x01000100u)) +
                                                          __builtin_bit_cast(half2_t, (uint32_t)lack | ((uint32_t)lack << 16)));
            } else {
                nz[f] = TT::to_f32((uint16_t)(zv[f] & 0xFFFFu)) + Pk4Fold<TT, BITS>::offset(f);
            }
        }
    };
    // One half block, out of stage `slot`; the next one's first step is read out of `next`, and `free`, the stage of the half
    // block before, takes the one of two rounds on.
    auto unit = [&](int r, auto hf_c, int slot) {
        constexpr int HF = decltype(hf_c)::value;
        const int i = KS * r + kq;
        const int next = slot == NS - 1 ? 0 : slot + 1, free = slot == 0 ? NS - 1 : slot - 1;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int st = 2 * HF + s;
            const bool fresh = st % SPS == 0, last = (st + 1) % SPS == 0;  // a group's sums start from zero: no clearing
            dma(i + 2 * KS, HF, free, 2 * s), dma(i + 2 * KS, HF, free, 2 * s + 1);
            read_x(s ? next : slot, 1 - s);
            uint32_t wp[WL][4];
#pragma unroll
            for (int h = 0; h < WL; ++h) wp[h][0] = wring[st][h][0], wp[h][1] = wring[st][h][1], wp[h][2] = wring[st][h][2], wp[h][3] = wring[st][h][3];
            auto frag = [&](int mt, uint32_t (&av)[4]) { av[0] = a[s][mt][0], av[1] = a[s][mt][1], av[2] = a[s][mt][2], av[3] = a[s][mt][3]; };
            auto row_sums = [&] {
                const uint32_t ones[4] = {TT::ONES, TT::ONES, TT::ONES, TT::ONES};
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    uint32_t av[4];
                    frag(mt, av);
                    tmps[mt] = Ops::mfma(av, ones, fresh ? zero4 : tmps[mt]);
                }
            };
            if (MINUS_ZERO ? fresh : last) constants(st / SPS);
            if (!MINUS_ZERO && last) row_sums();
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                uint32_t b[4];
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                    b[pp] = integers(wp[(f >> 1) % WL][pp], f);
                    if constexpr (MINUS_ZERO) b[pp] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, b[pp]) + __builtin_bit_cast(half2_t, nzp[f]));
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    uint32_t av[4];
                    frag(mt, av);
                    tmp[mt][f] = Ops::mfma(av, b, fresh ? zero4 : tmp[mt][f]);
                }
            }
            if (!MINUS_ZERO && !last) row_sums();
            if (last) {
#pragma unroll
                for (int f = 0; f < 4; ++f) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if constexpr (MINUS_ZERO) acc[mt][f][e] = fmaf(sf[f], tmp[mt][f][e], acc[mt][f][e]);
                            else acc[mt][f][e] = fmaf(sf[f], fmaf(nz[f], tmps[mt][e], tmp[mt][f][e]), acc[mt][f][e]);
                        }
                }
            }
            __builtin_amdgcn_sched_group_barrier(0x120, 2 + MT, 0);
#pragma unroll
            for (int n = 0; n < (MINUS_ZERO ? 4 : 5) * MT; ++n) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (last) __builtin_amdgcn_sched_group_barrier(0x002, MINUS_ZERO ? 7 : 9, 0);
                else __builtin_amdgcn_sched_group_barrier(0x002, MINUS_ZERO ? 3 : 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_w(i + KS, st);  // into the registers this step has just left
            if (MINUS_ZERO ? fresh : last) load_z(i + KS, st / SPS);
            __builtin_amdgcn_sched_barrier(0);
        }
        // The half block after the next is in LDS: the loads of this one and the one before are younger.
        meet(std::integral_constant<int, 2 * MT + 4 * WL + SETS>{});
        return next;
    };
    int slot = 0;
    for (int r = 0; r < NR; ++r) {
        slot = unit(r, std::integral_constant<int, 0>{}, slot);
        slot = unit(r, std::integral_constant<int, 1>{}, slot);
    }
    meet(std::integral_constant<int, 0>{});  // the stages past the end have been zeroed: nothing lands in LDS any more

    // slot of wave w: [mt][e][lane] x float4 (f = 0..3); wave kq of a column group finishes row tile kq
    const int l = lane_again();
    float4_t *red = (float4_t *)pk4_lds;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            red[((wave * MT + mt) * 4 + e) * 64 + l] = float4_t{acc[mt][0][e], acc[mt][1][e], acc[mt][2][e], acc[mt][3][e]};
    __syncthreads();
    if (!live) return;
    float4_t fin[4];  // row 16 kq + 4 kb + e
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        fin[e] = zero4;
#pragma unroll
        for (int k = 0; k < KS; ++k)  // K order: the same sum whatever the timing
            fin[e] += red[(((k * SPW + ws_) * MT + kq) * 4 + e) * 64 + l];
    }
    pk4m_store<TT, false>(fin, bias, y, M, N, j, l & 15, m0 + 16 * kq + 4 * (l >> 4), act);
}

template <typename TT, int BITS, int SETS>
static int midfold_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)PK4MF_STAGES * PK4M_KS * 16 * PK4M_MT * 128;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4_midfold_kernel<TT, BITS, SETS>, lds));
    hipLaunchKernelGGL((pk4_midfold_kernel<TT, BITS, SETS>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw,
                       (const uint16_t *)p.bias, (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <typename TT, int BITS>
static int midfold_sets(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    switch (pk4_sets(p.w.group_shift)) {
    case 1: return midfold_go<TT, BITS, 1>(s, grid, p, NG);
    case 2: return midfold_go<TT, BITS, 2>(s, grid, p, NG);
    default: return midfold_go<TT, BITS, 4>(s, grid, p, NG);
    }
}
int launch_pk4_midfold(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    const bool f16 = p.w.dtype == OXQ_F16;
    if (p.w.bits == 4) return f16 ? midfold_sets<F16Traits, 4>(s, grid, p, NG) : midfold_sets<BF16Traits, 4>(s, grid, p, NG);
    return f16 ? midfold_sets<F16Traits, 8>(s, grid, p, NG) : midfold_sets<BF16Traits, 8>(s, grid, p, NG);
}

}  // namespace oxq
