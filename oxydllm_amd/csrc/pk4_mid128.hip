// pk4_mid128_kernel: 128 rows x two groups of 64 columns a workgroup, for 4-bit layers of rounded weights where
// pk4_mid_kernel (pk4_mid.hpp: the four waves of a column group take every fourth block of K) would run two row tiles.
//
// What bounds pk4_mid_kernel is the issue port, and more than half of what it issues turns codes into weights that serve
// four MFMAs.  Here a weight serves eight row tiles: half a block's eight fragments (two steps, four columns) stay in
// registers while the 64 upper and then the 64 lower rows are multiplied.  128 registers of sums and 32 of fragments
// leave none for a second half block of x or of weights, so
//   - x comes in units of 64 rows and half a block through five stages of LDS (all 160 KB), and a step's four fragments
//     are read during the step before;
//   - a fragment is rebuilt in the place of the one it follows: columns 0 .. 3 of the next half block while the lower rows'
//     step 1 is multiplied, columns 4 .. 7 at the start of the upper rows' step 0, each pair of columns spread over twelve
//     MFMAs;
//   - weights come one block ahead, into the registers that the dequant has left (16-column strips: half blocks).
// (f16, groups of 128, with a column's zero and scale in two registers each: four spilled, and the loop drained its loads once a
// round.  In the halves of one: 4096 x 28672 at 65 / 128 rows 35.2 / 36.2 -> 32.1 / 33.5 us, 9344 x 18048 at 128 68.5 -> 62.3, 1024 x
// 12544 at 256 14.6 -> 13.5.)
// The partial tiles of the four waves meet in LDS 64 rows at a time, added in K order: the bits of pk4_mid_kernel.
#include "pk4_mid.hpp"

namespace oxq {

constexpr int PK4H_STAGES = 5;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

template <typename TT, int SETS, bool NARROW>
__global__ __launch_bounds__(512) void pk4_mid128_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                         const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                         int M, int K, int N, int NG, int act) {
    typedef MfmaOps<TT> Ops;
    constexpr int MT = PK4M_MT, KS = PK4M_KS, SPW = PK4M_GROUPS, ROWS = 16 * MT, NS = PK4H_STAGES;
    constexpr int BB = NARROW ? PK4N_BW * 4 : pk4_block_words(4, SETS) * 4;
    constexpr int TILE = ROWS * 128, STAGE = KS * TILE;  // bytes of x: a wave's unit (64 rows of half a block), a stage
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    constexpr bool PAIRED = BF && !NARROW;
    static_assert(!NARROW || SETS == 1, "16-column strips hold groups of 128 rows and more");
    constexpr int OOB = 0x7FFFFF00;
    // ring loads in the first and the second half of a block
    constexpr int RE = NARROW ? 5 : SETS == 4 ? 4 : 3, RO = NARROW ? 4 : SETS == 4 ? 4 : SETS == 2 ? 3 : 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws_ = wave % SPW, kq = wave / SPW;  // the wave's column group of the workgroup, and its share of K
    const int rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;  // (as in pk4_mid_kernel)
    const int j = g * SPW + ws_;
    const bool live = j < ((N + 63) >> 6);  // wave-uniform: the last workgroup of a layer may have one column group
    const int m0 = rt * 2 * ROWS;
    const int NB = SETS > 1 ? (K + 127) >> 7 : K >> 7, NR = (NB + KS - 1) / KS;  // blocks; rounds of KS blocks

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl =
        NARROW ? make_rsrc(pw + (size_t)(live ? 4 * j : 0) * NB * PK4N_BW, 4u * (uint32_t)NB * (uint32_t)BB)
               : make_rsrc(pw + (size_t)(live ? j : 0) * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    // the upper and the lower 64 rows; rows past M lie beyond the descriptor: LDS receives zeros
    const int lower = min(max(M - m0 - ROWS, 0), ROWS);
    const __amdgpu_buffer_rsrc_t rs_x0 = make_rsrc(x + (size_t)m0 * K, (uint32_t)min(M - m0, ROWS) * (uint32_t)K * 2u);
    const __amdgpu_buffer_rsrc_t rs_x1 = make_rsrc(x + (size_t)(lower ? m0 + ROWS : m0) * K, (uint32_t)lower * (uint32_t)K * 2u);
    // A register more than the loop has and it reloads one from memory behind a wait for everything under way.  So
    // offsets are made where they are used, from what the empty asm keeps the compiler from hoisting.
    auto lane_again = [] {
        uint32_t ones = ~0u;
        asm volatile("" : "+s"(ones));
        return (int)__builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u));
    };

    // a unit's loads: pk4_mid_kernel's, where load q + 2 lies 16 rows on (rows past M: beyond the descriptor by the lane's offset)
    int xo[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int r = 8 * (ws_ * MT + q) + (lane >> 3);
        xo[q] = r * K * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    // the lanes whose piece of 8 elements lies in the upper half of a half block: of even loads, odd ones the others
    const bool upper = (lane >> 2) & 1;
    auto dma = [&](int i, int hf, int rh, int slot, int q) {  // load q of a unit of block i
        // K may end inside the last block, at groups of 32 inside the half: zeros for the pieces past it, not the next row
        const int left = K - i * 128 - hf * 64;
        const __amdgpu_buffer_rsrc_t rs = (SETS > 1 ? left > 0 : i < NB) ? (rh ? rs_x1 : rs_x0) : rs_none;
        int rows16 = 32 * K;
        asm volatile("" : "+s"(rows16));
        int off = q < 2 ? xo[q] : xo[q & 1] + rows16;
        if constexpr (SETS == 4) {
            // f16: from the first load's offset, one register less - eight rows on, and the piece's half the other one
            if (q && !BF) off = xo[0] + ((q & 1) ? (upper ? rows16 / 2 - 64 : rows16 / 2 + 64) : 0) + (q >> 1) * rows16;
            off = left < 64 && upper == !(q & 1) ? OOB : off;
        }
        pk4g_load_lds16(rs, pk4_lds + slot * STAGE + kq * TILE + ws_ * (MT * 1024) + q * 1024, off, i * 256 + hf * 128);
    };
    // fragment of a half block's first step, row tile mt (+ 2048 mt): row ni; the second step's is a bit of the piece away
    constexpr int STEP = SETS == 4 ? 64 : 16;
    const int a_rd = kq * TILE + ni * 128 + (((pk4_x_chunk<SETS>(0, kb) & 7) ^ ((ni >> 1) & 7)) << 4);
    const NibbleMasks nm = nibble_masks();

    // a block of weights by step; 16-column strips: by half block (two of a lane's four words, so that a half's registers are
    // free before the next one's are used) and strip
    u32x4_t wring[NARROW ? 1 : 4];
    u32x2_t wnarrow[2][4];
    uint32_t zring[SETS];
    auto load_w = [&](int i, int st) {
        wring[st] = __builtin_amdgcn_raw_buffer_load_b128(i < NB ? rs_w : rs_none, lane_again() * 16, i * BB + st * 1024, 0);
    };
    auto load_narrow = [&](int i, int hf) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
        const int at = lane_again() * 16 + 8 * hf;
#pragma unroll
        for (int f = 0; f < 4; ++f) wnarrow[hf][f] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, at, (f * NB + i) * BB, 0));
    };
    // the pairs of a lane's four columns: lane group f brings those of column (strip) f, pk4_pair_words hands them round
    auto load_z = [&](int i, int set) {
        const int l = lane_again(), at = NARROW ? (l >> 4) * (NB * BB) + 1024 + (l & 15) * 4 : 4096 + ((l & 15) * 4 + (l >> 4)) * 4;
        zring[set] = __builtin_amdgcn_raw_buffer_load_b32(i < NB ? rs_w : rs_none, at, i * BB + set * 256, 0);
    };

    // The compiler orders nothing against the loads into LDS: the waits for them count the younger loads, whose order
    // the barriers of the scheduler keep.
#pragma unroll
    for (int q = 0; q < MT; ++q) dma(kq, 0, 0, 0, q);
#pragma unroll
    for (int q = 0; q < MT; ++q) dma(kq, 0, 1, 1, q);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < SETS; ++u) load_z(kq, u);
    if constexpr (NARROW) {
        load_narrow(kq, 0), load_narrow(kq, 1);
    } else {
#pragma unroll
        for (int st = 0; st < 4; ++st) load_w(kq, st);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rh = 0; rh < 2; ++rh)
#pragma unroll
        for (int q = 0; q < MT; ++q) dma(kq, 1, rh, 2 + rh, q);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[2 * MT][4];
#pragma unroll
    for (int mt = 0; mt < 2 * MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    // Raw barriers, as in pk4_mid_kernel: a wave's own reads of LDS are over before it arrives.
    auto meet = [&](auto younger) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(younger)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    auto column = [](int n) { return PAIRED ? (n >> 1) | ((n & 1) << 1) : n; };  // the n-th column worked on
    uint32_t pairs[4];  // f16: a column's constants in the two halves of a register, which the packed instructions select from
    Pk4gBf16 cb[4];
    Pk4N<TT> cst[4];
    auto constants = [&](int set) {  // of a group that the ring holds
        uint32_t zv[4];
        pk4_pair_words(zring[set], zv);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if constexpr (BF) cb[f].set(__builtin_bit_cast(float, zv[f] & 0xFFFF0000u), __builtin_bit_cast(float, zv[f] << 16) + (NARROW ? 0.0f : 128.0f));
            else if constexpr (NARROW) cst[f].prep(zv[f]);
            else pairs[f] = zv[f];
        }
    };
    auto deq_f16 = [](uint32_t q, uint32_t pair) {  // Pk4T<F16Traits>::deq
        const half2_t c = __builtin_bit_cast(half2_t, pair), zero = __builtin_shufflevector(c, c, 0, 0), scale = __builtin_shufflevector(c, c, 1, 1);
        return __builtin_bit_cast(uint32_t, (__builtin_bit_cast(half2_t, q) + zero) * scale);
    };
    uint32_t b[8][4];  // half a block's fragments: (step, column worked on)
    // fragments 2 ph and 2 ph + 1 of step st
    auto pair = [&](int st, auto ph_c) {
        constexpr int PH = decltype(ph_c)::value;
        const int at = 4 * (st & 1) + 2 * PH;
        if constexpr (NARROW) {
#pragma unroll
            for (int f = 2 * PH; f < 2 * PH + 2; ++f) {
                uint32_t(&o)[4] = b[at + (f & 1)];
                if constexpr (BF) {
                    cb[f].rows(wnarrow[st >> 1][f][st & 1], o);
                } else {
                    Pk4N<TT> c = cst[f];
                    c.odd_from_even();
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) o[pp] = c.deq(TT::unpack1(wnarrow[st >> 1][f][st & 1], pp, nm), pp);
                }
            }
        } else {
            const u32x4_t wv = wring[st];
            const uint32_t wp[4] = {wv[0], wv[1], wv[2], wv[3]};
            if constexpr (BF) {
                pk4g_columns<PH>(wp, cb[PH], cb[2 + PH], b[at], b[at + 1]);
            } else {
#pragma unroll
                for (int f = 2 * PH; f < 2 * PH + 2; ++f)
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) b[at + (f & 1)][pp] = deq_f16(TT::unpack1(wp[pp], f, nm), pairs[f]);
            }
        }
    };
    constexpr std::integral_constant<int, 0> P0{};
    constexpr std::integral_constant<int, 1> P1{};
    u32x4_t a[2][MT];  // fragments of x: the two steps
    auto read_x = [&](int slot, int st) {
        const unsigned char *from = pk4_lds + ((slot * STAGE + a_rd) ^ (st ? STEP : 0));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[st][mt] = *(const u32x4_t *)(from + mt * 2048);
    };
    // The first two units, counting as younger only the loads into LDS (the compiler may issue the ring loads behind this wait).
    meet(std::integral_constant<int, 2 * MT>{});
    read_x(0, 0);
    constants(0);
    pair(0, P0), pair(0, P1);
    __builtin_amdgcn_sched_barrier(0);

    constexpr int V = !BF ? 2 : PAIRED ? 3 : 4;  // vector instructions behind an MFMA where fragments are made
    // The order of a stretch: `mem` requests, `first` MFMAs, `reads` of LDS, `then` MFMAs.
    auto order = [](auto mem, auto first, auto reads, auto then, auto valu) {
        __builtin_amdgcn_sched_group_barrier(0x120, decltype(mem)::value, 0);
#pragma unroll
        for (int n = 0; n < decltype(first)::value; ++n) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (decltype(valu)::value) __builtin_amdgcn_sched_group_barrier(0x002, decltype(valu)::value, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, decltype(reads)::value, 0);
#pragma unroll
        for (int n = 0; n < decltype(then)::value; ++n) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (decltype(valu)::value) __builtin_amdgcn_sched_group_barrier(0x002, decltype(valu)::value, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#define OXQ_N(v) std::integral_constant<int, (v)>{}
    // One unit, out of stage `slot`: rows half RH of block half HF.  The next unit's first step is read out of `next`, and
    // `free`, the stage of the unit before, takes the unit of the next round.
    auto unit = [&](int r, auto hf_c, auto rh_c, int slot) {
        constexpr int HF = decltype(hf_c)::value, RH = decltype(rh_c)::value;
        const int i = KS * r + kq, i1 = i + KS;
        const int next = slot == NS - 1 ? 0 : slot + 1, free = slot == 0 ? NS - 1 : slot - 1;
        auto multiply = [&](int c) {
            const uint32_t(&bc)[4] = b[c];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const uint32_t av[4] = {a[c >> 2][mt][0], a[c >> 2][mt][1], a[c >> 2][mt][2], a[c >> 2][mt][3]};
                acc[RH * MT + mt][column(c & 3)] = Ops::mfma(av, bc, acc[RH * MT + mt][column(c & 3)]);
            }
        };
        if constexpr (RH == 0) {
            if constexpr (!NARROW) load_w(i1, 2 * HF);  // the step that the unit before has left
            if constexpr (HF == 0 || SETS > 1) load_z(i1, SETS == 4 ? 2 * HF : HF);  // its group
            dma(i1, HF, RH, free, 0), dma(i1, HF, RH, free, 1);
            read_x(slot, 1);
            if constexpr (SETS == 4) constants(2 * HF + 1);
            pair(2 * HF + 1, P0);
            multiply(0), multiply(1), multiply(2);
            order(OXQ_N(2 + MT + (NARROW ? 1 - HF : SETS > 1 ? 2 : 2 - HF)), OXQ_N(12), OXQ_N(0), OXQ_N(0), OXQ_N(V));
            dma(i1, HF, RH, free, 2);
            pair(2 * HF + 1, P1);
            multiply(3);
            read_x(next, 0);
            multiply(4), multiply(5);
            order(OXQ_N(1), OXQ_N(4), OXQ_N(4), OXQ_N(8), OXQ_N(V));
            if constexpr (NARROW) load_narrow(i1, HF);
            else load_w(i1, 2 * HF + 1);
            if constexpr (SETS == 4) load_z(i1, 2 * HF + 1);
            dma(i1, HF, RH, free, 3);
            multiply(6), multiply(7);
            order(OXQ_N(NARROW ? 5 : SETS == 4 ? 3 : 2), OXQ_N(8), OXQ_N(0), OXQ_N(0), OXQ_N(0));
        } else {
            dma(i1, HF, RH, free, 0), dma(i1, HF, RH, free, 1);
            read_x(slot, 1);
            multiply(0), multiply(1);
            order(OXQ_N(2 + MT), OXQ_N(8), OXQ_N(0), OXQ_N(0), OXQ_N(0));
            dma(i1, HF, RH, free, 2);
            if constexpr (HF == 1 || SETS > 1) constants(HF == 1 ? 0 : SETS / 2);
            pair(2 - 2 * HF, P0);
            multiply(2), multiply(3);
            read_x(next, 0);
            multiply(4);
            order(OXQ_N(1), OXQ_N(8), OXQ_N(4), OXQ_N(4), OXQ_N(V));
            dma(i1, HF, RH, free, 3);
            pair(2 - 2 * HF, P1);
            multiply(5), multiply(6), multiply(7);
            order(OXQ_N(1), OXQ_N(12), OXQ_N(0), OXQ_N(0), OXQ_N(V));
        }
        // The unit after the next is in LDS: the loads of this and the unit before are younger.
        meet(OXQ_N(2 * MT + (HF == 0 ? RE : RO)));
        return next;
    };
    int slot = 0;
    for (int r = 0; r < NR; ++r) {
        slot = unit(r, P0, P0, slot);
        slot = unit(r, P0, P1, slot);
        slot = unit(r, P1, P0, slot);
        slot = unit(r, P1, P1, slot);
    }
#undef OXQ_N
    meet(std::integral_constant<int, 0>{});  // the stages past the end have been zeroed: nothing lands in LDS any more

    const int l = lane_again();
    // 64 rows at a time: slot of wave w: [mt][e][lane] x float4 (f = 0..3); wave kq of a column group finishes row tile kq
    float4_t *red = (float4_t *)pk4_lds;
#pragma unroll
    for (int rh = 0; rh < 2; ++rh) {
        if (rh) __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                red[((wave * MT + mt) * 4 + e) * 64 + l] =
                    float4_t{acc[rh * MT + mt][0][e], acc[rh * MT + mt][1][e], acc[rh * MT + mt][2][e], acc[rh * MT + mt][3][e]};
        __syncthreads();
        if (!live) continue;
        float4_t fin[4];  // row 64 rh + 16 kq + 4 kb + e
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            fin[e] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k)  // K order: the same sum whatever the timing
                fin[e] += red[(((k * SPW + ws_) * MT + kq) * 4 + e) * 64 + l];
        }
        pk4m_store<TT, NARROW>(fin, bias, y, M, N, j, l & 15, m0 + ROWS * rh + 16 * kq + 4 * (l >> 4), act);
    }
}

template <typename TT, int SETS, bool NARROW>
static int mid128_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)PK4H_STAGES * PK4M_KS * 16 * PK4M_MT * 128;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4_mid128_kernel<TT, SETS, NARROW>, lds));
    hipLaunchKernelGGL((pk4_mid128_kernel<TT, SETS, NARROW>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw,
                       (const uint16_t *)p.bias, (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <typename TT>
static int mid128_layout(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    if (p.w.strip == 16) return mid128_go<TT, 1, true>(s, grid, p, NG);
    switch (pk4_sets(p.w.group_shift)) {
    case 1: return mid128_go<TT, 1, false>(s, grid, p, NG);
    case 2: return mid128_go<TT, 2, false>(s, grid, p, NG);
    default: return mid128_go<TT, 4, false>(s, grid, p, NG);
    }
}

int launch_pk4_mid128(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG) {
    return p.w.dtype == OXQ_F16 ? mid128_layout<F16Traits>(s, grid, p, NG) : mid128_layout<BF16Traits>(s, grid, p, NG);
}

}  // namespace oxq
