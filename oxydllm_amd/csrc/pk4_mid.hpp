// pk4_mid_kernel: resident layers between the decode forms and the prefill forms (33 to a few hundred rows; narrow
// layers up to about 1500), where workgroups of eight strips would leave most of the chip idle and workgroups of a single
// strip read x once per 64 columns.
//
// A workgroup is 64 rows x two groups of 64 columns; the four waves of a column group take every fourth block of K, at the
// end the partial tiles meet in LDS (where x was) and wave kq of a group finishes row tile kq, adding the four partials
// in K order.
//
// What bounds it: one workgroup a CU (128 KB of LDS) is two waves a SIMD, which issue 64 MFMAs of 17 clocks and 230
// (f16) or 340 (bf16) vector instructions of 4.5 clocks a block each; with both streams of memory switched off 14336 x
// 14336 at 64 rows takes 50 / 61 us of its 55 / 64.  So the loop is arranged for the issue port: x comes in half blocks
// (64 elements of K) through four stages of LDS, a fragment is read half a block before its MFMA, a column's dequant
// stands between the MFMAs of the column before, and loads and LDS reads are dealt over the columns - all eight waves
// issuing theirs right behind a barrier kept the address and LDS units busy for a third of the half block while the
// matrix cores waited.  Against one block of x a round behind one barrier, everything read where it is used (us, 64-row
// tiles, bf16 with pk4g_widen, called back to back; graph replays are 1 - 2 us shorter): 14336 x 4096 at 384 rows f16 60.6 ->
// 59.6, bf16 71.4 -> 65.0; 4096 x 14336 at 128 rows 22.4 -> 21.6, 24.1 -> 22.4; 8-bit f16 4096 x 14336 at 128 / 256 rows 26.3 /
// 45.6 -> 27.0 / 47.0.  Deeper requests alone (two blocks of weights, three stages of x) changed nothing, nor did
// K slices over workgroups on narrow layers (8192 x 8192 at 128 rows 28.6 -> 30.8, 14336 x 4096 at 64 rows 20.1 -> 23.4).
#pragma once

#include "pk4_common.hpp"

#include <type_traits>

namespace oxq {

constexpr int PK4M_MT = 4, PK4M_KS = 4, PK4M_GROUPS = 2, PK4M_STAGES = 4;

// Stores four rows of a lane's four columns: row row0 + e, fin[e][f] of column group j (64 columns).
template <typename TT, bool NARROW>
__device__ __forceinline__ void pk4m_store(const float4_t (&fin)[4], const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                           int M, int N, int j, int ni, int row0, int act) {
    // columns of fin[e][f]: NARROW 64 j + 16 f + ni, else 64 j + 4 ni + f
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (NARROW) {
        if (bias) {
#pragma unroll
            for (int f = 0; f < 4; ++f) bv[f] = TT::to_f32(bias[64 * j + 16 * f + ni]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (row0 + e >= M) continue;
#pragma unroll
            for (int f = 0; f < 4; ++f) y[(size_t)(row0 + e) * N + 64 * j + 16 * f + ni] = TT::from_f32(fin[e][f] + bv[f]);
        }
        return;
    }
    if (act) {
        // Fused gate|up layer, as in pk4_gemm_kernel: lane ni < 8 holds four gate columns, lane ni + 8 of the same row of
        // 16 their up columns; they exchange their values and finish two outputs each.  y is [M, N / 2].
        const int half_n = N >> 1, col = 32 * j + 4 * (ni & 7);
        const bool low = ni < 8;
        if (bias) {
            const uint2 bw = *(const uint2 *)(bias + (low ? 0 : half_n) + col);
            bv[0] = TT::to_f32((uint16_t)(bw.x & 0xFFFFu)), bv[1] = TT::to_f32((uint16_t)(bw.x >> 16));
            bv[2] = TT::to_f32((uint16_t)(bw.y & 0xFFFFu)), bv[3] = TT::to_f32((uint16_t)(bw.y >> 16));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float mine[4], other[4];
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                mine[f] = TT::to_f32(TT::from_f32(fin[e][f] + bv[f]));
                other[f] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, mine[f]), 0x128, 0xF, 0xF, false));
            }
            uint32_t o[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float gq = low ? mine[q] : other[2 + q], uq = low ? other[q] : mine[2 + q];
                o[q] = TT::from_f32(mul_f32_rn(act == 1 ? silu_f32(gq) : gelu_tanh_f32(gq), uq));
            }
            if (row0 + e < M) *(uint32_t *)(y + (size_t)(row0 + e) * half_n + col + (low ? 0 : 2)) = o[0] | (o[1] << 16);
        }
        return;
    }
    if (64 * j + 4 * ni >= N) return;
    if (bias) {
        const uint2 bw = *(const uint2 *)(bias + 64 * j + 4 * ni);
        bv[0] = TT::to_f32((uint16_t)(bw.x & 0xFFFFu)), bv[1] = TT::to_f32((uint16_t)(bw.x >> 16));
        bv[2] = TT::to_f32((uint16_t)(bw.y & 0xFFFFu)), bv[3] = TT::to_f32((uint16_t)(bw.y >> 16));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (row0 + e >= M) continue;
        const uint32_t o0 = TT::from_f32(fin[e][0] + bv[0]), o1 = TT::from_f32(fin[e][1] + bv[1]);
        const uint32_t o2 = TT::from_f32(fin[e][2] + bv[2]), o3 = TT::from_f32(fin[e][3] + bv[3]);
        *(uint2 *)(y + (size_t)(row0 + e) * N + 64 * j + 4 * ni) = uint2{o0 | (o1 << 16), o2 | (o3 << 16)};
    }
}

// NARROW: the layer is stored in strips of 16 columns; a wave's 64 columns are four neighbouring strips and a strip's
// block is one 16-byte load a lane whose words are the block's four steps.  SETS: as in pk4_mfma_kernel.
template <typename TT, int BITS, int SETS, bool NARROW>
__global__ __launch_bounds__(512) void pk4_mid_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                      const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                      int M, int K, int N, int NG, int act) {
    typedef MfmaOps<TT> Ops;
    static_assert(!NARROW || (BITS == 4 && SETS == 1), "16-column strips are a 4-bit layout with groups of 128 rows and more");
    constexpr int MT = PK4M_MT, KS = PK4M_KS, SPW = PK4M_GROUPS, ROWS = 16 * MT;
    constexpr int BB = NARROW ? PK4N_BW * 4 : pk4_block_words(BITS, SETS) * 4;
    constexpr int TILE = ROWS * 128, STAGE = KS * TILE;  // bytes of x: a wave's half block, a stage
    constexpr int WL = BITS / 4;                          // 1 KB weight loads a step (8-bit: column pairs 0, 1 and 2, 3)
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    constexpr bool PAIRED = BF && BITS == 4 && !NARROW;
    constexpr int SPS = 4 / SETS;                         // steps that share a set of pairs
    // ring loads that follow the loads of x in the first and the second half of a block
    constexpr int RE = NARROW ? 8 : 2 * WL + (SETS == 4 ? 2 : 1), RO = NARROW ? 0 : 2 * WL + SETS / 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws_ = wave % SPW, kq = wave / SPW;  // the wave's column group of the workgroup, and its share of K
    // a row tile's column groups are neighbours: the eight XCDs share its rows of x, and with NG a multiple of 8
    // the row tiles of a column group meet on one XCD, whose L2 then holds the group's weights
    const int rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;
    const int j = g * SPW + ws_;
    const bool live = j < ((N + 63) >> 6);  // wave-uniform: the last workgroup of a layer may have one column group
    const int m0 = rt * ROWS;
    const int NB = (K + 127) >> 7, NR = (NB + KS - 1) / KS;  // blocks; rounds of KS blocks
    const int xrows = min(M - m0, ROWS);

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl =
        NARROW ? make_rsrc(pw + (size_t)(live ? 4 * j : 0) * NB * PK4N_BW, 4u * (uint32_t)NB * (uint32_t)BB)
               : make_rsrc(pw + (size_t)(live ? j : 0) * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const int voff_w = lane * 16;
    const int voff_z = NARROW ? 1024 + ni * 4 : 1024 * WL * 4 + (ni * 4 + kb) * 4;

    // x: load q of a wave brings rows 8 (MT ws + q) .. + 7 of the wave's half block straight into LDS, lane l the 16
    // bytes that belong at position l % 8 of row l / 8 - chunk (l % 8) ^ ((row / 2) % 8) of the row, so that the 16 rows
    // that a fragment read takes from one chunk lie in different banks.  Rows past M lie beyond the descriptor: LDS
    // receives zeros.
    int xo[MT];
#pragma unroll
    for (int q = 0; q < MT; ++q) {
        const int r = 8 * (ws_ * MT + q) + (lane >> 3);
        xo[q] = r * K * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    auto dma_x1 = [&](int r, int hf, int stage, int q) {  // load q of half hf of round r
        const int i = KS * r + kq;
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_x : rs_none;
        unsigned char *dst = pk4_lds + stage * STAGE + kq * TILE + ws_ * (MT * 1024) + q * 1024;
        int off = xo[q];
        if constexpr (SETS > 1) {  // K may end inside the last block: zeros for the chunks past it, not the next row
            const int chunk = (lane & 7) ^ (((8 * (ws_ * MT + q) + (lane >> 3)) >> 1) & 7);
            off = i * 128 + hf * 64 + 8 * chunk < K ? off : 0x7FFFFF00;
        }
        pk4g_load_lds16(rs, dst, off, i * 256 + hf * 128);
    };
    auto dma_x = [&](int r, int hf, int stage) {
#pragma unroll
        for (int q = 0; q < MT; ++q) dma_x1(r, hf, stage, q);
    };
    int a_rd[2];  // fragment of a half block's step, row tile mt (+ 2048 mt): row ni
#pragma unroll
    for (int st = 0; st < 2; ++st) a_rd[st] = kq * TILE + ni * 128 + (((pk4_x_chunk<SETS>(st, kb) & 7) ^ ((ni >> 1) & 7)) << 4);
    const NibbleMasks nm = nibble_masks();

    // two blocks of the wave's weights and pairs; wide: by step, narrow: by strip
    u32x4_t wring[2][4][WL], cur[4];
    uint32_t zring[2][NARROW ? 4 : SETS];
    auto load_w = [&](int i, int par, int st) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
        if constexpr (NARROW) {
            wring[par][st][0] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_w, (st * NB + i) * BB, 0);
        } else {
#pragma unroll
            for (int h = 0; h < WL; ++h) wring[par][st][h] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_w, i * BB + (st * WL + h) * 1024, 0);
        }
    };
    auto load_z = [&](int i, int par, int set) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
        zring[par][set] = __builtin_amdgcn_raw_buffer_load_b32(rs, voff_z, NARROW ? (set * NB + i) * BB : i * BB + set * 256, 0);
    };
    // the ring loads of half hf of a block, in the numbers that RE and RO state
    auto load_half = [&](int i, int par, int hf) {
        if constexpr (NARROW) {
            if (hf == 0) {
#pragma unroll
                for (int f = 0; f < 4; ++f) load_w(i, par, f);
#pragma unroll
                for (int f = 0; f < 4; ++f) load_z(i, par, f);
            }
        } else {
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                if ((2 * hf + st) % SPS == 0) load_z(i, par, (2 * hf + st) / SPS);
                load_w(i, par, 2 * hf + st);
            }
        }
    };

    // The compiler orders nothing against the loads into LDS: the waits for them count the younger loads, whose order
    // the barriers of the scheduler keep.
    dma_x(0, 0, 0);
    dma_x(0, 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    load_half(kq, 0, 0);
    load_half(kq, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
    dma_x(1, 0, 2);
    __builtin_amdgcn_sched_barrier(0);
    load_half(KS + kq, 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    dma_x(1, 1, 3);
    __builtin_amdgcn_sched_barrier(0);
    load_half(KS + kq, 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    // Raw barriers: __syncthreads would wait for every load into LDS that is under way.  A wave's own reads of LDS are
    // over before it arrives (lgkmcnt), so what follows the barrier may overwrite them.
    auto meet = [&](auto younger) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(younger)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    u32x4_t a[2][2][MT];  // fragments of x: two half blocks
    auto read_x = [&](int stage, u32x4_t (&dst)[2][MT]) {
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) dst[st][mt] = *(const u32x4_t *)(pk4_lds + stage * STAGE + mt * 2048 + a_rd[st]);
    };
    // The first two stages, counting as younger only the loads of the other two: the compiler may issue the ring loads
    // above where they are first used, behind this wait (it does so with the second block's), but not those into LDS.
    meet(std::integral_constant<int, 2 * MT>{});
    read_x(0, a[0]);
    __builtin_amdgcn_sched_barrier(0);
    meet(std::integral_constant<int, 63>{});

    auto column = [](int n) { return PAIRED ? (n >> 1) | ((n & 1) << 1) : n; };  // the n-th column worked on
    uint32_t negzb[4], sp[4];
    Pk4gBf16 cb[4];
    Pk4N<TT> cst[4];
    // constants of column f from its pair word
    auto constant = [&](int f, uint32_t zw) {
        if constexpr (NARROW) {  // {-z, s}
            if constexpr (BF) cb[f].set(__builtin_bit_cast(float, zw & 0xFFFF0000u), __builtin_bit_cast(float, zw << 16));
            else cst[f].prep(zw);
        } else if constexpr (BF) {  // {-(bias + z), s}, bias = 128 for nibbles and 0 for bytes
            cb[f].set(__builtin_bit_cast(float, zw & 0xFFFF0000u), __builtin_bit_cast(float, zw << 16) + (BITS == 4 ? 128.0f : 0.0f));
        } else {
            Pk4T<TT>::prep(zw, negzb[f], sp[f]);
        }
    };
    // One half block.  PH = 0..3: half PH % 2 of the block in ring half PH / 2.  Its fragments of x came out of stage PH
    // during the half before; the next half's are read now, and the stage takes the x of four halves on.
    auto half = [&](int r, auto ph_c, auto younger) {
        constexpr int PH = decltype(ph_c)::value, HF = PH & 1, PAR = PH >> 1;
        const int i2 = KS * (r + 2) + kq;  // the block that takes this one's registers; past NB: zeros
        if constexpr (NARROW && HF == 0) {
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                cur[f] = wring[PAR][f][0];
                constant(f, zring[PAR][f]);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_half(i2, PAR, 0);
            __builtin_amdgcn_sched_barrier(0);  // not sunk to the end, where the next block would wait for them
        }
        uint32_t wp[WL][4];
        uint32_t b[2][4], bnext[4];
        // B fragment of the n-th column of step st
        auto frag = [&](int st, int n, uint32_t (&b)[4]) {
            const int f = column(n);
            if constexpr (!NARROW) {
                if (n == 0) {
                    if (st % SPS == 0) {
                        uint32_t zv[4];
                        pk4_pair_words(zring[PAR][st / SPS], zv);
                        constant(0, zv[0]), constant(2, zv[2]), constant(1, zv[1]), constant(3, zv[3]);
                        load_z(i2, PAR, st / SPS);
                    }
#pragma unroll
                    for (int h = 0; h < WL; ++h) {
                        const u32x4_t wv = wring[PAR][st][h];
                        wp[h][0] = wv[0], wp[h][1] = wv[1], wp[h][2] = wv[2], wp[h][3] = wv[3];
                    }
                }
            }
            if constexpr (NARROW && BF) {
                cb[f].rows(cur[f][st], b);
            } else if constexpr (PAIRED) {  // two columns come out of a word's low or high nibbles
                if (n == 0) pk4g_columns<0>(wp[0], cb[0], cb[2], b, bnext);
                else if (n == 2) pk4g_columns<1>(wp[0], cb[1], cb[3], b, bnext);
                else b[0] = bnext[0], b[1] = bnext[1], b[2] = bnext[2], b[3] = bnext[3];
            } else {
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                    if constexpr (NARROW) {
                        b[pp] = cst[f].deq(TT::unpack1(cur[f][st], pp, nm), pp);
                    } else if constexpr (BITS == 8) {
                        // word pp of half f / 2: bytes {row 2 pp, row 2 pp + 1} x {column 2 h, 2 h + 1}: the pair of
                        // column f in bytes f % 2 and f % 2 + 2
                        const uint32_t word = wp[f >> 1][pp];
                        if constexpr (BF) b[pp] = (f & 1) ? cb[f].template bytes<1>(word) : cb[f].template bytes<0>(word);
                        else b[pp] = Pk4T<TT>::deq(TT::unpack_bytes((f & 1) ? (word >> 8) : word), negzb[f], sp[f]);
                    } else {
                        b[pp] = Pk4T<TT>::deq(TT::unpack1(wp[0][pp], f, nm), negzb[f], sp[f]);
                    }
                }
            }
            if constexpr (!NARROW) {
                if (n == 3) load_w(i2, PAR, st);  // into the registers this step has just left
            }
        };
        // A column's fragment is made while the matrix cores work on the column before, and the loads and LDS reads are
        // dealt over the columns: eight waves that leave a barrier and first issue all of theirs keep the address and
        // LDS units busy for half of the time while the matrix cores wait.
        frag(2 * HF, 0, b[0]);
        __builtin_amdgcn_sched_barrier(0);
        // vector instructions behind an MFMA, for an even and an odd column (paired columns: both with the even one's)
        constexpr int EVEN = (PAIRED ? 36 : BF ? 20 : 12) / MT, ODD = PAIRED ? 1 : EVEN;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c % 2 == 0 && c / 2 < MT) dma_x1(r + 2, HF, PH, c / 2);
            if (c < 2 * MT) a[1 - HF][c / MT][c % MT] = *(const u32x4_t *)(pk4_lds + ((PH + 1) & 3) * STAGE + (c % MT) * 2048 + a_rd[c / MT]);
            if (c < 7) frag(2 * HF + ((c + 1) >> 2), (c + 1) & 3, b[(c + 1) & 1]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const uint32_t av[4] = {a[HF][c >> 2][mt][0], a[HF][c >> 2][mt][1], a[HF][c >> 2][mt][2], a[HF][c >> 2][mt][3]};
                acc[mt][column(c & 3)] = Ops::mfma(av, b[c & 1], acc[mt][column(c & 3)]);
            }
            __builtin_amdgcn_sched_group_barrier(0x120, 2, 0);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (c & 1) __builtin_amdgcn_sched_group_barrier(0x002, EVEN, 0);
                else __builtin_amdgcn_sched_group_barrier(0x002, ODD, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        meet(younger);
    };
    {
        // This wave's part of the stage after the next is in LDS: all loads of the last two halves are younger.  In the last
        // round of an odd number nothing uses the weights that are requested, and the compiler leaves those loads out:
        // there only those into LDS count.  (tests/test_wait_counts.py holds the compiled code to it.)
        constexpr std::integral_constant<int, 2 * MT + RE + RO> loads;
        constexpr std::integral_constant<int, 2 * MT> lds_loads;
        int r = 0;
        for (; r + 1 < NR; r += 2) {
            half(r, std::integral_constant<int, 0>{}, loads);
            half(r, std::integral_constant<int, 1>{}, loads);
            half(r + 1, std::integral_constant<int, 2>{}, loads);
            half(r + 1, std::integral_constant<int, 3>{}, loads);
        }
        if (r < NR) {
            half(r, std::integral_constant<int, 0>{}, lds_loads);
            half(r, std::integral_constant<int, 1>{}, lds_loads);
        }
    }
    meet(std::integral_constant<int, 0>{});  // the stages past the end have been zeroed: nothing lands in LDS any more

    // slot of wave w: [mt][e][lane] x float4 (f = 0..3); wave kq of a column group finishes row tile kq
    float4_t *red = (float4_t *)pk4_lds;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            red[((wave * MT + mt) * 4 + e) * 64 + lane] = float4_t{acc[mt][0][e], acc[mt][1][e], acc[mt][2][e], acc[mt][3][e]};
    __syncthreads();
    if (!live) return;
    float4_t fin[4];  // row 16 kq + 4 kb + e
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        fin[e] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KS; ++k)  // K order: the same sum whatever the timing
            fin[e] += red[(((k * SPW + ws_) * MT + kq) * 4 + e) * 64 + lane];
    }
    pk4m_store<TT, NARROW>(fin, bias, y, M, N, j, ni, m0 + 16 * kq + 4 * kb, act);
}

}  // namespace oxq
