// pk4_gemm_kernel: the prefill kernel of the resident 64-column layout (described in pk4_gemm.hip), for quantization
// groups of 32, 64 and 128 or more rows.
#pragma once

#include "pk4_common.hpp"

namespace oxq {

constexpr int PK4G_STRIPS = 8;  // strips (= waves) of a workgroup

// KS = 1: eight strips a workgroup, a wave takes every block of its strip.  KS = 4 (the form for 65 to a few hundred
// rows, where workgroups of eight strips are too few to fill the chip): two strips a workgroup, the four waves of
// a strip take every fourth block; a round brings four blocks of x into LDS, each loaded by the two waves that use
// it; at the end the waves' partial tiles meet in LDS (where x was) and wave kq of a strip finishes row tile kq,
// adding the four partials in K order - the epilogue then runs on the accumulator layout as for KS = 1.
// SETS: as in pk4_mfma_kernel (groups of 128 rows and more, 64, 32).
template <typename TT, int MT, int BITS, int KS, int SETS = 1>
__global__ __launch_bounds__(512) void pk4_gemm_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                       const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                       int M, int K, int N, int NG, int RT, int act) {
    typedef MfmaOps<TT> Ops;
    static_assert(KS == 1 || KS == MT, "wave kq of a strip finishes row tile kq");
    constexpr int SPW = PK4G_STRIPS / KS;  // strips a workgroup
    constexpr int ROWS = 16 * MT, BB = pk4_block_words(BITS, SETS) * 4, XBUF = KS * ROWS * 256;
    constexpr int WL = BITS / 4;          // 1 KB weight loads a step (8-bit: column pairs 0, 1 and 2, 3)
    constexpr int RING = 4 * WL + SETS;      // ring loads of a block: younger than the block's loads of x
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    constexpr int SPS = 4 / SETS;         // steps that share a set of pairs
    constexpr int XV = ROWS / 4 / SPW;  // loads of x a wave issues per round: 64 lanes x 16 bytes = 4 rows each
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws = wave % SPW, kq = wave / SPW;  // the wave's strip of the workgroup, and its share of K
    int rt, g;
    if constexpr (KS == 1) {
        pk4g_tile_of((int)blockIdx.x, RT, NG, rt, g);
        if (g >= NG) return;  // the whole workgroup, before any barrier: the ragged last column of squares
    } else {
        // a row tile's strip groups are neighbours: the eight XCDs share its rows of x, and with NG a multiple of 8
        // the row tiles of a strip group meet on one XCD, whose L2 then holds the group's weights
        rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;
    }
    const int j = g * SPW + ws;
    const bool live = j < ((N + 63) >> 6);  // wave-uniform: the last group of a layer may have fewer strips
    const int m0 = rt * ROWS;
    const int NB = SETS > 1 ? (K + 127) >> 7 : K >> 7, NR = (NB + KS - 1) / KS;  // blocks; rounds of KS blocks
    const int xrows = min(M - m0, ROWS);

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl = make_rsrc(pw + (size_t)(live ? j : 0) * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const int voff_w = lane * 16;
    const int voff_z = 1024 * WL * 4 + (ni * 4 + kb) * 4;
    // x: load q of a wave brings rows 4 (XV ws + q) .. + 3 of the wave's block of the round straight into LDS, lane l
    // the 16 bytes that belong at position l % 16 of row l / 16 - chunk (l % 16) ^ (row % 16) of the row, the
    // swizzle the fragment reads undo.  Rows past M lie beyond the descriptor: LDS receives zeros.
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (ws * XV + q) + (lane >> 4);
        xo[q] = r * K * 2 + (((lane & 15) ^ (r & 15)) << 4);
    }
    int a_rd[4];  // fragment of step st, row tile mt (+ 4096 mt): row ni
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + ((pk4_x_chunk<SETS>(st, kb) ^ ni) << 4);
    const NibbleMasks nm = nibble_masks();

    u32x4_t wring[4][WL];
    uint32_t zring[SETS];
    // The compiler orders nothing against these loads: the wait for them (the ring loads of a block are
    // younger) is written out in front of the barrier that publishes the block.
    // round r: the wave's block is KS r + kq; its tile of x lies at kq ROWS 256 of the round's buffer
    auto dma_x = [&](int r_) {
        const int i = KS * r_ + kq;
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_x : rs_none;
        if constexpr (SETS > 1) {
            if (i == NB - 1 && (K & 127)) {  // K ends inside the block: zeros for the chunks past it, not the next row
#pragma unroll
                for (int q = 0; q < XV; ++q) {
                    const int r = 4 * (ws * XV + q) + (lane >> 4), chunk = (lane & 15) ^ (r & 15);
                    pk4g_load_lds16(rs, pk4_lds + (r_ & 1) * XBUF + kq * (ROWS * 256) + (ws * XV + q) * 1024,
                                    i * 128 + 8 * chunk < K ? xo[q] : 0x7FFFFF00, i * 256);
                }
                return;
            }
        }
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (r_ & 1) * XBUF + kq * (ROWS * 256) + (ws * XV + q) * 1024, xo[q], i * 256);
    };
    auto load_w = [&](int i, int st) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
#pragma unroll
        for (int h = 0; h < WL; ++h) wring[st][h] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_w, i * BB + (st * WL + h) * 1024, 0);
    };
    auto load_z = [&](int i, int set) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
        zring[set] = __builtin_amdgcn_raw_buffer_load_b32(rs, voff_z, i * BB + set * 256, 0);
    };
    auto zs_words = [&](uint32_t z, uint32_t (&zv)[4]) {
        const auto p16 = __builtin_amdgcn_permlane16_swap(z, z, false, false);
        const uint32_t even = p16[0], odd = p16[1];
        const auto pe = __builtin_amdgcn_permlane32_swap(even, even, false, false);
        const auto po = __builtin_amdgcn_permlane32_swap(odd, odd, false, false);
        zv[0] = pe[0], zv[2] = pe[1], zv[1] = po[0], zv[3] = po[1];
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
#pragma unroll
    for (int u = 0; u < SETS; ++u) load_z(kq, u);
#pragma unroll
    for (int st = 0; st < 4; ++st) load_w(kq, st);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    pk4g_wait_vmcnt<RING>();
    __syncthreads();

    for (int r = 0; r < NR; ++r) {
        const int i = KS * r + kq;  // past NB (a ragged last round): zeros from both streams
        // the other buffer was last read in the previous round, which every wave has left (the barrier below)
        dma_x(r + 1);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *buf = pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256);
        uint32_t zv[4], negzb[4], sp[4];
        Pk4gBf16 cb[4];
        auto constants = [&](int set) {  // of a set of pairs; then the next block's are requested
        zs_words(zring[set], zv);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if constexpr (BF) {  // the pair word holds {-(bias + z), s}, bias = 128 for nibbles and 0 for bytes
                cb[f].set(__builtin_bit_cast(float, zv[f] & 0xFFFF0000u), __builtin_bit_cast(float, zv[f] << 16) + (BITS == 4 ? 128.0f : 0.0f));
            } else {
                Pk4T<TT>::prep(zv[f], negzb[f], sp[f]);
            }
        }
        load_z(i + KS, set);
        };
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st % SPS == 0) constants(st / SPS);
            uint32_t wp[WL][4];
#pragma unroll
            for (int h = 0; h < WL; ++h) {
                const u32x4_t wv = wring[st][h];
                wp[h][0] = wv[0], wp[h][1] = wv[1], wp[h][2] = wv[2], wp[h][3] = wv[3];
            }
            uint32_t a[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4_t av = *(const u32x4_t *)(buf + mt * 4096 + a_rd[st]);
                a[mt][0] = av[0], a[mt][1] = av[1], a[mt][2] = av[2], a[mt][3] = av[3];
            }
            uint32_t tl[4], th[4];
            if constexpr (BF && BITS == 4) {
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) pk4g_nibbles(wp[0][pp], tl[pp], th[pp]);
            }
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                uint32_t b[4];
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                    if constexpr (BITS == 8) {
                        // word pp of half f / 2: bytes {row 2 pp, row 2 pp + 1} x {column 2 h, 2 h + 1}: the pair of
                        // column f in bytes f % 2 and f % 2 + 2
                        const uint32_t word = wp[f >> 1][pp];
                        if constexpr (BF) b[pp] = (f & 1) ? cb[f].template pair<1, false>(word) : cb[f].template pair<0, false>(word);
                        else b[pp] = Pk4T<TT>::deq(TT::unpack_bytes((f & 1) ? (word >> 8) : word), negzb[f], sp[f]);
                    } else {
                        // column f of word pp: nibble f of each 16-bit half = the low or high nibble of bytes f / 2 and 2 + f / 2
                        if constexpr (!BF) b[pp] = Pk4T<TT>::deq(TT::unpack1(wp[0][pp], f, nm), negzb[f], sp[f]);
                        else if (f == 0) b[pp] = cb[0].template pair<0, false>(tl[pp]);
                        else if (f == 1) b[pp] = cb[1].template pair<0, true>(th[pp]);
                        else if (f == 2) b[pp] = cb[2].template pair<1, false>(tl[pp]);
                        else b[pp] = cb[3].template pair<1, true>(th[pp]);
                    }
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
            }
            load_w(i + KS, st);  // into the registers this step has just left
        }
        __builtin_amdgcn_sched_barrier(0);
        pk4g_wait_vmcnt<RING>();  // this wave's part of the next round of x is in LDS; its ring loads may still fly
        __syncthreads();
    }

    // the finished tile rows of this wave: all of them (KS = 1), or row tile kq summed over the strip's waves
    float4_t fin[KS == 1 ? MT : 1][4];
    if constexpr (KS == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < 4; ++f) fin[mt][f] = acc[mt][f];
    } else {
        // slot of wave w: [mt][e][lane] x float4 (f = 0..3), 16 KB; the last round's barrier has freed the buffers
        float4_t *red = (float4_t *)pk4_lds;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                red[((wave * MT + mt) * 4 + e) * 64 + lane] = float4_t{acc[mt][0][e], acc[mt][1][e], acc[mt][2][e], acc[mt][3][e]};
        __syncthreads();
#pragma unroll
        for (int f = 0; f < 4; ++f) fin[0][f] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KS; ++k)  // K order: the same sum whatever the timing
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float4_t v = red[(((k * SPW + ws) * MT + kq) * 4 + e) * 64 + lane];
                fin[0][0][e] += v[0], fin[0][1][e] += v[1], fin[0][2][e] += v[2], fin[0][3][e] += v[3];
            }
    }
    if (!live) return;
    constexpr int FT = KS == 1 ? MT : 1;  // row tiles this wave stores: fin[t] is row tile (KS == 1 ? t : kq)
    if (act) {
        // Fused gate|up layer (pk4_src_col): columns 0..31 of the strip are gate columns 32 j .. 32 j + 31, columns
        // 32..63 the up columns they meet - lane ni < 8 holds four gate columns, lane ni + 8 of the same row of 16
        // their up columns.  As in pk4_epilogue: both factors rounded to the layer type (what the projection's own
        // output would hold, ffn.rs:388-400), act(gate) * up in f32, one rounding; y is [M, N / 2].
        // The two lanes of a pair exchange all four values (row_ror:8) and share the work: lane ni takes outputs
        // 0 and 1 of its four columns, lane ni + 8 outputs 2 and 3.
        const int half = N >> 1, col = 32 * j + 4 * (ni & 7);
        const bool low = ni < 8;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias) {
            const uint2 bw = *(const uint2 *)(bias + (low ? 0 : half) + col);
            bv[0] = TT::to_f32((uint16_t)(bw.x & 0xFFFFu)), bv[1] = TT::to_f32((uint16_t)(bw.x >> 16));
            bv[2] = TT::to_f32((uint16_t)(bw.y & 0xFFFFu)), bv[3] = TT::to_f32((uint16_t)(bw.y >> 16));
        }
#pragma unroll
        for (int t = 0; t < FT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * (KS == 1 ? t : kq) + 4 * kb + e;
                float mine[4], other[4];
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    mine[f] = TT::to_f32(TT::from_f32(fin[t][f][e] + bv[f]));
                    other[f] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, mine[f]), 0x128, 0xF, 0xF, false));
                }
                uint32_t o[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const float gq = low ? mine[q] : other[2 + q], uq = low ? other[q] : mine[2 + q];
                    o[q] = TT::from_f32(mul_f32_rn(act == 1 ? silu_f32(gq) : gelu_tanh_f32(gq), uq));
                }
                if (row < M) *(uint32_t *)(y + (size_t)row * half + col + (low ? 0 : 2)) = o[0] | (o[1] << 16);
            }
        return;
    }
    // row 16 mt + 4 kb + e, columns 64 j + 4 ni + f: four neighbours, one 8-byte store
    if (64 * j + 4 * ni >= N) return;  // columns (a multiple of 8) that end inside the last strip
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
        const uint2 bw = *(const uint2 *)(bias + 64 * j + 4 * ni);
        bv[0] = TT::to_f32((uint16_t)(bw.x & 0xFFFFu)), bv[1] = TT::to_f32((uint16_t)(bw.x >> 16));
        bv[2] = TT::to_f32((uint16_t)(bw.y & 0xFFFFu)), bv[3] = TT::to_f32((uint16_t)(bw.y >> 16));
    }
#pragma unroll
    for (int t = 0; t < FT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + 16 * (KS == 1 ? t : kq) + 4 * kb + e;
            if (row >= M) continue;
            const uint32_t o0 = TT::from_f32(fin[t][0][e] + bv[0]), o1 = TT::from_f32(fin[t][1][e] + bv[1]);
            const uint32_t o2 = TT::from_f32(fin[t][2][e] + bv[2]), o3 = TT::from_f32(fin[t][3][e] + bv[3]);
            *(uint2 *)(y + (size_t)row * N + 64 * j + 4 * ni) = uint2{o0 | (o1 << 16), o2 | (o3 << 16)};
        }
}

template <typename TT, int MT, int BITS, int KS, int SETS>
static int pk4_gemm_wide_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)2 * KS * 16 * MT * 256;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4_gemm_kernel<TT, MT, BITS, KS, SETS>, lds));
    hipLaunchKernelGGL((pk4_gemm_kernel<TT, MT, BITS, KS, SETS>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw, (const uint16_t *)p.bias,
                       (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, RT, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

}  // namespace oxq
