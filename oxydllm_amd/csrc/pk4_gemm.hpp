// pk4_gemm_kernel: the prefill kernel of the resident 64-column layout (described in pk4_gemm.hip), for quantization
// groups of 32, 64 and 128 or more rows.
#pragma once

#include "pk4_common.hpp"

namespace oxq {

constexpr int PK4G_STRIPS = 8;  // strips (= waves) of a workgroup

// The integers bias + q of the folded form as pairs of 16-bit floats, with the smallest bias that a pair comes out of the
// word with two instructions: what the bias adds to a group's sum is taken out again in f32, and the rounding of that sum
// grows with it.  pair(): row pair pp of column f from word pp of the column's half; offset(): what the copy's
// pair word (-(bias_f + z) of Pk4T) lacks to -(BIAS + z).
template <typename TT, int BITS> struct Pk4Fold {
    static constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    static constexpr int AT = BF ? 3 : 6;  // 4 bits: mantissa bit of the nibble's lowest at an exponent of 16
    static constexpr float BIAS = BITS == 4 ? 16.0f : BF ? 0.0f : 256.0f;
    __device__ static __forceinline__ uint32_t pair(uint32_t word, int f) {
        if constexpr (BITS == 4) {
            const int left = AT - 4 * f;
            return ((left >= 0 ? word << left : word >> -left) & ((0xFu << AT) * 0x10001u)) | (BF ? 0x41804180u : 0x4C004C00u);
        } else if constexpr (BF) {
            return TT::unpack_bytes((f & 1) ? (word >> 8) : word);
        } else {
            return (((f & 1) ? word >> 6 : word << 2) & 0x03FC03FCu) | 0x5C005C00u;
        }
    }
    __device__ static __forceinline__ float offset(int f) {
        return BITS == 4 ? (BF ? 112.0f : (f & 1) ? 48.0f : 1008.0f) : BF ? 0.0f : 768.0f;
    }
};

// Eight strips a workgroup, a wave takes every block of its strip.
// SETS: as in pk4_mfma_kernel (groups of 128 rows and more, 64, 32).
// FOLD (layers with `unrounded`): the folded form of pk4_mfma_kernel - the matrix cores multiply x by the integers, one
// more MFMA a step against ones yields the row sums of x, and a group's sums enter the accumulators through
// s * (sum - (bias + z) * rowsum), all f32.
// Rows from m0 on, strip group g.
template <typename TT, int MT, int BITS, int SETS, bool FOLD>
__device__ __forceinline__ void pk4_gemm_tile(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                              const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, int M, int K, int N,
                                              int m0, int g, int act) {
    typedef MfmaOps<TT> Ops;
    constexpr int ROWS = 16 * MT, BB = pk4_block_words(BITS, SETS) * 4, XBUF = ROWS * 256;
    constexpr int WL = BITS / 4;          // 1 KB weight loads a step (8-bit: column pairs 0, 1 and 2, 3)
    constexpr int RING = 4 * WL + SETS;      // ring loads of a block: younger than the block's loads of x
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    constexpr int SPS = 4 / SETS;         // steps that share a set of pairs
    constexpr int XV = ROWS / 4 / PK4G_STRIPS;  // loads of x a wave issues per block: 64 lanes x 16 bytes = 4 rows each
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int j = g * PK4G_STRIPS + wave;
    const bool live = j < ((N + 63) >> 6);  // wave-uniform: the last group of a layer may have fewer strips
    const int NB = SETS > 1 ? (K + 127) >> 7 : K >> 7;
    const int xrows = min(M - m0, ROWS);

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl = make_rsrc(pw + (size_t)(live ? j : 0) * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const int voff_w = lane * 16;
    const int voff_z = 1024 * WL * 4 + (ni * 4 + kb) * 4;
    // x: load q of a wave brings rows 4 (XV wave + q) .. + 3 of a block straight into LDS, lane l
    // the 16 bytes that belong at position l % 16 of row l / 16 - chunk (l % 16) ^ (row % 16) of the row, the
    // swizzle the fragment reads undo.  Rows past M lie beyond the descriptor: LDS receives zeros.
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (wave * XV + q) + (lane >> 4);
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
    auto dma_x = [&](int i) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_x : rs_none;
        if constexpr (SETS > 1) {
            if (i == NB - 1 && (K & 127)) {  // K ends inside the block: zeros for the chunks past it, not the next row
#pragma unroll
                for (int q = 0; q < XV; ++q) {
                    const int r = 4 * (wave * XV + q) + (lane >> 4), chunk = (lane & 15) ^ (r & 15);
                    pk4g_load_lds16(rs, pk4_lds + (i & 1) * XBUF + (wave * XV + q) * 1024,
                                    i * 128 + 8 * chunk < K ? xo[q] : 0x7FFFFF00, i * 256);
                }
                return;
            }
        }
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (i & 1) * XBUF + (wave * XV + q) * 1024, xo[q], i * 256);
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

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
#pragma unroll
    for (int u = 0; u < SETS; ++u) load_z(0, u);
#pragma unroll
    for (int st = 0; st < 4; ++st) load_w(0, st);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    pk4g_wait_vmcnt<RING>();
    __syncthreads();

    for (int i = 0; i < NB; ++i) {
        // the other buffer was last read in the previous block, which every wave has left (the barrier below)
        dma_x(i + 1);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *buf = pk4_lds + (i & 1) * XBUF;
        uint32_t zv[4], negzb[4], sp[4];
        Pk4gBf16 cb[4];
        auto constants = [&](int set) {  // of a set of pairs; then the next block's are requested
        pk4_pair_words(zring[set], zv);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if constexpr (BF) {  // the pair word holds {-(bias + z), s}, bias = 128 for nibbles and 0 for bytes
                cb[f].set(__builtin_bit_cast(float, zv[f] & 0xFFFF0000u), __builtin_bit_cast(float, zv[f] << 16) + (BITS == 4 ? 128.0f : 0.0f));
            } else {
                Pk4T<TT>::prep(zv[f], negzb[f], sp[f]);
            }
        }
        load_z(i + 1, set);
        };
        float4_t tmp[FOLD ? MT : 1][4], tmps[FOLD ? MT : 1];  // a group's sums of the folded form
        auto fold = [&](int set) {
            pk4_pair_words(zring[set], zv);
            load_z(i + 1, set);
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const float sf = TT::to_f32((uint16_t)(zv[f] >> 16)), nz = TT::to_f32((uint16_t)(zv[f] & 0xFFFFu)) + Pk4Fold<TT, BITS>::offset(f);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[mt][f][e] = fmaf(sf, fmaf(nz, tmps[mt][e], tmp[mt][f][e]), acc[mt][f][e]);
            }
        };
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (!FOLD && st % SPS == 0) constants(st / SPS);
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
            auto column = [&](int f, const uint32_t (&b)[4]) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
            };
            if constexpr (FOLD) {
                const bool fresh = st % SPS == 0;  // a group's sums start from zero: no clearing
                const float4_t zero4 = float4_t{0.f, 0.f, 0.f, 0.f};
                const uint32_t ones[4] = {TT::ONES, TT::ONES, TT::ONES, TT::ONES};
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    uint32_t b[4];
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) b[pp] = Pk4Fold<TT, BITS>::pair(wp[(f >> 1) % WL][pp], f);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) tmp[mt][f] = Ops::mfma(a[mt], b, fresh ? zero4 : tmp[mt][f]);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) tmps[mt] = Ops::mfma(a[mt], ones, fresh ? zero4 : tmps[mt]);
            } else if constexpr (BF && BITS == 4 && MT == 4) {
                // 64-row workgroups share a CU in pairs with up to 128 registers, which two columns at a time exceed
                // (135: 4096 x 14336 at 1536 rows 195 -> 216 us): one column, a conversion a weight.  The high nibbles
                // stay where they are: bytes of 16 q, times s / 16.
                uint32_t tl[4], th[4];
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                    tl[pp] = pk4g_low(wp[0][pp]), th[pp] = wp[0][pp] & 0xF0F0F0F0u;
                    asm volatile("" : "+v"(tl[pp]), "+v"(th[pp]));  // the masks stay here: folded into the byte extracts they cost one each
                }
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    uint32_t b[4];
                    Pk4gBf16 c = cb[f];
                    if (f & 1) c.s *= 0.0625f;
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) {
                        const uint32_t v = (f & 1) ? th[pp] : tl[pp];
                        b[pp] = (f >> 1) ? c.template bytes<1>(v) : c.template bytes<0>(v);
                    }
                    column(f, b);
                }
            } else if constexpr (BF && BITS == 4) {
                uint32_t b0[4], b2[4];
                pk4g_columns<0>(wp[0], cb[0], cb[2], b0, b2);
                column(0, b0), column(2, b2);
                pk4g_columns<1>(wp[0], cb[1], cb[3], b0, b2);
                column(1, b0), column(3, b2);
            } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    uint32_t b[4];
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) {
                        if constexpr (BITS == 8) {
                            // word pp of half f / 2: bytes {row 2 pp, row 2 pp + 1} x {column 2 h, 2 h + 1}: the pair of
                            // column f in bytes f % 2 and f % 2 + 2
                            const uint32_t word = wp[f >> 1][pp];
                            if constexpr (BF) b[pp] = (f & 1) ? cb[f].template bytes<1>(word) : cb[f].template bytes<0>(word);
                            else b[pp] = Pk4T<TT>::deq(TT::unpack_bytes((f & 1) ? (word >> 8) : word), negzb[f], sp[f]);
                        } else {
                            b[pp] = Pk4T<TT>::deq(TT::unpack1(wp[0][pp], f, nm), negzb[f], sp[f]);
                        }
                    }
                    column(f, b);
                }
            }
            load_w(i + 1, st);  // into the registers this step has just left
            if constexpr (FOLD) {
                if ((st + 1) % SPS == 0) fold(st / SPS);
                __builtin_amdgcn_sched_barrier(0);  // one step's operands in the registers at a time
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        pk4g_wait_vmcnt<RING>();  // this wave's part of the next block of x is in LDS; its ring loads may still fly
        __syncthreads();
    }

    if (!live) return;
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
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * t + 4 * kb + e;
                float mine[4], other[4];
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    mine[f] = TT::to_f32(TT::from_f32(acc[t][f][e] + bv[f]));
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
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + 16 * t + 4 * kb + e;
            if (row >= M) continue;
            const uint32_t o0 = TT::from_f32(acc[t][0][e] + bv[0]), o1 = TT::from_f32(acc[t][1][e] + bv[1]);
            const uint32_t o2 = TT::from_f32(acc[t][2][e] + bv[2]), o3 = TT::from_f32(acc[t][3][e] + bv[3]);
            *(uint2 *)(y + (size_t)row * N + 64 * j + 4 * ni) = uint2{o0 | (o1 << 16), o2 | (o3 << 16)};
        }
}

// LIGHT: the rows behind the RT whole tiles, at most 16 LIGHT, are a tile of their own size in the NG workgroups after them.
template <typename TT, int MT, int BITS, int SETS = 1, bool FOLD = false, int LIGHT = 0>
__global__ __launch_bounds__(512) void pk4_gemm_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                       const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                       int M, int K, int N, int NG, int RT, int act) {
    int rt, g;
    if constexpr (LIGHT > 0) {
        const int whole = RT * NG;
        if ((int)blockIdx.x >= whole + NG) return;
        if ((int)blockIdx.x >= whole) {
            pk4_gemm_tile<TT, LIGHT, BITS, SETS, FOLD>(x, pw, bias, y, M, K, N, RT * 16 * MT, (int)blockIdx.x - whole, act);
            return;
        }
    }
    if ((int)blockIdx.x >= RT * NG) return;  // the whole workgroup, before any barrier
    pk4g_tile_of((int)blockIdx.x, RT, NG, rt, g);
    pk4_gemm_tile<TT, MT, BITS, SETS, FOLD>(x, pw, bias, y, M, K, N, rt * 16 * MT, g, act);
}

template <typename TT, int MT, int BITS, int SETS, bool FOLD = false, int LIGHT = 0>
static int pk4_gemm_wide_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)2 * 16 * MT * 256;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4_gemm_kernel<TT, MT, BITS, SETS, FOLD, LIGHT>, lds));
    hipLaunchKernelGGL((pk4_gemm_kernel<TT, MT, BITS, SETS, FOLD, LIGHT>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw, (const uint16_t *)p.bias,
                       (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, RT, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

}  // namespace oxq
