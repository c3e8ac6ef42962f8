// Resident MXFP4 experts at prefill sizes (moe.rs:563-607 runs every expert's tokens through its projections;
// mxfp4.rs:119-154 is the layer): the decomposition of pk4n_gemm_kernel on the tile-major expert copy.
//
// The copy (mxfp4_repack_kernel) stores a tile of 16 weight rows as chunks of 1 KB - 128 elements of K, lane
// (ni, kb) the 16 bytes of block 4 c + kb of row ni, whose four words are the chunk's four MFMA steps - which is
// the shape of a block of the 16-column AWQ layout.  So a workgroup takes 16 rows of one expert's pairs and, a wave,
// four neighbouring tiles (64 weight rows = 64 columns of y): the pairs' rows of x come from global memory straight
// into LDS (gathered through the token list, a chunk of K at a time, two buffers, one barrier a chunk), every wave
// streams its tiles through a ring of two chunks, turns a word into an MFMA B fragment with four
// v_cvt_scalef32_pk_bf16_fp4 (the values are exact in bf16, so this is the tile matmul's B) and keeps the whole K in
// its accumulators: mxfp4_gemm_kernel, for few pairs an expert.  With more, mxfp4_wide_kernel below.
// (The K split inside the workgroup that serves AWQ layers at mid sizes was slower than either at every pair count: with
// 32 experts there are always enough workgroups.)
#include "oxq_device.hpp"
#include "oxq_internal.hpp"
#include "oxq_mfma.hpp"
#include "pk4_common.hpp"

#include <type_traits>

namespace oxq {

constexpr int MXG_WAVES = 8;

template <int NW>
__global__ __launch_bounds__(NW * 64) void mxfp4_gemm_kernel(const uint16_t *__restrict__ x, const unsigned char *__restrict__ pw,
                                                             const unsigned char *__restrict__ ps, const uint16_t *__restrict__ bias,
                                                             uint16_t *__restrict__ y, const int32_t *__restrict__ offsets,
                                                             const int32_t *__restrict__ token_ids, int K, int N, int NC, int NG,
                                                             int E, uint32_t x_bytes, int swiglu, float limit) {
    typedef MfmaOps<BF16Traits> Ops;
    constexpr int ROWS = 16, XBUF = ROWS * 256;
    constexpr int OOB = 0x7FFFFF00;
    extern __shared__ __attribute__((aligned(16))) unsigned char mxg_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    // blockIdx.y -> (expert, row tile of its pairs); all values workgroup-uniform
    int rem = blockIdx.y, e = 0;
    for (; e < E; ++e) {
        const int tiles = (offsets[e + 1] - offsets[e] + ROWS - 1) / ROWS;
        if (rem < tiles) break;
        rem -= tiles;
    }
    if (e == E) return;  // the whole workgroup, before any barrier
    const int m0 = offsets[e] + rem * ROWS, m_end = offsets[e + 1];
    const int j = (int)blockIdx.x * NW + wave;  // the wave's 64 columns: tiles 4 j .. 4 j + 3
    const int ntiles = N >> 4, nb = K >> 5;
    const int live_tiles = min(4, ntiles - 4 * j);  // wave-uniform; <= 0: a wave past the last tile
    const bool live = live_tiles > 0;

    const size_t et = (size_t)e * ntiles + (live ? 4 * j : 0);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(pw + et * nb * 256, live ? (uint32_t)live_tiles * (uint32_t)nb * 256u : 0u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(ps + et * NG * 256, live ? (uint32_t)live_tiles * (uint32_t)NG * 256u : 0u);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, x_bytes);
    const int voff_w = lane * 16, voff_s = lane * 4;
    // x: waves 0 .. 3 bring rows 4 wave .. + 3 of a chunk straight into LDS, lane l the 16 bytes that belong at position
    // l % 16 of row l / 16.  Piece p = 4 kb + st of a row's 128 elements (what lane group kb reads in step st) is kept at
    // position (4 st + kb) ^ (row % 16): the four lane groups of a fragment read then start in different banks (at position
    // p ^ row, groups 0 and 2 would meet 128 bytes apart: four conflict cycles a read).
    // Rows past the expert's pairs, and the elements past K in the last chunk, get an offset beyond the descriptor:
    // LDS receives zeros.
    const int r = 4 * wave + (lane >> 4), m = m0 + r, pos = (lane & 15) ^ (r & 15);
    const int xc = ((pos & 3) << 2) | (pos >> 2);  // the piece kept at this position
    int src = 0;
    if (m < m_end) src = token_ids ? token_ids[m] : m;
    const int xo = m < m_end ? src * K * 2 + (xc << 4) : OOB;
    // fragment of step st: row ni, elements 32 kb + 8 st .. + 7 of the chunk = piece 4 kb + st
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + (((4 * st + kb) ^ ni) << 4);

    u32x4_t wring[2][4];
    uint32_t sring[4];
    const bool loads_x = 4 * wave < ROWS;  // wave-uniform
    auto dma_x = [&](int c) {
        const int lim = (K - c * 128) >> 3;  // 16-byte pieces of the row left in this chunk (<= 0 past the row)
        if (!loads_x) return;
        pk4g_load_lds16(rs_x, mxg_lds + (c & 1) * XBUF + wave * 1024, xc < lim ? xo : OOB, c * 256);
    };
    // blocks past the row, and tiles past the layer's last, lie beyond the tile but not beyond what the range check
    // looks at (the lane's offset, not the scalar one): the lane carries an offset that is
    auto load_w = [&](int c, u32x4_t (&w)[4]) {
        const int vo = 4 * c + kb < nb ? voff_w : OOB;
#pragma unroll
        for (int f = 0; f < 4; ++f) w[f] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, f < live_tiles ? vo : OOB, f * nb * 256 + c * 1024, 0);
    };
    auto load_s = [&](int c) {
        const int vo = c < NC ? voff_s : OOB;
#pragma unroll
        for (int f = 0; f < 4; ++f) sring[f] = __builtin_amdgcn_raw_buffer_load_b32(rs_s, f < live_tiles ? vo : OOB, (f * NG + (c >> 2)) * 256, 0);
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
    load_s(0);
    load_w(0, wring[0]);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] = float4_t{0.f, 0.f, 0.f, 0.f};
    pk4g_wait_vmcnt<8>();
    __syncthreads();

    // one chunk, its weights in ring half CUR; eight ring loads are younger than the chunk's loads of x
    auto round = [&](int c, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        dma_x(c + 1);
        __builtin_amdgcn_sched_barrier(0);
        load_w(c + 1, wring[CUR ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *buf = mxg_lds + (c & 1) * XBUF;
        float scale[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) scale[f] = e8m0_to_f32((sring[f] >> (8 * (c & 3))) & 0xFFu);
        load_s(c + 1);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const u32x4_t av = *(const u32x4_t *)(buf + a_rd[st]);
            const uint32_t a[4] = {av[0], av[1], av[2], av[3]};
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const uint32_t w = wring[CUR][f][st];
                uint32_t b[4];
                b[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale[f], 0));
                b[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale[f], 1));
                b[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale[f], 2));
                b[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale[f], 3));
                acc[f] = Ops::mfma(a, b, acc[f]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        pk4g_wait_vmcnt<8>();  // this wave's part of the next chunk of x is in LDS
        __syncthreads();
    };
    {
        int c = 0;
        for (; c + 1 < NC; c += 2) {
            round(c, std::integral_constant<int, 0>{});
            round(c + 1, std::integral_constant<int, 1>{});
        }
        if (c < NC) round(c, std::integral_constant<int, 0>{});
    }

    if (!live) return;
    // lane (ni, kb), value i of acc[f]: pair m0 + 4 kb + i, weight row 64 j + 16 f + ni
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < 4; ++f)
        if (bias && f < live_tiles) bv[f] = BF16Traits::to_f32(bias[(size_t)e * N + 64 * j + 16 * f + ni]);
    // Neighbouring lanes hold neighbouring weight rows: the two lanes of a pair exchange their values (quad_perm
    // [1, 0, 3, 2]) and share the work - the even lane finishes pairs i = 0 and 2 of the four, the odd lane 1 and 3.
    const bool odd = ni & 1;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const int n = 64 * j + 16 * f + (ni & ~1);  // the lane pair's two weight rows: n, n + 1
        float mine[4], other[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // rounded to bf16 as the projection's own output is (for the SwiGLU: what it would read)
            mine[i] = BF16Traits::to_f32(BF16Traits::from_f32(acc[f][i] + bv[f]));
            other[i] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, mine[i]), 0xB1, 0xF, 0xF, false));
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int i = 2 * h + (odd ? 1 : 0);
            const int m = m0 + 4 * kb + i;
            const float lo = odd ? other[2 * h + 1] : mine[2 * h], hi = odd ? mine[2 * h + 1] : other[2 * h];  // rows n, n + 1
            if (m >= m_end || f >= live_tiles) continue;
            if (swiglu) {
                // rows 2 c / 2 c + 1 are the gate / up of output c (moe.rs:152-173)
                y[(size_t)m * (N >> 1) + (n >> 1)] = BF16Traits::from_f32(gpt_oss_swiglu_f32(lo, hi, limit));
            } else {
                *(uint32_t *)(y + (size_t)m * N + n) = (uint32_t)BF16Traits::from_f32(lo) | ((uint32_t)BF16Traits::from_f32(hi) << 16);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// mxfp4_wide_kernel: all the pairs of an expert in one workgroup (up to 128, else even tiles), so that its weights come out
// of HBM and through the conversion once.
//
// What bounds it: at 16 pairs an expert the stream of weights (4.6 TB/s, with a workgroup's prologue and epilogue beside
// its neighbour's loop); at 64 and more the issue port, MFMAs and conversions about equal.  A conversion makes two weights
// and an MFMA of 32 x 32 x 16 takes four of them, so a wave has 32 columns and all the rows, not 64 columns and half of them:
// 16 conversions a unit serve up to 16 MFMAs.  (Waves of 64 columns and 64 rows, the units of K dealt over two sets of
// waves: 113 + 68 us below at 515 tokens, half of the vector instructions; 128 rows of them, one workgroup a CU: 112 + 69.)
// 126 registers and 64 KB of LDS leave room for two workgroups a CU, which is what covers barriers, prologue and
// epilogue: one a CU was up to 30 % slower.  x goes through four stages of LDS, weights through four units of registers.
// Against row tiles of 16 - 128 with 16 x 16 x 32 MFMAs, 32 experts x (5760 + 2880) x 2880, top-4 of random logits, gate_up +
// down in us at 128 / 256 / 515 / 1024 / 2048 tokens: 67 + 41, 91 + 56, 120 + 70, 200 + 108, 322 + 171 -> 63 + 37, 71 + 42,
// 97 + 55, 161 + 94, 273 + 140; 128 experts x (3328 + 1600) x 1600, 1820 tokens: 171 + 98 -> 119 + 69.
// ---------------------------------------------------------------------------
typedef float float16v_t __attribute__((ext_vector_type(16)));

constexpr int MXW_ROWS = 128, MXW_STAGES = 4, MXW_RING = 4;  // rows of a tile; units of x in LDS, of weights in registers

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {  // one hardware conversion, to nearest even
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{lo, hi}, bf16x2_t));
}

// One tile: RT x 32 rows of x (pairs m0 .. m_end - 1 of one expert) by NW groups of 32 columns, a wave each, in
// 32 x 32 x 16 MFMAs over units of 64 elements of K (two blocks).
template <int RT, int NW>
__device__ __forceinline__ void mxw_tile(unsigned char *lds, const uint16_t *__restrict__ x, const unsigned char *__restrict__ pw,
                                         const unsigned char *__restrict__ ps, const uint16_t *__restrict__ bias,
                                         uint16_t *__restrict__ y, const int32_t *__restrict__ token_ids, int K, int N, int NG,
                                         uint32_t x_bytes, int swiglu, float limit, int e, int c0, int m0, int m_end) {
    constexpr int NS = MXW_STAGES, D = MXW_RING;
    constexpr int XL = (4 * RT + NW - 1) / NW;    // loads of x a wave issues a unit, 8 rows each (past the tile: zeros)
    constexpr int STAGE = XL * NW * 1024;         // bytes of x: a unit
    constexpr int OOB = 0x7FFFFF00;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n32 = lane & 31, h = lane >> 5, ni = lane & 15;
    const int j = c0 * NW + wave;                 // the wave's 32 columns: tiles 2 j and 2 j + 1 of 16 weight rows
    const int ntiles = N >> 4, nb = K >> 5, NU = (nb + 1) >> 1;
    const int live_tiles = min(2, ntiles - 2 * j);  // wave-uniform; <= 0: a wave past the last tile
    const bool live = live_tiles > 0;

    const size_t et = (size_t)e * ntiles + (live ? 2 * j : 0);
    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(pw + et * nb * 256, live ? (uint32_t)live_tiles * (uint32_t)nb * 256u : 0u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(ps + et * NG * 256, live ? (uint32_t)live_tiles * (uint32_t)NG * 256u : 0u);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, x_bytes);

    // x: load q of a wave brings rows 8 (XL wave + q) .. + 7 of a unit straight into LDS, lane l the 16 bytes that belong at
    // position l % 8 of row l / 8: piece (l % 8) ^ ((row / 2) % 8), so that the rows a fragment read takes from one piece
    // lie in different banks.  Rows past the tile and elements past K get an offset beyond the descriptor: zeros.
    int xo[XL];
    bool upper[XL];  // the lanes whose piece lies in the second block of a unit
#pragma unroll
    for (int q = 0; q < XL; ++q) {
        const int row = 8 * (XL * wave + q) + (lane >> 3), m = m0 + row, pc = (lane & 7) ^ ((row >> 1) & 7);
        int src = 0;
        if (m < m_end) src = token_ids ? token_ids[m] : m;
        xo[q] = m < m_end ? src * K * 2 + (pc << 4) : OOB;
        upper[q] = pc >= 4;
    }
    auto dma_x = [&](int u, int slot) {
        const __amdgpu_buffer_rsrc_t rs = u < NU ? rs_x : rs_none;
        const bool past = 2 * u + 1 == nb;  // the last unit holds one block
#pragma unroll
        for (int q = 0; q < XL; ++q)
            pk4g_load_lds16(rs, lds + slot * STAGE + (XL * wave + q) * 1024, past && upper[q] ? OOB : xo[q], u * 128);
    };
    // weights: lane (n32, h) the block 2 u + h of weight row n32; step st multiplies the block's word st.  (Past a row's
    // last block: the next row's finite codes, scaled by the 1 that pads the scales, times zeros of x.)
    const int t16 = n32 >> 4;
    const int wo = t16 < live_tiles ? t16 * nb * 256 + h * 256 + ni * 16 : OOB;
    const int so = t16 < live_tiles ? t16 * NG * 256 + (h * 16 + ni) * 4 : OOB;
    u32x4_t wring[D];
    uint32_t sring[D];
    auto load_w = [&](int u, int d) {
        wring[d] = __builtin_amdgcn_raw_buffer_load_b128(u < NU ? rs_w : rs_none, wo, u * 512, 0);
        sring[d] = __builtin_amdgcn_raw_buffer_load_b8(u < NU ? rs_s : rs_none, so, (u >> 3) * 256 + (u & 1) * 128 + ((u >> 1) & 3), 0);
    };
    int a_rd[4];  // fragment of step st, row tile t (+ 4096 t): row n32, piece 4 h + st
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = n32 * 128 + (((4 * h + st) ^ ((n32 >> 1) & 7)) << 4);

    // The waits below count the loads that are younger than the stage that a barrier publishes: requests keep this order.
#pragma unroll
    for (int s = 0; s < D; ++s) {
        if (s < NS - 1) dma_x(s, s);
        __builtin_amdgcn_sched_barrier(0);
        load_w(s, s);
        __builtin_amdgcn_sched_barrier(0);
    }
    float16v_t acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;

    auto round = [&](int u, auto d_c, auto tail_c) {
        constexpr int DI = decltype(d_c)::value;
        constexpr bool TAIL = decltype(tail_c)::value;
        // Own loads of stage u are over.  Younger are those of the NS - 2 stages behind it and the weights requested since;
        // the last rounds, which request no more weights, do not count on any.
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(TAIL ? (NS - 2) * XL : 2 + (NS - 2) * (XL + 2)) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int slot = u % NS;
        dma_x(u + NS - 1, slot == 0 ? NS - 1 : slot - 1);  // the stage read in the round before
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *buf = lds + slot * STAGE;
        const float scale = e8m0_to_f32(sring[DI]);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            u32x4_t a[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t) a[t] = *(const u32x4_t *)(buf + t * 4096 + a_rd[st]);
            const uint32_t w = wring[DI][st];
            u32x4_t b;
            b[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 0));
            b[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 1));
            b[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 2));
            b[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 3));
#pragma unroll
            for (int t = 0; t < RT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[t]), __builtin_bit_cast(bf16x8_t, b), acc[t], 0, 0, 0);
        }
        if constexpr (!TAIL) load_w(u + D, DI);
        __builtin_amdgcn_sched_barrier(0);
    };
    static_assert(D == 4, "the rounds below");
    int u = 0;
    for (; u + D <= NU; u += D) {
        round(u, std::integral_constant<int, 0>{}, std::false_type{});
        round(u + 1, std::integral_constant<int, 1>{}, std::false_type{});
        round(u + 2, std::integral_constant<int, 2>{}, std::false_type{});
        round(u + 3, std::integral_constant<int, 3>{}, std::false_type{});
    }
    if (u < NU) {
        round(u, std::integral_constant<int, 0>{}, std::true_type{});
        if (u + 1 < NU) {
            round(u + 1, std::integral_constant<int, 1>{}, std::true_type{});
            if (u + 2 < NU) round(u + 2, std::integral_constant<int, 2>{}, std::true_type{});
        }
    }

    // lane (n32, h), value 4 q + i of acc[t]: pair m0 + 32 t + 8 q + 4 h + i, weight row 32 j + n32
    const int n = 32 * j + n32;
    const bool col = t16 < live_tiles;
    const float bv = bias && col ? BF16Traits::to_f32(bias[(size_t)e * N + n]) : 0.f;
    // Neighbouring lanes hold neighbouring weight rows: the two lanes of a pair exchange their values (quad_perm
    // [1, 0, 3, 2]) and share the work: the even lane finishes pairs i = 0 and 2 of the four, the odd lane 1 and 3.
    const bool odd = ni & 1;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // rounded to bf16 as the projection's own output is (for the SwiGLU: what it would read)
            uint32_t mine[2], other[2];  // pairs i = 0, 1 and 2, 3
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                mine[g] = bf16_pair(acc[t][4 * q + 2 * g] + bv, acc[t][4 * q + 2 * g + 1] + bv);
                other[g] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine[g], 0xB1, 0xF, 0xF, false);
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int m = m0 + 32 * t + 8 * q + 4 * h + 2 * g + (odd ? 1 : 0);
                // weight rows n & ~1 and n | 1 of pair m
                const uint32_t v = odd ? perm_b32(mine[g], other[g], 0x07060302u) : perm_b32(other[g], mine[g], 0x05040100u);
                if (m >= m_end || !col) continue;
                if (swiglu) {
                    // rows 2 c / 2 c + 1 are the gate / up of output c (moe.rs:152-173)
                    const float r = gpt_oss_swiglu_f32(__builtin_bit_cast(float, v << 16), __builtin_bit_cast(float, v & 0xFFFF0000u), limit);
                    y[(size_t)m * (N >> 1) + (n >> 1)] = (uint16_t)bf16_pair(r, 0.f);
                } else {
                    *(uint32_t *)(y + (size_t)m * N + (n & ~1)) = v;
                }
            }
        }
}

template <int NW>
__device__ __forceinline__ void mxw_workgroup(const uint16_t *__restrict__ x, const unsigned char *__restrict__ pw, const unsigned char *__restrict__ ps,
                                              const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, const int32_t *__restrict__ offsets,
                                              const int32_t *__restrict__ token_ids, int K, int N, int NG, int E, int col_groups, int tiles_bound,
                                              uint32_t x_bytes, int swiglu, float limit) {
    extern __shared__ __attribute__((aligned(16))) unsigned char mxg_lds[];
    const int id = ((int)blockIdx.z * (int)gridDim.y + (int)blockIdx.y) * (int)gridDim.x + (int)blockIdx.x;
    if (id >= tiles_bound * col_groups) return;
    // lane l: expert b + l, its pairs lo .. hi - 1, their tiles, and the tiles up to and with it (every wave does the same)
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = 0, own = 0, upto = 0;
    auto scan = [&](int b) {
        const int ee = b + lane;
        lo = ee < E ? offsets[ee] : 0, hi = ee < E ? offsets[ee + 1] : 0;
        own = upto = (hi - lo + MXW_ROWS - 1) / MXW_ROWS;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(upto, d);
            if (lane >= d) upto += v;
        }
        return __builtin_amdgcn_readlane(upto, 63);
    };
    int total = 0;
    for (int b = 0; b < E; b += 64) total += scan(b);
    const int items = total * col_groups;
    if (id >= items) return;  // the whole workgroup, before any barrier
    // Workgroup i runs on XCD i % 8 (or a rotation of that): an XCD takes a contiguous eighth of the tiles in the order
    // expert, column group, row tile, so that what shares weights or rows of x shares an L2.
    const int xcd = id & 7, item = xcd * (items >> 3) + min(xcd, items & 7) + (id >> 3);
    int e = 0, before = 0, pairs0 = 0, pairs1 = 0;  // the expert whose tiles x column groups hold the item
    for (int b = 0, base = 0; b < E; b += 64) {
        const int last = E > 64 ? scan(b) : total;
        const bool here = (base + upto - own) * col_groups <= item && item < (base + upto) * col_groups;
        const uint64_t found = __ballot(here);
        if (found) {
            const int l = __builtin_ctzll(found);
            e = b + l, before = base + __builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(own, l);
            pairs0 = __builtin_amdgcn_readlane(lo, l), pairs1 = __builtin_amdgcn_readlane(hi, l);
            break;
        }
        base += last;
    }
    // (the compiler does not see that they are the same in all lanes)
    e = __builtin_amdgcn_readfirstlane(e), before = __builtin_amdgcn_readfirstlane(before);
    pairs0 = __builtin_amdgcn_readfirstlane(pairs0), pairs1 = __builtin_amdgcn_readfirstlane(pairs1);
    const int units = (pairs1 - pairs0 + 31) >> 5, tiles = (units + MXW_ROWS / 32 - 1) / (MXW_ROWS / 32);
    const int within = item - before * col_groups, c = within / tiles, t = within % tiles;
    // the units of 32 rows dealt evenly over the tiles, the first ones taking one more
    const int small = units / tiles, more = units % tiles;
    const int u0 = t * small + min(t, more), rt = small + (t < more ? 1 : 0);
    const int m0 = pairs0 + 32 * u0, m_end = min(pairs1, m0 + 32 * rt);
    auto go = [&](auto rt_c) {
        mxw_tile<decltype(rt_c)::value, NW>(mxg_lds, x, pw, ps, bias, y, token_ids, K, N, NG, x_bytes, swiglu, limit, e, c, m0, m_end);
    };
    if (rt == 4) go(std::integral_constant<int, 4>{});
    else if (rt == 3) go(std::integral_constant<int, 3>{});
    else if (rt == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
}

__global__ __launch_bounds__(512, 4) void mxfp4_wide_kernel(const uint16_t *__restrict__ x, const unsigned char *__restrict__ pw,
                                                            const unsigned char *__restrict__ ps, const uint16_t *__restrict__ bias,
                                                            uint16_t *__restrict__ y, const int32_t *__restrict__ offsets,
                                                            const int32_t *__restrict__ token_ids, int K, int N, int NG, int E,
                                                            int col_groups, int tiles_bound, uint32_t x_bytes, int swiglu, float limit) {
    mxw_workgroup<MXG_WAVES>(x, pw, ps, bias, y, offsets, token_ids, K, N, NG, E, col_groups, tiles_bound, x_bytes, swiglu, limit);
}

// Twelve waves, one workgroup a CU: where its workgroups of 384 columns are at most one a CU and those of 256 are more.  Then some CUs
// hold two of the latter and the others one, and the launch lasts as long as 512 columns; 27 % of the time of the 2880 x 2880 experts at
// 515 tokens their CUs stood idle.  us, 256 columns a workgroup -> 384, pairs an expert 3 / 16 / 64: 32 experts of 2880 x 2880 (K x N)
// 31.7 / 31.8 / 51.9 -> 26.3 / 26.0 / 44.8, of 2560 x 2752 25.0 / 26.9 / 45.3 -> 19.8 / 23.8 / 39.3, 64 of 3456 x 1088 31.7 / 32.1 / 55.8 ->
// 25.6 / 26.1 / 46.0.  In two rounds it is behind (5760 columns 58.3 / 87.6 -> 59.5 / 91.3 at 16 / 64 pairs): nothing covers its prologue.
constexpr int MXG_WAVES12 = 12;
__global__ __launch_bounds__(768, 3) void mxfp4_wide12_kernel(const uint16_t *__restrict__ x, const unsigned char *__restrict__ pw,
                                                              const unsigned char *__restrict__ ps, const uint16_t *__restrict__ bias,
                                                              uint16_t *__restrict__ y, const int32_t *__restrict__ offsets,
                                                              const int32_t *__restrict__ token_ids, int K, int N, int NG, int E,
                                                              int col_groups, int tiles_bound, uint32_t x_bytes, int swiglu, float limit) {
    mxw_workgroup<MXG_WAVES12>(x, pw, ps, bias, y, offsets, token_ids, K, N, NG, E, col_groups, tiles_bound, x_bytes, swiglu, limit);
}

// Takes the grouped problem from three pairs an expert on average (below, the decode kernel's passes of four tokens
// read the weights once): 0 = not taken, else the rows of a tile that the grid is sized for, which follow the average (the
// pairs of an expert are only known on the device; workgroups past the last tile leave at once).  They stand in the
// plan's name; mxfp4_wide_kernel's tiles have up to 128 rows whatever the grid.  OXQ_MXFP4_GEMM_ROWS gives them: 32, 64 and 128
// leave the wide kernel alone, 16 lets the rule of launch_mxfp4_res_gemm choose.
int mxfp4_gemm_form(const oxq_ctx *ctx, int64_t n_pairs, int64_t E, int64_t K, int64_t N) {
    const int64_t min_pairs = tune(ctx, OXQ_TUNE_MXFP4_GEMM_MIN_PAIRS, 3);
    if (min_pairs <= 0 || E <= 0 || n_pairs < min_pairs * E || N % 16 != 0 || K % 32 != 0) return 0;
    const int forced = tune(ctx, OXQ_TUNE_MXFP4_GEMM_ROWS, 0);
    if (forced == 16 || forced == 32 || forced == 64 || forced == 128) return forced;
    const int64_t avg = n_pairs / E;
    return avg <= 12 ? 16 : avg < 96 ? 32 : avg < 200 ? 64 : 128;
}

template <int NW>
static int mxfp4_wide_go(hipStream_t s, dim3 grid, const Mxfp4Problem &p, int NG, uint32_t x_bytes) {
    static LdsGrant grant;  // one per instantiation
    constexpr auto kernel = NW == MXG_WAVES12 ? mxfp4_wide12_kernel : mxfp4_wide_kernel;
    const size_t lds = (size_t)MXW_STAGES * ((MXW_ROWS / 8 + NW - 1) / NW) * NW * 1024;
    OXQ_HIP_CHECK(grant.ensure((const void *)kernel, lds));
    const int64_t bound = p.n_pairs / MXW_ROWS + p.n_experts;
    hipLaunchKernelGGL(kernel, grid, dim3(NW * 64), lds, s, (const uint16_t *)p.x, (const unsigned char *)p.blocks,
                       (const unsigned char *)p.scales, (const uint16_t *)p.bias, (uint16_t *)p.y, p.expert_offsets, p.token_ids,
                       (int)p.K, (int)p.N, NG, (int)p.n_experts, (int)ceil_div(p.N, 32 * NW), (int)bound, x_bytes, p.swiglu, p.swiglu_limit);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

static int mxfp4_gemm_go(hipStream_t s, dim3 grid, const Mxfp4Problem &p, int NC, int NG, uint32_t x_bytes) {
    static LdsGrant grant;
    const size_t lds = (size_t)2 * 16 * 256;
    OXQ_HIP_CHECK(grant.ensure((const void *)mxfp4_gemm_kernel<MXG_WAVES>, lds));
    hipLaunchKernelGGL((mxfp4_gemm_kernel<MXG_WAVES>), grid, dim3(MXG_WAVES * 64), lds, s, (const uint16_t *)p.x, (const unsigned char *)p.blocks,
                       (const unsigned char *)p.scales, (const uint16_t *)p.bias, (uint16_t *)p.y, p.expert_offsets, p.token_ids,
                       (int)p.K, (int)p.N, NC, NG, (int)p.n_experts, x_bytes, p.swiglu, p.swiglu_limit);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

// p.blocks / p.scales hold the resident copy; grouped form only; p.M = rows of x
int launch_mxfp4_res_gemm(oxq_ctx *ctx, hipStream_t s, const Mxfp4Problem &p) {
    const int rows = mxfp4_gemm_form(ctx, p.n_pairs, p.n_experts, p.K, p.N);
    if (rows == 0) return fail(OXQ_ERR_UNSUPPORTED, "mxfp4 experts prefill: shape not taken");
    const int nb = (int)(p.K / 32), NC = (int)ceil_div(nb, 4), NG = (int)ceil_div(NC, 4);
    // sum over experts of ceil(pairs_e / rows) <= pairs / rows + experts
    const int64_t ytiles = p.n_pairs / rows + p.n_experts;
    if (ytiles > 65535) return fail(OXQ_ERR_UNSUPPORTED, "mxfp4 experts prefill: %lld row tiles exceed the grid limit of 65535", (long long)ytiles);
    // The 16-row tiles have workgroups of 512 columns that start with less to do: at up to a dozen pairs an expert they are
    // the faster ones where K is long and the wide kernel's workgroups of 256 columns do not fill two places a compute unit (32
    // experts x 2880 x 2880 at 24 / 48 / 96 tokens 32.2 / 34.1 / 34.6 against 34.6 / 36.4 / 36.7 us; 5760 x 2880, which fills
    // them, 60.5 / 63.6 / 63.6 against 57.6 / 60.6 / 61.6; 64 experts x 1024 x 1024 at 64 tokens 16.8 against 9.4).
    const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    // (up to 96 pairs an expert, few of which then hold more than one tile of rows)
    const bool wide12 = !tune_given(ctx, OXQ_TUNE_MXFP4_GEMM_ROWS) && p.n_pairs <= 96 * p.n_experts &&
                        ceil_div(p.N, 32 * MXG_WAVES12) * p.n_experts <= cus && ceil_div(p.N, 32 * MXG_WAVES) * p.n_experts > cus;
    const bool narrow = !wide12 && rows == 16 && p.K >= 2048 && ceil_div(p.N, 32 * MXG_WAVES) * p.n_experts < 2 * cus;
    dim3 grid((unsigned)ceil_div(p.N / 16, (int64_t)4 * MXG_WAVES), (unsigned)ytiles, narrow ? 1 : 2);
    if (wide12) grid = dim3((unsigned)ceil_div(p.N, 32 * MXG_WAVES12), (unsigned)ytiles);
    char name[64];
    plan_name(name, sizeof name, "mxfp4_experts_gemm_bf16_r%dx%d%s", rows, wide12 ? MXG_WAVES12 : MXG_WAVES, p.swiglu ? "_swiglu" : "");
    set_plan(ctx, name, grid, dim3(wide12 ? 64 * MXG_WAVES12 : 512), 1, 1, 0);
    if (ctx->plan_only) return OXQ_OK;
    const uint64_t x_bytes = (uint64_t)p.M * (uint64_t)p.K * 2u;
    if (x_bytes >= (1ull << 31)) return fail(OXQ_ERR_UNSUPPORTED, "mxfp4 experts prefill: x of %llu bytes exceeds 2 GiB", (unsigned long long)x_bytes);
    if ((uintptr_t)p.x & 15) return fail(OXQ_ERR_UNSUPPORTED, "mxfp4 experts prefill: x must be 16-byte aligned");
    if ((uintptr_t)p.y & 3) return fail(OXQ_ERR_UNSUPPORTED, "mxfp4 experts prefill: out must be 4-byte aligned");
    if (wide12) return mxfp4_wide_go<MXG_WAVES12>(s, grid, p, NG, (uint32_t)x_bytes);
    return narrow ? mxfp4_gemm_go(s, grid, p, NC, NG, (uint32_t)x_bytes) : mxfp4_wide_go<MXG_WAVES>(s, grid, p, NG, (uint32_t)x_bytes);
}

}  // namespace oxq
