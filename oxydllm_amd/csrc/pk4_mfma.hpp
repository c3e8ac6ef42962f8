// pk4_mfma_kernel: the ring kernel of the resident 64-column layout (described in pk4.hip), for every row count and for
// quantization groups of 32, 64 and 128 or more rows.
#pragma once

#include "pk4_common.hpp"

namespace oxq {

// ---------------------------------------------------------------------------
// y[M, N] = x[M, K] . W   on the repacked layout
//
// grid.x = strip (64 output columns), grid.z = block of 16*MT rows of x,
// grid.y = K slice (1 unless the layer has few strips and a long K, see the
// launcher); the 8 waves deal the slice's blocks of 128 rows (4 MFMA steps) out
// round-robin, so that at any moment the workgroup reads one contiguous stretch of
// its strip (a plain read of the same bytes is 4 % faster that way than with one
// contiguous eighth per wave).  With more than one slice the workgroup writes its
// f32 partial tile to the workspace and a second launch adds the slices in order.
//
// Weights: one 1 KB wave load per step, issued one block (4 steps) ahead; the block's
// zero/scale pairs ride in the same ring (one 16-byte load per lane and block).
// Activations: the matrix-core fragment pattern (16 rows x 64 bytes per load)
// is served by L2 at a third of the rate of 256-byte row reads, so a wave
// fetches its next 16*MT x 128 block of x with 4-rows-x-256-bytes loads one
// block ahead, parks it in its private LDS slot (16-byte chunks XOR-swizzled by
// row, so both the row-wise write and the fragment read are conflict-free)
// and reads fragments from there.  Rows past M are never fetched (out-of-range
// lane offset: the buffer unit returns zero without touching memory).
// All vector loads are issued unconditionally - steps past the end of a
// wave's share also use the out-of-range offset - so the compiler can count
// exactly how many loads are younger than the one it waits for; a conditionally
// issued load makes it wait for all of them, which serialises the pipeline.
// The 8 partial 16*MT x 64 tiles meet in LDS (each wave's slot is its own
// activation slot) and are added in wave order, which fixes the summation order.
//
// Two arithmetic forms, both with f32 accumulation:
//  * GS = false (m > 16, the reference's tile-GEMM range): B = T((q - z) * s),
//    bit-identical to the dense dequant, fed to the matrix cores.
//  * GS = true (m <= 16, the reference's fused-GEMV range, which never rounds
//    the dequantized weight: quant_kernels.metal w4a16 GEMV keeps (q - z) * s in
//    f32): the matrix cores multiply x by the exact integers bias + q, one
//    extra MFMA against a fragment of ones yields the row sums of x in the
//    accumulator layout, and once per block
//        y += s * (acc_b - (bias + z) * rowsum_b(x))            (all f32).
// ---------------------------------------------------------------------------
// Ring depth: weights WD steps (1 KB wave loads).  One block of weights in flight per wave is
// the measured optimum (4096 x 14336, f16, M = 1 / 16): 2 steps equal, 8 steps 5 - 10 % slower,
// 16 steps 17 % slower.  A CU takes only so many vector loads in flight: what the first waves
// issue beyond their next block keeps the other waves' first loads waiting.
template <int MT, int BITS> struct Pk4Ring {
    static constexpr int WD = 4;
};

// XQ: activation loads per block and lane that can hold rows below M (4 rows each); the
// launcher passes 4 * MT, or fewer for a short single tile, whose other rows stay zero in LDS.
// NBLK > 0: every wave has exactly NBLK blocks and the block loop is straight-line code.
// SETS > 1: quantization groups of 64 (2) or 32 (4) rows, see pk4_fine.hip: the folded form folds a group at a time, the
// tile form takes a step's constants from its group's pairs, and K may end inside a block (weights and scales of the
// missing rows are zero in the copy; x is masked, so that a row's neighbour in memory cannot reach it).
template <typename TT, int BITS, int MT, bool GS, int WD, int XQ, bool PLZ = false, int NBLK = 0, int SETS = 1>
__global__ __launch_bounds__(512) void pk4_mfma_kernel(const uint16_t *__restrict__ x,
                                                       const uint32_t *__restrict__ pw,
                                                       const uint16_t *__restrict__ bias,
                                                       uint16_t *__restrict__ y, float *__restrict__ ws,
                                                       int M, int K, int N, int bslice, int contiguous, int act) {
    typedef MfmaOps<TT> Ops;
    constexpr int NW = 8;                      // waves per workgroup (4 and 16 waves measured 30 % slower)
    constexpr int ROWS = 16 * MT;
    constexpr int AQ = XQ;                     // activation loads per block and lane
    constexpr int SLOT = ROWS * 256;           // bytes of one wave's LDS slot (= its partial tile)
    constexpr int OOB = 0x7FFFFF00;
    constexpr int WL = BITS / 4;               // 1 KB weight loads per step
    constexpr int BB = pk4_block_words(BITS, SETS) * 4;  // bytes of one block: weights, then the zero/scale pairs
    // Up to 48 rows there is one row tile, so every weight is read once per launch: nontemporal
    // loads (cache policy bit 1), which a bare read of the same 30 MB also gains 7 % from.
    // From 49 rows on several row tiles may share a strip through L2, so those keep the default - except the
    // forms that are only launched with one row-tile workgroup a strip (NBLK, PLZ).  64 rows, same box, default ->
    // nontemporal: 4096 x 14336 f16 15.93 -> 15.45 us, bf16 17.48 -> 17.02; 5120 x 13824 f16 19.33 -> 18.54, 8-bit 24.14 ->
    // 22.60; 8192 x 28672 51.7 -> 50.8.  (4096 x 11008 measures 14.44 -> 14.60: its 12 rotated copies, 270 MB, are
    // partly still in the 256 MB memory-side cache when their turn comes again, which a decoder's layers are not.)
    constexpr int WNT = (MT < 4 || NBLK > 0 || PLZ) ? 2 : 0;
    // Hand-placed memory operations (the three places marked PLACED below) instead of the compiler's own order,
    // where that measured faster - same box, 48 / 64 / 128 rows: 8-bit f16 5120 x 13824 21.8 / 27.3 / 42.5 ->
    // 20.6 / 24.3 / 41.0 us; 4-bit bf16 4096 x 14336 at 33 / 48 rows 16.4 / 16.7 -> 15.2 / 15.9 us.  The 4-bit f16
    // kernels and bf16 at four row tiles are as fast or faster as the compiler orders them (f16 at 64 / 128
    // rows 16.9 / 29.4 against 16.6 / 30.8; bf16 19.6 / 33.8 against 18.7 / 34.3).
    // PLZ: the 4-bit kernel at four row tiles when a strip has one row-tile workgroup and the tile is (nearly)
    // full, 57 - 64 rows: placed it is 1.5 - 5 % faster there (same box, 64 rows: f16 16.48 -> 16.24, bf16 19.39 ->
    // 18.43, 5120 x 13824 f16 20.3 -> 19.9 us), slower at 49 rows (f16 15.33 -> 15.71) and when two or more
    // row-tile workgroups share a strip's weights through L2 (128 rows: f16 29.4 -> 30.8).
    constexpr bool PLACED = PLZ || (MT >= 3 && (BITS == 8 || (TT::DTYPE == BF16Traits::DTYPE && MT == 3)));
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int j = blockIdx.x;
    const int m0 = blockIdx.z * ROWS;
    const int NB = SETS > 1 ? (K + 127) >> 7 : K >> 7;
    // K slice of this workgroup: blocks [sb0, sb0 + SB).  The wave's blocks inside it, by local index
    // i: every 8th block starting at its own number (the default), or one contiguous run (a tuning
    // switch; the shares differ by at most one block either way).
    const int sb0 = blockIdx.y * bslice;
    const int SB = min(NB, sb0 + bslice) - sb0;
    const int cbase = SB / NW, crem = SB % NW;
    const int nloc = contiguous ? cbase + (wave < crem ? 1 : 0) : (SB > wave ? (SB - wave + NW - 1) / NW : 0);
    const int cb0 = sb0 + wave * cbase + min(wave, crem);
    auto blk_of = [&](int i) { return contiguous ? cb0 + i : sb0 + i * NW + wave; };
    unsigned char *slot = pk4_lds + wave * SLOT;

    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(pw + (size_t)j * NB * (BB / 4), (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, (uint32_t)M * (uint32_t)K * 2u);
    const int voff_w = lane * 16;
    // The block's zero/scale pairs: lane (ni, kb) fetches word kb of column quad ni (one 4-byte load a lane,
    // 256 contiguous bytes a wave: a quarter of what a 16-byte load costs the address unit, which is the
    // busiest unit from 32 rows on) and the four lane groups then exchange their words (pk4_pair_words).
    const int voff_z = 1024 * WL * 4 + (ni * 4 + kb) * 4;
    // activation load q of a block: row 4q + lane/16, 16-byte chunk lane%16 of the row's 256 bytes; rows
    // past M get an offset beyond any buffer, for which the buffer unit returns zeros without touching
    // memory (the scalar offset of a buffer load is not part of its bounds check, so the lane offset
    // has to carry the row)
    // Up to two row tiles every load keeps its own offset register; the larger kernels are at their
    // register budget and derives them from the first one (a row past M then lies beyond the end of x by
    // its lane offset alone, which the bounds check does cover).
    constexpr bool VA1 = MT >= 3;
    int voff_a[VA1 ? 1 : AQ];
#pragma unroll
    for (int q = 0; q < (VA1 ? 1 : AQ); ++q) {
        const int r = m0 + 4 * q + kb;
        voff_a[q] = r < M ? (r * K * 2 + ni * 16) : OOB;
    }
    uint32_t rowstep = 4u * (uint32_t)K * 2u;
    // LDS position of (row = 4q + kb, chunk ni): chunk index XORed with row % 16 = kb | (q % 4) << 2
    int a_wr[4];
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) a_wr[qq] = kb * 256 + (((ni ^ kb) ^ (qq << 2)) << 4);  // + 1024 q
    // fragment read of step s (0..3), row tile mt: row 16mt + ni, chunk 8*(s/2) + 2kb + (s%2)
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + ((pk4_x_chunk<SETS>(st, kb) ^ ni) << 4);
    const NibbleMasks nm = nibble_masks();
    // rows no load covers: zero once, no block writes them again
#pragma unroll
    for (int q = AQ; q < 4 * MT; ++q) {
        const int row = 4 * q + kb;
        *(u32x4_t *)(slot + row * 256 + ((ni ^ (row & 15)) << 4)) = u32x4_t{0u, 0u, 0u, 0u};
    }

    static_assert(WD == 4, "the ring holds exactly one block");
    u32x4_t aring[AQ], wring[WD][WL];
    uint32_t zring[SETS];
    constexpr int SPS = 4 / SETS;  // steps that share a set of pairs
    // Past the end of the wave's share the loads go through an empty descriptor: a scalar select,
    // no vector instruction, and the buffer unit returns zero without touching memory.
    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    auto load_a = [&](int i, u32x4_t (&a)[AQ]) {
        const __amdgpu_buffer_rsrc_t rs = i < nloc ? rs_x : rs_none;  // wave-uniform
        const int blk = blk_of(i);
        const bool past_k = SETS > 1 && blk * 128 + 8 * ni >= K;
#pragma unroll
        for (int q = 0; q < AQ; ++q) {
            if constexpr (SETS > 1) {
                const uint32_t at = VA1 ? (uint32_t)voff_a[0] + (uint32_t)q * rowstep : (uint32_t)voff_a[VA1 ? 0 : q];
                a[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, past_k ? OOB : (int)at, blk * 256, 0);
            } else if (VA1) {
                if (q == 0) asm volatile("" : "+s"(rowstep));  // recomputed per block: 15 registers less to hold
                // no wrap-around: 15 row steps stay below 2^31 (K <= 2^24, checked on the host), so a row
                // past M - from the first offset or by the steps - lies beyond x (< 2 GiB) and reads zeros
                a[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)((uint32_t)voff_a[0] + (uint32_t)q * rowstep), blk * 256, 0);
            } else {
                a[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_a[q], blk * 256, 0);
            }
        }
    };
    auto load_w = [&](int i, int st, u32x4_t (&w)[WL]) {
        const __amdgpu_buffer_rsrc_t rs = i < nloc ? rs_w : rs_none;
#pragma unroll
        for (int h = 0; h < WL; ++h)
            w[h] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_w, blk_of(i) * BB + (st * WL + h) * 1024, WNT);
    };
    auto load_z = [&](int i, int set) {
        const __amdgpu_buffer_rsrc_t rs = i < nloc ? rs_w : rs_none;
        zring[set] = __builtin_amdgcn_raw_buffer_load_b32(rs, voff_z, blk_of(i) * BB + set * 256, WNT);
    };
    auto store_a = [&](const u32x4_t (&a)[AQ]) {
#pragma unroll
        for (int q = 0; q < AQ; ++q) *(u32x4_t *)(slot + q * 1024 + a_wr[q & 3]) = a[q];
    };

    // issue order = consumption order.  The tile form needs the pairs before its first B fragment,
    // the folded form after the block's last step.
    u32x4_t afirst[AQ];
    load_a(0, afirst);
    if (!GS) {
#pragma unroll
        for (int u = 0; u < SETS; ++u) load_z(0, u);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) load_w(0, g, wring[g]);
    if (GS) {
#pragma unroll
        for (int u = 0; u < SETS; ++u) load_z(0, u);
    }
    load_a(1, aring);

    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    constexpr bool WIDEN = !GS && BITS == 4 && TT::DTYPE == BF16Traits::DTYPE;
    uint32_t negzb[4], sp[4];          // GS = false: the two Pk4T constants per column
    Pk4gBf16 cb[4];                    // the same of a 4-bit bf16 layer
    const uint32_t ones[4] = {TT::ONES, TT::ONES, TT::ONES, TT::ONES};
    const float4_t zero4 = float4_t{0.f, 0.f, 0.f, 0.f};

    store_a(afirst);

    // PLACED (1).  The counter a wave waits on counts its loads in issue order, and what the loop waits for at
    // its top is the stricter of what its two entries require.  From three row tiles on the compiler requests
    // the second x block before the first pairs and weights here, but after them inside the loop: coming from
    // here the pairs have 4 younger loads, so the loop would wait with "at most 4 outstanding" - that is, for
    // 12 of the 16 x loads it has just issued - in every iteration.  With block 0's pairs and weights
    // complete before the loop, only the loop's own order counts.
    if constexpr (PLACED) {
        asm volatile("" ::"v"(zring[0]));
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int h = 0; h < WL; ++h) asm volatile("" ::"v"(wring[g][h]));
    }
    // Two blocks an iteration where placed by hand: the ring registers a block loads are copied to the ones
    // the loop carries at the loop's end, which waits for those loads; twice as rarely this way.
    // With the block count known (NBLK) there is no loop at all (figures where it is launched).
    constexpr int UF = NBLK > 0 ? 1 : PLACED ? 2 : 1;
    const int trip = NBLK > 0 ? NBLK : nloc;
    constexpr int UNROLL = NBLK > 0 ? NBLK : 1;
#pragma unroll UNROLL
    for (int i0 = 0; i0 < trip; i0 += UF)
#pragma unroll
    for (int u = 0; u < UF; ++u) {
        const int i = i0 + u;
        if (u > 0 && i >= nloc) break;
        // Straight-line code knows its last block, behind which nothing is requested: a load from the empty descriptor takes its turn
        // in the address unit as any other, and what follows waits for the registers it writes.
        const bool last = NBLK > 0 && i + 1 >= NBLK;
        float4_t tmp[GS ? MT : 1][4], tmps[GS ? MT : 1];  // per-block integer sums of the GS form
        // the tile form's constants of a set, and the request for the next block's
        auto constants = [&](int set) {
            uint32_t zv[4];
            pk4_pair_words(zring[set], zv);
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                if constexpr (WIDEN) cb[f].set(__builtin_bit_cast(float, zv[f] & 0xFFFF0000u), __builtin_bit_cast(float, zv[f] << 16) + 128.0f);
                else Pk4T<TT>::prep(zv[f], negzb[f], sp[f]);
            }
            if (!last) load_z(i + 1, set);
        };
        // the folded form: y += s * (sum - (bias + z) * rowsum), all f32
        auto fold = [&](int set) {
            uint32_t zv[4];
            pk4_pair_words(zring[set], zv);
            if (!last) load_z(i + 1, set);
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const float sf = TT::to_f32((uint16_t)(zv[f] >> 16));
                const float nszb = sf * TT::to_f32((uint16_t)(zv[f] & 0xFFFFu));  // -s * (bias_f + z)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[mt][f][e] = fmaf(sf, tmp[mt][f][e], fmaf(nszb, tmps[mt][e], acc[mt][f][e]));
            }
        };
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (!GS && st % SPS == 0) constants(st / SPS);
            u32x4_t wv[WL];
#pragma unroll
            for (int h = 0; h < WL; ++h) wv[h] = wring[st][h];
            uint32_t wp[WL][4];
#pragma unroll
            for (int h = 0; h < WL; ++h) {
                const uint32_t w0 = wv[h][0], w1 = wv[h][1], w2 = wv[h][2], w3 = wv[h][3];
                wp[h][0] = w0, wp[h][1] = w1, wp[h][2] = w2, wp[h][3] = w3;
            }
            // row pair pp of column f as two exact 16-bit floats bias + q
            auto pair = [&](int pp, int f) -> uint32_t {
                if (BITS == 4) return TT::unpack1(wp[0][pp], f, nm);
                const uint32_t word = wp[(f >> 1) % WL][pp];
                return TT::unpack_bytes((f & 1) ? (word >> 8) : word);
            };
            uint32_t a[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4_t av = *(const u32x4_t *)(slot + mt * 4096 + a_rd[st]);
                const uint32_t a0 = av[0], a1 = av[1], a2 = av[2], a3 = av[3];
                a[mt][0] = a0, a[mt][1] = a1, a[mt][2] = a2, a[mt][3] = a3;
            }
            if (GS) {
                const bool fresh = st % SPS == 0;  // a group's sums start from zero: no clearing
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    uint32_t b[4];
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) b[pp] = pair(pp, f);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        tmp[mt][f] = Ops::mfma(a[mt], b, fresh ? zero4 : tmp[mt][f]);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) tmps[mt] = Ops::mfma(a[mt], ones, fresh ? zero4 : tmps[mt]);
            } else if constexpr (WIDEN) {
                uint32_t b0[4], b2[4];
                auto column = [&](int f, const uint32_t (&b)[4]) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
                };
                pk4g_columns<0>(wp[0], cb[0], cb[2], b0, b2);
                column(0, b0), column(2, b2);
                pk4g_columns<1>(wp[0], cb[1], cb[3], b0, b2);
                column(1, b0), column(3, b2);
            } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    uint32_t b[4];
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) b[pp] = Pk4T<TT>::deq(pair(pp, f), negzb[f], sp[f]);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
                }
            }
            // PLACED (2).  Vector-memory requests, LDS writes and MFMAs stay inside their step (vector and
            // scalar arithmetic and LDS reads may move across): the ring refill above is then issued a block
            // ahead of its use, as written, instead of at the block's end with the other three.
            // Refill this ring slot after its last use, so that the new block can land in the same registers
            // (requested while the old value is live it lands in others, copied at the loop's end behind a wait
            // for the request): 17 / 33 / 48 rows f16 9.96 / 12.76 / 13.57 -> 9.85 / 12.57 / 13.44 us.
            if (!last) load_w(i + 1, st, wring[st]);
            if constexpr (PLACED) __builtin_amdgcn_sched_barrier(0x106);
            if (GS && (st + 1) % SPS == 0) fold(st / SPS);
        }
        // the next block's activations replace this one's (same wave: LDS accesses stay in order)
        // PLACED (3).  The x block stays in its registers until here: hoisted to the block's start (with all 16
        // fragments of the current block held in registers instead), its reload comes late in the block and
        // is waited for at the next block's start.
        if constexpr (PLACED) __builtin_amdgcn_sched_barrier(0);
        if (!last) {
            store_a(aring);
            if (NBLK == 0 || i + 2 < NBLK) load_a(i + 2, aring);
        }
        // two and four row tiles as straight-line code: the requests for the block after next stay at the block's
        // end (four tiles at 64 rows, same box: f16 16.54 -> 16.37 us, bf16 18.42 -> 17.90; three tiles the same
        // either way)
        if constexpr (NBLK > 0 && (MT == 2 || MT == 4)) __builtin_amdgcn_sched_barrier(0);
    }

    pk4_epilogue<TT, MT>(acc, bias, y, ws, M, N, j, m0, act, wave, lane);
}

// one instantiation: its LDS grant, the launch, the error check
template <typename TT, int BITS, int MT, bool GS, int WD, int XQ, bool PLZ = false, int NBLK = 0, int SETS = 1>
static int pk4_mfma_go(oxq_ctx *ctx, hipStream_t s, dim3 grid, const Pk4Problem &p, int bslice) {
    const size_t lds = (size_t)8 * MT * 4096;
    static LdsGrant lds_grant;
    OXQ_HIP_CHECK(lds_grant.ensure((const void *)pk4_mfma_kernel<TT, BITS, MT, GS, WD, XQ, PLZ, NBLK, SETS>, lds));
    hipLaunchKernelGGL((pk4_mfma_kernel<TT, BITS, MT, GS, WD, XQ, PLZ, NBLK, SETS>), grid, dim3(512), lds, s,
                       (const uint16_t *)p.x, p.w.pw, (const uint16_t *)p.bias, (uint16_t *)p.y, (float *)ctx->workspace,
                       (int)p.M, (int)p.w.K, (int)p.w.N, bslice, tune(ctx, OXQ_TUNE_PK4_CONTIGUOUS, 1), p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

}  // namespace oxq
