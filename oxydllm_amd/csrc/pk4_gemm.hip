// Resident layers at prefill sizes (linear.rs:494-509: m >= 64 takes the staged tile GEMM,
// mpp_gemm.metal:101-266): the tile arithmetic of pk4_mfma_kernel - B = T((q - z) * s) rounded once to the
// activation type, f32 accumulate - in a decomposition for many rows.
//
// pk4_mfma_kernel gives a workgroup one strip of 64 columns and 64 rows of x, and its 8 waves split K: every
// (row tile, strip) pair reads its 64 rows of x again, each wave for itself through the vector-memory unit.
// At 2048 rows of a 4096 x 14336 layer that is 7168 workgroups x 512 KB = 3.7 GB of activations out of L2 for
// 16.8 MB of x, and the kernel runs at the speed it has at 64 rows (0.6 PFLOP/s).  Here a workgroup takes 64
// rows and EIGHT strips: its waves share one copy of the rows in LDS (a block of 128 elements of K at a time,
// loaded from global memory straight into LDS - no registers, nothing for the compiler to sink behind the
// arithmetic - two buffers, one barrier a block), each wave owns a strip, streams its blocks with the
// one-block ring of pk4_mfma_kernel and keeps the whole K in its own accumulators - no partial tiles, no
// second launch.  x out of L2 falls to an eighth.  Workgroups are numbered so that 64 neighbours form a square
// of 8 row tiles x 8 strip groups, whose rows of x and weights the neighbours find in L2.
#include "oxq_device.hpp"
#include "oxq_internal.hpp"
#include "oxq_mfma.hpp"
#include "pk4_common.hpp"
#include "pk4_gemm.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace oxq {

// The same decomposition on a layer stored in 16-column strips (the narrow layout of attention and down
// projections): a wave's 64 columns are four neighbouring strips, a strip's block is one 16-byte load a lane
// whose words are the block's four steps - so the ring holds whole blocks, two of them: the next block is
// requested into the other half when a block starts.  Lane (ni, kb) holds column 16 f + ni of strip f.
template <typename TT, int MT>
__global__ __launch_bounds__(512) void pk4n_gemm_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ pw,
                                                        const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                        int M, int K, int N, int NG, int RT) {
    typedef MfmaOps<TT> Ops;
    constexpr int ROWS = 16 * MT, BB = PK4N_BW * 4, XBUF = ROWS * 256, XV = ROWS / 4 / PK4G_STRIPS;
    constexpr bool BF = TT::DTYPE == BF16Traits::DTYPE;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    int rt, g;
    if ((int)blockIdx.x >= RT * NG) return;  // the whole workgroup, before any barrier
    pk4g_tile_of((int)blockIdx.x, RT, NG, rt, g);
    const int j = g * PK4G_STRIPS + wave;  // the wave's 64 columns: strips 4 j .. 4 j + 3
    const bool live = j < (N >> 6);
    const int m0 = rt * ROWS;
    const int NB = K >> 7;
    const int xrows = min(M - m0, ROWS);

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl =
        make_rsrc(pw + (size_t)(live ? 4 * j : 0) * NB * PK4N_BW, 4u * (uint32_t)NB * (uint32_t)BB);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const int voff_w = lane * 16, voff_z = 1024 + ni * 4;
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (wave * XV + q) + (lane >> 4);
        xo[q] = r * K * 2 + (((lane & 15) ^ (r & 15)) << 4);
    }
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + (((8 * (st >> 1) + 2 * kb + (st & 1)) ^ ni) << 4);
    const NibbleMasks nm = nibble_masks();

    u32x4_t wring[2][4];
    uint32_t zring[4];
    auto dma_x = [&](int i) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_x : rs_none;
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (i & 1) * XBUF + (wave * XV + q) * 1024, xo[q], i * 256);
    };
    auto load_w = [&](int i, u32x4_t (&w)[4]) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
#pragma unroll
        for (int f = 0; f < 4; ++f) w[f] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_w, (f * NB + i) * BB, 0);
    };
    auto load_z = [&](int i) {
        const __amdgpu_buffer_rsrc_t rs = i < NB ? rs_w : rs_none;
#pragma unroll
        for (int f = 0; f < 4; ++f) zring[f] = __builtin_amdgcn_raw_buffer_load_b32(rs, voff_z, (f * NB + i) * BB, 0);
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
    load_z(0);
    load_w(0, wring[0]);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    pk4g_wait_vmcnt<8>();
    __syncthreads();

    // one block, its weights in ring half CUR; eight ring loads are younger than the block's loads of x
    auto block = [&](int i, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        dma_x(i + 1);
        __builtin_amdgcn_sched_barrier(0);
        load_w(i + 1, wring[CUR ^ 1]);
        __builtin_amdgcn_sched_barrier(0);  // not sunk to the block's end, where the next block would wait for them
        const unsigned char *buf = pk4_lds + (i & 1) * XBUF;
        Pk4N<TT> cst[4];
        Pk4gBf16 cb[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if constexpr (BF) {  // the pair word holds {-z, s}
                cb[f].set(__builtin_bit_cast(float, zring[f] & 0xFFFF0000u), __builtin_bit_cast(float, zring[f] << 16));
            } else {
                cst[f].prep(zring[f]);
            }
        }
        load_z(i + 1);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            uint32_t a[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4_t av = *(const u32x4_t *)(buf + mt * 4096 + a_rd[st]);
                a[mt][0] = av[0], a[mt][1] = av[1], a[mt][2] = av[2], a[mt][3] = av[3];
            }
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const uint32_t w = wring[CUR][f][st];
                uint32_t b[4];
                if constexpr (BF) {  // row pair pp: nibble pp of each 16-bit half
                    cb[f].rows(w, b);
                } else {
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) b[pp] = cst[f].deq(TT::unpack1(w, pp, nm), pp);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        pk4g_wait_vmcnt<8>();  // this wave's part of the next block of x is in LDS
        __syncthreads();
    };
    {
        int i = 0;
        for (; i + 1 < NB; i += 2) {
            block(i, std::integral_constant<int, 0>{});
            block(i + 1, std::integral_constant<int, 1>{});
        }
        if (i < NB) block(i, std::integral_constant<int, 0>{});
    }

    if (!live) return;
    // row 16 mt + 4 kb + e, column 64 j + 16 f + ni
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
        for (int f = 0; f < 4; ++f) bv[f] = TT::to_f32(bias[64 * j + 16 * f + ni]);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + 16 * t + 4 * kb + e;
            if (row >= M) continue;
#pragma unroll
            for (int f = 0; f < 4; ++f) y[(size_t)row * N + 64 * j + 16 * f + ni] = TT::from_f32(acc[t][f][e] + bv[f]);
        }
}

// Which decomposition a resident layer runs at M rows: 0 = the split-K tiles of pk4_mfma_kernel /
// pk4n_mfma_kernel, else the rows of a workgroup here.  Costs are in units of a full round (one 64-row workgroup
// on every CU), fitted to sweeps over 128..8192 rows in both types (64-column strips: 4096 x 14336, 8192 x 28672;
// 16-column strips: 4096 x 4096, 4096 x 6144, 14336 x 4096, 8192 x 8192; 8-bit: 4096 x 14336, 5120 x 13824):
//   - 128-row workgroups (203..230 registers: one a CU) run in whole rounds; a round costs `full128`, a last
//     round that fills at most 0.7 of the CUs `part128`;
//   - 64-row workgroups of the 64-column layout (121..125 registers) share a CU in pairs: up to one a CU the launch
//     costs 1 (`part64` up to three quarters of the CUs), up to two a CU a64 + b64 w, beyond that slope64 w
//     (w = workgroups / CUs); those of the 16-column layout (144..145 registers) run in whole rounds;
//   - the last rows behind whole tiles of 128, if at most 32, can be tiles of 32 of the same launch (64-column strips, groups of 128
//     and more), on the CUs that the whole tiles leave idle: a padded tile of 128 costs four times its rows' arithmetic and
//     often one more round.  Us, 64- or 128-row tiles alone -> with them: 4-bit bf16 3584 x 18944 at 777 rows 127 -> 103,
//     gate|up 4096 x 28672 at 520 rows 155 -> 122, 4096 x 11008 at 1300, 4100 rows 192 -> 156, 397 -> 362; 8-bit f16
//     4096 x 14336 at 1160 rows 204 -> 170;
//   - the split-K tiles cost `split_lo` (below one round) or `split_hi` times w at any M: small workgroups, no
//     ragged round, but the rate they have at 64 rows.
// The bf16 conversion and the two-strip form are newer than these fits, and groups of 32 and 64 rows are in none.  With every
// form forced at 14 row counts from 65 to 4096 (4- and 8-bit layers of 3584 x 18944, 4096 x 6144, 4096 x 11008, 4096 x 14336,
// 5120 x 6144) the choice is within 8 % of the fastest, except where a launch holds one to one and a half rounds: 8-bit
// 4096 x 6144 at 150 rows split-K 32 us, two strips 23; groups of 64, 4096 x 11008 at 150 rows 46 and 40; groups of 32,
// 5120 x 6144 at 150 / 777 / 900 / 1200 rows f16 33 / 96 / 96 / 143 as chosen, 26 / 81 / 84 / 108 with two strips.
// The fits are older than the numbering without gaps too.  Where the strip groups are no multiple of eight (32 layers of 64-column
// strips with 1 - 21 groups, K 1280 - 10240, both types and widths, 160 calls of 256 - 4000 rows, every form forced) the choice is
// within 3 % of the fastest at 129, within 8 % at 152, 15 % at all.
// OXQ_PK4_GEMM_ROWS = 64 | 128 | 32 (128 and the last tile of 32) takes the choice (tests, sweeps); OXQ_PK4_GEMM_MIN_M = 0 switches the kernels off.
// a round of the two-strip form (one workgroup a CU) against a full round of 64-row workgroups of eight strips:
// 19 - 24 us against 65 - 78 at K = 4096 over both widths and types
constexpr double PK4_MID_ROUND = 0.31;
// 16-column strips: the same for a whole round, 0.27 for a last round on at most half of the CUs (4096 x 4096,
// 4096 x 6144, 8192 x 8192, 14336 x 4096 over 65..2048 rows in both types: 18.7 - 24.4 us a round at K = 4096)
constexpr double PK4N_MID_ROUND = 0.31, PK4N_MID_PART = 0.27;
// pk4_mid128_kernel, 128 rows and two strips, one workgroup a CU: a round (f16: a last round on at most 0.7 of the CUs) in the
// same units.  bf16 takes 31 - 33 us a round at K = 4096 where one of 64 rows takes 22 - 25, f16 28 - 32 against 19 - 20.  Us, best
// of the other forms -> this: bf16 4096 x 28672 at 65 / 128 / 256 rows 45 / 45 / 75 -> 33 / 34 / 66, 4096 x 14336 at 256 / 512 rows
// 42 / 72 -> 33 / 65, 3584 x 18944 at 128 / 384 rows 38 / 65 -> 29 / 60; f16 4096 x 28672 at 128 rows 43 -> 34, 4096 x 11008 at 256
// 39 -> 32.  At 4096 x 28672 and 512 rows 128-row workgroups of eight strips are ahead (bf16 107 against 132).
// Beyond one round it counts 11 % more in bf16, and 7 % where K is long (from 3968 in up to two rounds, groups of 64 in any; groups of
// 32 at any K).  Us, the form of eight strips -> this at 118 calls of other layers that lie between the two figures: groups of 128 in up to two rounds
// 4096 x 14336 at 448 / 512 rows 70 / 74 -> 65 / 67, 3968 x 20992 at 286 69 -> 68, 4480 x 14464 at 461 79 -> 76, but 3840 x 7424 at 953
// 67 / 71, 3328 x 10048 at 630 59 / 61; in three 7936 x 13888 at 856 181 / 195, 7040 x 11328 at 994 162 / 168; groups of 64 3968 x 16320 at 492
// 75 -> 71, 8960 x 9920 at 1059 231 -> 209, but 3200 x 15936 at 489 63 / 68; groups of 32 3456 x 14272 at 477 71 -> 65, 7808 x 17088 at
// 1137 397 -> 335.  Against three rounds of 64 rows 9344 x 18048 at 236 rows takes 132 against 128, 5120 x 8576 at 487 77 against 75.  Against
// the forms of eight strips, which add no partial tiles, a short K tells: 1024 x 12544 at 583 rows bf16 28.2 against 25.2, 1152 x 6272 at
// 994 rows f16 30.9 against 23.0.  (f16: figures 7 % lower, what its kernel has gained since they were fitted, choose no better: 2.1 % behind the
// fastest form together over ten layers, 80 calls, 1.9 % with these.)
// Groups of 64 and 32 go by the same figures (115 layers, 345 calls at 65 - 2200 rows: 65 came here, 1.27 times as fast, the
// least 1.05; 4096 x 15488, groups of 64, bf16 at 448 rows 80 -> 72, 8960 x 14720, groups of 32, at 243 100 -> 78).
// 16-column strips: a round, and a last one on at most 0.8 of the CUs.  bf16 at K = 4096 takes 31 - 32 and 36 us, f16 30 - 31 and 36; us,
// best of the other forms -> this: bf16 4096 x 4096 at 768 / 1024 rows 43 / 43 -> 32 / 36, 4096 x 6144 at 384 / 512 42 / 42 -> 32 /
// 32, 14336 x 4096 at 768 / 1024 124 / 132 -> 94 / 109, 8192 x 8192 at 384 / 512 75 / 78 -> 56 / 65; f16 4096 x 4096 at 768 rows
// 38 -> 31; 4096 x 6144 at 1024 rows, one and a half rounds, bf16 64 / 65.  Two rounds and more are behind the
// forms of eight strips (5760 x 4480 at 1639 rows bf16 104 / 95, 8320 x 6336 at 1913 203 / 187, 5632 x 7552 at 1488 f16 135 / 122).
struct Pk4Mid128Cost {
    double full, part, part_upto, more_from, more;  // times `more` beyond `more_from` rounds
};
constexpr Pk4Mid128Cost PK4_MID128_BF16 = {0.455, 0.455, 0.7, 1.0, 1.11}, PK4_MID128_F16 = {0.505, 0.45, 0.7, 1.0, 1.04};
constexpr Pk4Mid128Cost PK4N_MID128_BF16 = {0.52, 0.465, 0.8, 1.0, 1.08}, PK4N_MID128_F16 = {0.57, 0.50, 0.8, 1.0, 1.04};
constexpr double PK4_MID128_LONG_K = 0.92, PK4_MID128_OVER_K = 314.0;
constexpr double PK4_MID128_BF16_MORE_LONG_K = 1.07;  // 64-column strips

struct Pk4GemmCost {
    bool pairs64;
    double part64, a64, b64, slope64, full128, part128, split_lo, split_hi;
};
// rows of a workgroup (0: the split-K tiles) and the K split inside it (4: pk4_mid_kernel, two strips a workgroup)
struct Pk4GemmForm {
    int rows, ks;  // (128 rows and 4: pk4_mid128_kernel)
    bool light = false;  // 128 rows, and those behind the whole tiles in tiles of 32
};
// pk4_mid_kernel at up to 64 rows of 64-column strips, against the one-strip workgroups of pk4_mfma_kernel and
// pk4_tile64_kernel, both one a CU: a round of it costs 1.6 - 1.8 of theirs (4096 x 28672 at 48 / 64 rows: bf16 28.5 / 31.3 ->
// 25.2 / 26.3 us, f16 at 64 rows 29.3 -> 25.5; 8-bit 4096 x 22016 at 64 rows 39.2 -> 30.4; bf16 at 32 rows 23.0 -> 24.3).
// f16 only from where its weights are rounded anyway (pk4_folds).
static bool pk4_mid_decode(double cus, const Pk4Problem &p) {
    const int64_t from = p.w.dtype == OXQ_F16 ? 49 : 33;
    if (p.w.strip != 64 || p.M < from || p.M > 64 || pk4_sets(p.w.group_shift) > 1) return false;
    const double strips = (double)ceil_div(p.w.N, (int64_t)64);
    return 1.8 * std::ceil(strips / (2 * cus)) < std::ceil(strips / cus);
}
// Unrounded layers: the folded prefill form (one workgroup a CU, whole rounds) against row tiles of 32 of pk4_mfma_kernel, whose
// time goes with their number.  A round costs as much as `unit` tiles on every CU, fitted to 4096 x 11008, 11008 x 4096,
// 4096 x 4096, 2048 x 28672 and 4096 x 11000 at 33 - 2048 rows in both types (us, row tiles / prefill form, f16 except the
// last): GPTQ 4-bit groups of 64 4096 x 11008 at 256 / 512 / 2048 rows 67.9 / 86.3, 128.6 / 88.7, 493 / 265; groups of 32
// 4096 x 4096 at 1024 / 2048 rows 100 / 116, 195 / 124; AWQ 8-bit groups of 64 11008 x 4096 at 512 / 1024 rows 131 / 235,
// 267 / 235 (bf16).
// Between them pk4_midfold_kernel, whole rounds too: a round costs as much as `mid` rounds of tiles (both counted in whole rounds),
// one of the prefill form then `wide` (the tiles of 8-bit layers are faster in full rounds than the fit above has them).  Us at
// K = 4096, best of the other two -> this: GPTQ 4-bit groups of 64 N = 4096 at 512 / 1024 rows f16 43 / 85 -> 27 / 50, bf16 44 / 83 -> 29 /
// 54, N = 11008 at 128 / 256 / 512 f16 33 / 65 / 87 -> 26 / 48 / 74; groups of 32 N = 4096 at 512 rows f16 55 -> 32; 8-bit groups of 64
// N = 4096 at 512 rows f16 51 -> 29, N = 11008 at 256 bf16 91 -> 63; at 256 rows of N = 4096, two rounds of tiles, f16 21 / 25.  Against the
// prefill form, which adds no partial tiles, a short K tells (GPTQ 4-bit groups of 128 2048 x 7352 at 515 rows f16 35 / 38).  60 layers of
// 1024 - 10240 x 600 - 24000, 180 calls at 33 - 2200 rows: 63 came here, 1.31 times as fast.
static Pk4GemmForm pk4_fold_form(double cus, const Pk4Problem &p, bool mid) {
    static const double unit4[3] = {6.3, 8.0, 9.0}, unit8[3] = {4.8, 5.7, 6.9};  // groups of 128 rows and more, 64, 32
    static const double mid4[2][3] = {{2.08, 2.33, 2.2}, {2.35, 2.55, 2.7}}, wide4[3] = {6.3, 8.0, 8.5};  // f16, bf16
    static const double mid8[2][3] = {{2.1, 2.13, 2.1}, {2.35, 2.34, 2.35}}, wide8[3] = {5.4, 6.5, 7.3};
    const int sets = pk4_sets(p.w.group_shift), i = sets == 1 ? 0 : sets == 2 ? 1 : 2, b = p.w.dtype == OXQ_F16 ? 0 : 1;
    // the row tiles address the whole of x with 32 bits and are one grid dimension
    if ((uint64_t)p.M * (uint64_t)p.w.K * 2 >= (1ull << 31) || ceil_div(p.M, (int64_t)32) > 65535) return {64, 1};
    const int64_t strips = ceil_div(p.w.N, (int64_t)64), row_tiles = ceil_div(p.M, (int64_t)64);
    const double rounds = std::ceil((double)(ceil_div(strips, (int64_t)PK4G_STRIPS) * row_tiles) / cus);
    const double tiles = (double)(strips * ceil_div(p.M, (int64_t)32)) / cus;
    const double c_mid = std::ceil((double)(ceil_div(strips, (int64_t)2) * row_tiles) / cus) * (p.w.bits == 4 ? mid4 : mid8)[b][i];
    const double short_k = 0.88 + 500.0 / (double)p.w.K;
    if (mid && c_mid < std::ceil(tiles) && c_mid * short_k < rounds * (p.w.bits == 4 ? wide4 : wide8)[i]) return {64, 4};
    return {rounds * (p.w.bits == 4 ? unit4 : unit8)[i] < tiles ? 64 : 0, 1};
}
static Pk4GemmForm pk4_gemm_form(const oxq_ctx *ctx, const Pk4Problem &p) {
    const double cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    const int64_t min_m = tune(ctx, OXQ_TUNE_PK4_GEMM_MIN_M, pk4_sets(p.w.group_shift) > 1 ? 49 : pk4_mid_decode(cus, p) ? 33 : 65);
    if (min_m <= 0 || (p.w.bits != 4 && p.w.bits != 8) || (p.act && p.w.strip == 16) || p.M < min_m) return {0, 1};
    if ((uintptr_t)p.bias & 7) return {0, 1};  // (fused gate|up layers only: oxq_api.cpp, prepack_layer)
    if (p.w.bits == 8 && p.w.strip == 16) return {0, 1};  // (16-column strips are a 4-bit layout)
    const int forced = tune(ctx, OXQ_TUNE_PK4_GEMM_ROWS, 0), forced_ks = tune(ctx, OXQ_TUNE_PK4_GEMM_KS, 0);
    if (p.w.unrounded) {
        if (forced_ks == 4) return {64, 4};
        return forced ? Pk4GemmForm{64, 1} : pk4_fold_form(cus, p, forced_ks != 1);
    }
    const bool can_mid128 = p.w.bits == 4;
    if (forced_ks == 4) return {forced == 128 && can_mid128 ? 128 : 64, 4};
    const int64_t rest = p.M % 128;
    const bool can_light = p.M > 128 && rest >= 1 && rest <= 32 && p.w.strip != 16 && pk4_sets(p.w.group_shift) == 1;
    if (forced == 32 && can_light) return {128, 1, true};
    if (forced == 64 || forced == 128) return {forced, 1};
    if (p.M <= 64 && pk4_mid_decode(cus, p) && forced_ks != 1) return {64, 4};
    static const Pk4GemmCost WIDE_F16 = {true, 0.88, 1.20, 0.30, 0.97, 1.50, 1.27, 1.93, 1.50};
    static const Pk4GemmCost WIDE_BF16 = {true, 0.93, 1.29, 0.27, 0.98, 1.44, 1.35, 2.00, 1.53};
    static const Pk4GemmCost NARROW_F16 = {false, 0.86, 0, 0, 0, 1.64, 1.30, 1.60, 1.50};
    static const Pk4GemmCost NARROW_BF16 = {false, 0.94, 0, 0, 0, 1.51, 1.35, 1.60, 1.50};
    static const Pk4GemmCost WIDE8_F16 = {false, 0.88, 0, 0, 0, 1.47, 1.27, 1.92, 1.71};  // 8-bit: 137 registers at 64 rows
    static const Pk4GemmCost WIDE8_BF16 = {false, 0.91, 0, 0, 0, 1.47, 1.32, 2.00, 1.78};
    const bool f16 = p.w.dtype == OXQ_F16;
    const Pk4GemmCost &c = p.w.bits == 8      ? (f16 ? WIDE8_F16 : WIDE8_BF16)
                           : p.w.strip == 16 ? (f16 ? NARROW_F16 : NARROW_BF16)
                                             : (f16 ? WIDE_F16 : WIDE_BF16);
    const int64_t groups = ceil_div(ceil_div(p.w.N, (int64_t)64), (int64_t)PK4G_STRIPS);
    const double w64 = (double)(groups * ceil_div(p.M, (int64_t)64)) / cus, w128 = (double)(groups * ceil_div(p.M, (int64_t)128)) / cus;
    auto rounds = [](double w, double full, double part, double part_upto) {
        const double whole = std::floor(w), rest = w - whole;
        return whole * full + (rest <= 0.0 ? 0.0 : rest <= part_upto ? part : full);
    };
    const double c64 = !c.pairs64 || w64 <= 1.0 ? rounds(w64, 1.0, c.part64, 0.75) : w64 <= 2.0 ? c.a64 + c.b64 * w64 : c.slope64 * w64;
    const double c128 = rounds(w128, c.full128, c.part128, 0.7);
    // 128-row workgroups whose last rows (at most 32 behind the whole tiles) are tiles of 32: they start on the CUs that the whole
    // tiles leave idle and take 0.59 of a round.  (At 0.9 - 1 64-row workgroups a CU those are ahead, now that each gets one: us, last rows in
    // tiles of 32 / 64-row workgroups, f16 7552 x 10368 at 651 rows 151 / 112, 1152 x 4672 at 1557 31.5 / 23.3, bf16 4736 x 11712 at 662
    // 111 / 88, 8064 x 18176 at 406 181 / 148.)
    double c_light = 1e30;
    if (can_light) {
        const int64_t whole = groups * (p.M / 128), ncu = (int64_t)cus, h = whole % ncu;
        const double after = h == 0 ? 0.59 * std::ceil((double)groups / cus) * c.full128
                                    : std::max((double)(h + groups) / cus <= 0.7 ? c.part128 : c.full128,
                                               std::min(1.59, 0.59 * std::ceil((double)groups / (double)(ncu - h))) * c.full128);
        c_light = (double)(whole / ncu) * c.full128 + after;
    }
    // the split-K tiles are one workgroup a row tile and 64 columns, in whole rounds too (64-column strips: up to two of them,
    // beyond that fitted without; 1664 x 4224 f16 at 200 rows, 264 tiles, 15.4 us, 12.1 at 300 rows in the two-strip form)
    const double tiles = (double)(ceil_div(p.w.N, (int64_t)64) * ceil_div(p.M, (int64_t)64)) / cus;
    const double c_split = (w64 < 1.0 ? c.split_lo : c.split_hi) *
                           (p.w.strip == 16 ? std::ceil(8.0 * w64 - 1e-9) / 8.0 : tiles <= 2.0 ? std::ceil(tiles) / 8.0 : w64);
    // two strips a workgroup (128 KB of LDS: one a CU), whole rounds of `PK4_MID_ROUND` each
    const double w_mid = (double)(ceil_div(ceil_div(p.w.N, (int64_t)64), (int64_t)2) * ceil_div(p.M, (int64_t)64)) / cus;
    const double c_mid = forced_ks == 1        ? 1e30
                         : p.w.strip == 16 ? rounds(w_mid, PK4N_MID_ROUND, PK4N_MID_PART, 0.5)
                                           : std::ceil(w_mid) * PK4_MID_ROUND;
    // (the split-K tiles address the whole of x with 32 bits)
    const double w_mid128 = (double)(ceil_div(ceil_div(p.w.N, (int64_t)64), (int64_t)2) * ceil_div(p.M, (int64_t)128)) / cus;
    const Pk4Mid128Cost &h = p.w.strip == 16 ? (f16 ? PK4N_MID128_F16 : PK4N_MID128_BF16) : (f16 ? PK4_MID128_F16 : PK4_MID128_BF16);
    const int sets = pk4_sets(p.w.group_shift);
    const bool long_k = !f16 && p.w.strip != 16 && (sets == 4 || (p.w.K >= 3968 && (sets == 2 || w_mid128 <= 2.0)));
    const double c_mid128 = !can_mid128 || forced_ks == 1
                                ? 1e30
                                : rounds(w_mid128, h.full, h.part, h.part_upto) *
                                      (w_mid128 <= h.more_from ? 1.0 : long_k ? PK4_MID128_BF16_MORE_LONG_K : h.more);
    const double c_mid128_k = c_mid128 * (PK4_MID128_LONG_K + PK4_MID128_OVER_K / (double)p.w.K);
    // (against split-K tiles in whole rounds: 3584 x 18944 at 128 rows, 2.3 of them, takes 38 us in bf16, by 2.3 / 8 it would be 28)
    if (c_mid128_k < c64 && c_mid128_k < c128 && c_mid128_k < c_light && c_mid128 < c_mid &&
        c_mid128 < std::max(c_split, c.split_lo * std::ceil(tiles) / 8.0)) return {128, 4};
    if (c_split <= c64 && c_split <= c128 && c_split <= c_light && c_split <= c_mid && (uint64_t)p.M * (uint64_t)p.w.K * 2 < (1ull << 31)) return {0, 1};
    if (c_mid < c64 && c_mid < c128 && c_mid < c_light) return {64, 4};
    // (in f16 the 64-row workgroups are ahead at equal estimates: 2048 x 22016 at 1040 rows 98 us against 102)
    if (c_light <= (f16 ? 0.99 : 1.02) * c64 && c_light <= 1.02 * c128) return {128, 1, true};
    return {c128 < c64 ? 128 : 64, 1};
}
bool pk4_gemm_takes(const oxq_ctx *ctx, const Pk4Problem &p) { return pk4_gemm_form(ctx, p).rows != 0; }

template <typename TT, int MT>
static int pk4n_gemm_go(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)2 * 16 * MT * 256;
    OXQ_HIP_CHECK(grant.ensure((const void *)pk4n_gemm_kernel<TT, MT>, lds));
    hipLaunchKernelGGL((pk4n_gemm_kernel<TT, MT>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w.pw, (const uint16_t *)p.bias,
                       (uint16_t *)p.y, (int)p.M, (int)p.w.K, (int)p.w.N, NG, RT);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <typename TT, int MT>
static int pk4_gemm_go_layout(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    if (p.w.strip == 16) return pk4n_gemm_go<TT, MT>(s, grid, p, NG, RT);
    return p.w.bits == 8 ? pk4_gemm_wide_go<TT, MT, 8, 1>(s, grid, p, NG, RT) : pk4_gemm_wide_go<TT, MT, 4, 1>(s, grid, p, NG, RT);
}
template <typename TT>
static int pk4_gemm_go_light(hipStream_t s, dim3 grid, const Pk4Problem &p, int NG, int RT) {
    return p.w.bits == 8 ? pk4_gemm_wide_go<TT, 8, 8, 1, false, 2>(s, grid, p, NG, RT) : pk4_gemm_wide_go<TT, 8, 4, 1, false, 2>(s, grid, p, NG, RT);
}

int launch_pk4_gemm(oxq_ctx *ctx, hipStream_t s, const Pk4Problem &p) {
    const Pk4GemmForm form = pk4_gemm_form(ctx, p);
    const int rows = form.rows, spw = PK4G_STRIPS / form.ks;
    const int64_t NG = ceil_div(ceil_div(p.w.N, (int64_t)64), (int64_t)spw), RT = form.light ? p.M / rows : ceil_div(p.M, (int64_t)rows);
    // eight strips a workgroup: in the order of pk4g_tile_of; two strips: row tile by row tile
    const int64_t wgs = form.ks == 1 ? pk4g_workgroups(RT, NG) + (form.light ? NG : 0) : RT * NG;
    if (wgs > 0x7FFFFFFF) return fail(OXQ_ERR_UNSUPPORTED, "repacked matmul: m = %lld exceeds the grid", (long long)p.M);
    dim3 grid((unsigned)wgs);
    char name[64];
    plan_name(name, sizeof name, "pk%d_gemm_%s_r%dx%d%s%s%s%s", p.w.bits, p.w.dtype == OXQ_F16 ? "f16" : "bf16", rows, spw,
             form.ks > 1 ? "k4" : form.light ? "r32" : "", p.w.unrounded ? "_gs" : "", p.w.strip == 16 ? "_n16" : "",
             p.act == 1 ? "_silu" : p.act == 2 ? "_gelu" : "");
    set_plan(ctx, name, grid, dim3(512), 1, 1, 0);
    if (ctx->plan_only) return OXQ_OK;
    // (32-bit offsets into the rows of a descriptor: 64 in the two-strip forms)
    if ((uint64_t)(form.ks > 1 ? 64 : rows) * (uint64_t)p.w.K * 2 >= (1ull << 31)) return fail(OXQ_ERR_UNSUPPORTED, "repacked matmul: K too large");
    if (((uintptr_t)p.x | (uintptr_t)p.y) & 15) return fail(OXQ_ERR_UNSUPPORTED, "repacked matmul: x and y must be 16-byte aligned");
    if (p.bias && ((uintptr_t)p.bias & 7)) return fail(OXQ_ERR_UNSUPPORTED, "repacked matmul: bias must be 8-byte aligned");
    if (p.w.unrounded) return form.ks == 4 ? launch_pk4_midfold(s, grid, p, (int)NG) : launch_pk4_gemm_fold(s, grid, p, (int)NG, (int)RT);
    if (form.ks == 4) return rows == 128 ? launch_pk4_mid128(s, grid, p, (int)NG) : launch_pk4_mid(s, grid, p, (int)NG);
    if (pk4_sets(p.w.group_shift) > 1) return launch_pk4_gemm_fine(s, grid, p, rows, (int)NG, (int)RT);
    const bool f16 = p.w.dtype == OXQ_F16;
    if (form.light) return f16 ? pk4_gemm_go_light<F16Traits>(s, grid, p, (int)NG, (int)RT) : pk4_gemm_go_light<BF16Traits>(s, grid, p, (int)NG, (int)RT);
    if (rows == 128)
        return f16 ? pk4_gemm_go_layout<F16Traits, 8>(s, grid, p, (int)NG, (int)RT) : pk4_gemm_go_layout<BF16Traits, 8>(s, grid, p, (int)NG, (int)RT);
    return f16 ? pk4_gemm_go_layout<F16Traits, 4>(s, grid, p, (int)NG, (int)RT) : pk4_gemm_go_layout<BF16Traits, 4>(s, grid, p, (int)NG, (int)RT);
}

}  // namespace oxq
