// Block-scaled F8E4M3 weights times bf16 rows on the matrix cores, straight from the checkpoint tensor [N, K]
// (moe.rs:106-113 Fp8Cached::forward beyond the GEMV: dequantize to bf16, then the product).  The weight the matrix
// cores see is the reference's bf16(f32(f8) * scale) (quant_kernels.metal:3877-3911), bit for bit; f32 accumulation.
//
// What bounds these sizes (an expert of 2048 x 5632 is 11.5 MB, resident in the Infinity Cache) is latency and, from a
// few row tiles on, the decode: 16 vector instructions for the 8 weights a lane brings to an MFMA step.  The staged tile
// matmul of blockq_mm.hip pays two barriers for every 256 rows of K, and slices K over workgroups with a second launch.
// Two forms here, after the matrix-core kernels of the GGUF layers (gguf_mfma.hip):
//   f8_tile_kernel   16 MT rows x NS strips of 16 columns a workgroup; its eight waves split K, each stages its own x and
//                    weights, no barrier before the sum - up to a few hundred rows of an expert;
//   f8_gemm_kernel   64 rows x two groups of 64 columns with K split over four waves each (KS = 4, and over workgroups
//                    where columns are few), or x eight groups (KS = 1);
//   f8_gemm128_kernel  128 rows x four groups of 32 columns with K split over two waves each, or x eight groups.
// A strip's rows lie K bytes apart, so loads that fill operands directly touch 16 lines each, one lane at a time: 64
// cycles of the address unit for 1 KB, and that bound the first version (2.45 us for 64 x 512 x 128 a CU).  Loads now
// take whole 128-byte (64-byte) runs of a row and turn to operand order through the wave's own LDS: 2.1 us.
// Measured, us, before (GEMV / staged tiles) -> now: 5632 x 5632 at 1, 33, 96, 256, 1024 rows 11.3 -> 8.3, 22.9 -> 15.9,
// 31.5 -> 18.4, 52 -> 34, 144 -> 75; 2048 x 5632 at 3, 33, 96 rows 8.5 -> 4.8, 12.5 -> 7.0, 17.0 -> 10.0; 512 x 768 at
// 33 rows 6.6 -> 3.0.
// Needs block_r a multiple of 16 (a strip has one scale a chunk), block_c 128 times a power of two; other grids keep
// blockq_mm.hip.
#include "oxq_device.hpp"
#include "oxq_internal.hpp"
#include "oxq_mfma.hpp"
#include "pk4_common.hpp"

#include <algorithm>
#include <cmath>

namespace oxq {

__device__ __forceinline__ uint32_t f8_pair(float a, float b) {
    return (uint32_t)BF16Traits::from_f32(a) | ((uint32_t)BF16Traits::from_f32(b) << 16);
}
// eight bytes times the scale as four bf16 pairs: exact conversion, one product, one rounding each
__device__ __forceinline__ void f8_operand(uint32_t w0, uint32_t w1, float s, uint32_t (&b)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = i < 2 ? w0 : w1;
        const float2_t v = (i & 1) ? (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)w, true)
                                   : (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
        b[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{v[0] * s, v[1] * s}, bf16x2_t));
    }
}

template <int N, typename F> __device__ __forceinline__ void each(F f) {  // f(0) .. f(N - 1), constants
    if constexpr (N > 1) each<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
}

// XQ: loads of x a chunk (four rows each).  RD chunks in flight a wave: what hides the cache's latency; two or three are
// what the registers hold (48 rows: 256 registers, one chunk of x; the LDS slots fill the CU's 160 KB).
// NL > 0: no wave has more than NL chunks and none fewer than NL - 1, all of them requested at once; 0: a loop.  A load that brings
// nothing (past a wave's last chunk) takes its turn in the address unit as any other, and a kernel's instructions come from memory
// anew at each launch: with a body for each number of chunks neither a load nor a jump is left over.  us, one loop with such loads for
// all -> now: 5632 x 2816 (N x K) at 1 / 8 / 16 rows 5.8 / 6.6 / 7.9 -> 5.5 / 6.0 / 6.8, 5632 x 2048 at 24 / 48 / 96 / 144 6.8 / 7.8 / 10.6 / 16.6 ->
// 6.1 / 7.2 / 10.0 / 15.5, 768 x 512 at 33 3.3 -> 3.0; with bodies for all of them in one kernel 1 and 3 rows were 2 - 6 % behind.
template <int MT, int NS, int NW, int XQ, int NL>
__global__ __launch_bounds__(NW * 64) void f8_tile_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ w,
                                                          const float *__restrict__ scales, uint16_t *__restrict__ y,
                                                          int M, int K, int N, int block_r, int cshift, int s_cols, int s_rows) {
    typedef BF16Traits TT;
    typedef MfmaOps<TT> Ops;
    constexpr int ROWS = 16 * MT, AQ = XQ, SLOT = ROWS * 256, WSLOT = NS * 2048, OOB = 0x7FFFFF00;
    constexpr int RD = NL > 0 ? NL : NS > 1 ? 2 : 3;  // chunks in flight a wave
    constexpr int XD = MT == 3 ? 1 : RD;              // and of x, which comes from L2 (48 rows: the registers allow one)
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int j = blockIdx.x;
    const int m0 = blockIdx.z * ROWS, n0 = 16 * NS * j;  // grid y is K slices to the epilogue: always 1 here
    const int NC = K >> 7;
    const int cbase = NC / NW, crem = NC % NW;
    const int nloc = cbase + (wave < crem ? 1 : 0);
    const int cc0 = wave * cbase + min(wave, crem);
    unsigned char *slot = pk4_lds + wave * SLOT, *wslot = pk4_lds + NW * SLOT + wave * WSLOT;

    const int wrows = min(N - n0, 16 * NS), xrows = min(M - m0, ROWS);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(w + (size_t)n0 * K, (uint32_t)wrows * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(scales, (uint32_t)(s_rows * s_cols) * 4u);
    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(w, 0u);
    // load h of strip f: rows 8 h + lane / 8, whole 128-byte lines; into LDS with the 16-byte pieces of row r swapped by
    // r % 8, out of it as operands
    int voff_w[NS][2], soff_s[NS];
#pragma unroll
    for (int f = 0; f < NS; ++f) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 16 * f + 8 * h + (lane >> 3);
            voff_w[f][h] = r < wrows ? r * K + (lane & 7) * 16 : OOB;
        }
        soff_s[f] = min((n0 + 16 * f) / block_r, s_rows - 1) * s_cols;
    }
    const int w_wr = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);  // + 1024 h + 2048 f
    int w_rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) w_rd[h] = ni * 128 + (((4 * h + kb) ^ (ni & 7)) << 4);
    int voff_a[AQ];
#pragma unroll
    for (int q = 0; q < AQ; ++q) {
        const int r = 4 * q + kb;
        voff_a[q] = r < xrows ? (r * K * 2 + ni * 16) : OOB;
    }
    int a_wr[4];
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) a_wr[qq] = kb * 256 + (((ni ^ kb) ^ (qq << 2)) << 4);
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + ((pk4_x_chunk<1>(st, kb) ^ ni) << 4);
#pragma unroll
    for (int q = AQ; q < 4 * MT; ++q) {  // rows no call of this instantiation brings stay zero
        const int row = 4 * q + kb;
        *(u32x4_t *)(slot + row * 256 + ((ni ^ (row & 15)) << 4)) = u32x4_t{0u, 0u, 0u, 0u};
    }

    u32x4_t wr[RD][NS][2], ar[XD][AQ];
    float sr[RD][NS];
    auto request_x = [&](int i, u32x4_t (&a)[AQ]) {
        const __amdgpu_buffer_rsrc_t rx = i < nloc ? rs_x : rs_none;  // wave-uniform
#pragma unroll
        for (int k = 0; k < AQ; ++k) a[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, voff_a[k], (cc0 + i) * 256, 0);
    };
    auto request = [&](int i, u32x4_t (&q)[NS][2], float (&s)[NS]) {
        const bool live = i < nloc;
        const __amdgpu_buffer_rsrc_t rw = live ? rs_w : rs_none, rs = live ? rs_s : rs_none;
        const int c = cc0 + i, sc = c >> cshift;
#pragma unroll
        for (int f = 0; f < NS; ++f) {
            s[f] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, 0, (soff_s[f] + sc) * 4, 0));
#pragma unroll
            for (int h = 0; h < 2; ++h) q[f][h] = __builtin_amdgcn_raw_buffer_load_b128(rw, voff_w[f][h], c * 128, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // chunks are requested in the order they are used
    };

    float4_t acc[MT][NS];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NS; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};

    // placed: x lies in the slot.  more: request chunk i + RD; next: x of chunk i + 1
    auto chunk = [&](int i, auto cur_c, bool placed, auto more_c, auto next_c) {
        constexpr int CUR = decltype(cur_c)::value;
        if (!placed) {
#pragma unroll
            for (int q = 0; q < AQ; ++q) *(u32x4_t *)(slot + q * 1024 + a_wr[q & 3]) = ar[CUR % XD][q];
        }
#pragma unroll
        for (int f = 0; f < NS; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h) *(u32x4_t *)(wslot + f * 2048 + h * 1024 + w_wr) = wr[CUR][f][h];
        if constexpr (XD == 1 && next_c.value) {
            request_x(i + 1, ar[0]);
            __builtin_amdgcn_sched_barrier(0);
        }
        u32x4_t wq[NS];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st % 2 == 0) {
#pragma unroll
                for (int f = 0; f < NS; ++f) wq[f] = *(const u32x4_t *)(wslot + f * 2048 + w_rd[st >> 1]);
            }
            uint32_t a[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const u32x4_t av = *(const u32x4_t *)(slot + mt * 4096 + a_rd[st]);
                a[mt][0] = av[0], a[mt][1] = av[1], a[mt][2] = av[2], a[mt][3] = av[3];
            }
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                uint32_t b[4];
                f8_operand(wq[f][2 * (st & 1)], wq[f][2 * (st & 1) + 1], sr[CUR][f], b);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
            }
            if constexpr (MT == 3) __builtin_amdgcn_sched_barrier(0);  // no operands of the next step early: no registers for them
        }
        if constexpr (more_c.value) {
            if constexpr (XD > 1) request_x(i + RD, ar[CUR]);
            request(i + RD, wr[CUR], sr[CUR]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (NL > 0) {
        // 48 rows have registers for one chunk of x: the first goes straight into its slot, so that the second is under way beside it
        // (us: 5632 x 2048 at 33 / 48 rows 7.2 / 7.5 -> 7.0 / 7.2; 48 rows x 64 columns of two chunks, 96 rows, 10.0 -> 10.15, stay).
        constexpr bool DMA = MT == 3 && (NS == 2 || NL == 1);
        if constexpr (DMA) {
            static_assert(NL <= 2 && AQ == 4 * MT, "one chunk in the slot, one in registers; whole slots");
            if (nloc > 0) {
#pragma unroll
                for (int q = 0; q < AQ; ++q) {  // lane 16 kb + ni fills piece ni of row r: that of the columns ni ^ (r % 16)
                    const int r = 4 * q + kb;
                    pk4g_load_lds16(rs_x, slot + q * 1024, r < xrows ? r * K * 2 + ((ni ^ (r & 15)) << 4) : OOB, cc0 * 256);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        each<NL>([&](auto s_c) {
            constexpr int S = decltype(s_c)::value;
            const int i = nloc - NL + S;
            if (S == 0 && i < 0) return;
            if (XD > 1 || (i > 0) == DMA) request_x(i, ar[S % XD]);
            request(i, wr[S], sr[S]);
        });
        each<NL>([&](auto s_c) {
            constexpr int S = decltype(s_c)::value;
            const int i = nloc - NL + S;
            if (S == 0 && i < 0) return;
            if constexpr (DMA) {
                pk4g_wait_vmcnt<(NL - 1 - S) * (AQ + 3 * NS)>();  // the first chunk is here, the second under way
                __builtin_amdgcn_sched_barrier(0);
            }
            chunk(i, s_c, DMA && i == 0, std::false_type{}, std::integral_constant<bool, (!DMA && S + 1 < NL)>{});
        });
    } else {
#pragma unroll
        for (int d = 0; d < RD; ++d) {
            if (d < XD) request_x(d, ar[d]);
            request(d, wr[d], sr[d]);
        }
        int i = 0;
        for (; i + RD < nloc; i += RD)
            each<RD>([&](auto s_c) { chunk(i + s_c.value, s_c, false, std::true_type{}, std::true_type{}); });
        each<RD>([&](auto s_c) {
            constexpr int S = decltype(s_c)::value;
            if (i + S < nloc) chunk(i + S, s_c, false, std::false_type{}, std::integral_constant<bool, (S + 1 < RD)>{});
        });
    }
    pk4n_epilogue<TT, MT, NS, NW, true>(acc, nullptr, y, nullptr, M, N, j, m0, wave, lane);
}

// The sums of a workgroup's waves: column groups of 16 NS, wave = column group + (8 / KS) x share of K.  All row tiles of this wave
// (KS = 1), or MT / KS of them summed over the waves of the column group, in K order: the same sum whatever the timing.
template <int MT, int NS, int KS>
__device__ __forceinline__ void f8_gemm_finish(float4_t (&acc)[MT][NS], uint16_t *__restrict__ y, float *__restrict__ part, int M, int N,
                                               int m0, int n0, int wave, int lane, bool live) {
    static_assert(MT % KS == 0, "the waves of a column group finish as many row tiles each");
    constexpr int SPW = 8 / KS, FT = MT / KS;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];
    const int ni = lane & 15, kb = lane >> 4, ws = wave % SPW, kq = wave / SPW;
    float4_t fin[FT][NS];
    if constexpr (KS == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < NS; ++f) fin[mt][f] = acc[mt][f];
    } else {
        // over the buffers of x, once the zeros requested past the last round are in them
        typedef float part_t __attribute__((ext_vector_type(NS)));
        pk4g_wait_vmcnt<0>();
        __syncthreads();
        part_t *red = (part_t *)pk4_lds;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                part_t v;
#pragma unroll
                for (int f = 0; f < NS; ++f) v[f] = acc[mt][f][e];
                red[((wave * MT + mt) * 4 + e) * 64 + lane] = v;
            }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < FT; ++t) {
#pragma unroll
            for (int f = 0; f < NS; ++f) fin[t][f] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const part_t v = red[(((k * SPW + ws) * MT + FT * kq + t) * 4 + e) * 64 + lane];
#pragma unroll
                    for (int f = 0; f < NS; ++f) fin[t][f][e] += v[f];
                }
        }
    }
    if (!live) return;
    // row 16 mt + 4 kb + e, column n0 + 16 f + ni
    // In groups of four columns, one store each: with 2 (4) bytes a lane and store the epilogue of 64 x 512 took 7 us and that of
    // 128 x 256 as much (512 x 768 at 65 - 2048 rows 20 -> 15 and 18.6 -> 12.4 us a launch).
    if (N % 4 == 0 && (gridDim.y > 1 || ((uintptr_t)y & 7) == 0)) {
#pragma unroll
        for (int t = 0; t < FT; ++t)
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                const int row = m0 + 16 * (FT * kq + t) + 4 * kb + (ni & 3), n = n0 + 16 * f + (ni & 12);
                const bool there = row < M && n < N;
                if (gridDim.y > 1) {
                    const float4_t v = quad_turn32(fin[t][f], lane);
                    if (there) *(float4_t *)(part + ((size_t)blockIdx.y * M + row) * N + n) = v;
                } else {
                    const uint2 v = quad_turn16(f8_pair(fin[t][f][0], fin[t][f][1]), f8_pair(fin[t][f][2], fin[t][f][3]), lane);
                    if (there) *(uint2 *)(y + (size_t)row * N + n) = v;
                }
            }
        return;
    }
#pragma unroll
    for (int t = 0; t < FT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + 16 * (FT * kq + t) + 4 * kb + e;
            if (row >= M) continue;
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                const int n = n0 + 16 * f + ni;
                if (n >= N) continue;
                if (gridDim.y > 1) part[((size_t)blockIdx.y * M + row) * N + n] = fin[t][f][e];
                else y[(size_t)row * N + n] = BF16Traits::from_f32(fin[t][f][e]);
            }
        }
}

template <int MT, int KS>
__global__ __launch_bounds__(512) void f8_gemm_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ w,
                                                      const float *__restrict__ scales, uint16_t *__restrict__ y,
                                                      float *__restrict__ part, int M, int K, int N, int NG, int RT,
                                                      int cslice, int block_r, int cshift, int s_cols, int s_rows) {
    typedef BF16Traits TT;
    typedef MfmaOps<TT> Ops;
    static_assert(KS == 1 || KS == MT, "wave kq of a column group finishes row tile kq");
    constexpr int SPW = 8 / KS;  // waves of 64 columns a workgroup
    constexpr int ROWS = 16 * MT, XBUF = KS * ROWS * 256, XV = ROWS / 4 / SPW, OOB = 0x7FFFFF00;
    constexpr int RING = 12;  // vector loads of weights and scales between two rounds' loads of x
    static_assert(MT == 4, "the way of a half chunk through LDS is written for four groups a step");
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws = wave % SPW, kq = wave / SPW;  // the wave's column group of the workgroup, and its share of K
    int rt, g;
    if constexpr (KS == 1) {
        if ((int)blockIdx.x >= RT * NG) return;  // the whole workgroup, before any barrier
        pk4g_tile_of((int)blockIdx.x, RT, NG, rt, g);
    } else {
        rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;
    }
    const int n0 = 64 * (g * SPW + ws);
    const bool live = n0 < N;
    const int m0 = rt * ROWS;
    const int NC = K >> 7;
    const int cbeg = (int)blockIdx.y * cslice, cend = min(NC, cbeg + cslice);
    const int NR = (cend - cbeg + KS - 1) / KS;
    const int xrows = min(M - m0, ROWS), wrows = live ? min(N - n0, 64) : 0;

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(w, 0u);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(w + (size_t)(live ? n0 : 0) * K, (uint32_t)wrows * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(scales, (uint32_t)(s_rows * s_cols) * 4u);
    // half h of a chunk (64 bytes a row, two steps): load f brings rows 16 f + lane / 4, and goes through the wave's 4 KB
    // of LDS to become operands, the 16-byte pieces of row r swapped by (r / 4) % 4
    int voff_w[4], soff_s[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const int r = 16 * f + (lane >> 2);
        voff_w[f] = r < wrows ? r * K + (lane & 3) * 16 : OOB;
        soff_s[f] = min((n0 + 16 * f) / block_r, s_rows - 1) * s_cols;
    }
    unsigned char *wslot = pk4_lds + 2 * XBUF + wave * 4096;
    const int w_wr = (lane >> 2) * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4), w_rd = ni * 64 + ((kb ^ ((ni >> 2) & 3)) << 4);
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (ws * XV + q) + (lane >> 4);
        xo[q] = r * K * 2 + (((lane & 15) ^ (r & 15)) << 4);
    }
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + ((pk4_x_chunk<1>(st, kb) ^ ni) << 4);

    u32x4_t wr[2][4], wq[2][4];  // [half][strip]: as loaded, as operands
    float sr[2][4];
    auto dma_x = [&](int r) {
        const int i = cbeg + KS * r + kq;
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_x : rs_none;
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256) + (ws * XV + q) * 1024, xo[q], i * 256);
    };
    auto load_w = [&](int i, int h) {
        const __amdgpu_buffer_rsrc_t rw = i < cend ? rs_w : rs_none;
#pragma unroll
        for (int f = 0; f < 4; ++f) wr[h][f] = __builtin_amdgcn_raw_buffer_load_b128(rw, voff_w[f], i * 128 + h * 64, 0);
    };
    auto load_s = [&](int i, float (&s)[4]) {
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_s : rs_none;
#pragma unroll
        for (int f = 0; f < 4; ++f) s[f] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, 0, (soff_s[f] + (i >> cshift)) * 4, 0));
    };
    auto put_w = [&](int h, int f) { *(u32x4_t *)(wslot + f * 1024 + w_wr) = wr[h][f]; };
    auto get_w = [&](int h, int f) { wq[h][f] = *(const u32x4_t *)(wslot + f * 1024 + w_rd); };

    // Software pipeline.  The products of step st run on operands decoded during step st - 1, with the fragment of x
    // read three groups (of four products) before its use; the barrier that hands the next round's x over stands where
    // the last fragment of this round has been read, three groups before the round's end, so no wait is exposed there.
    constexpr int GROUPS = 4 * MT, AH = 3;
    u32x4_t a[4];
    uint32_t b[2][4][4];
    auto read_x = [&](int r, int u) { a[u & 3] = *(const u32x4_t *)(pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256) + (u % MT) * 4096 + a_rd[u / MT]); };
    auto decode = [&](int st, int f, int pp, const float (&sc)[4]) {
        const uint32_t word = wq[st >> 1][f][2 * (st & 1) + (pp >> 1)];
        const float2_t v = (pp & 1) ? (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)word, true)
                                    : (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)word, false);
        b[st & 1][f][pp] = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{v[0] * sc[f], v[1] * sc[f]}, bf16x2_t));
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
    load_w(cbeg + kq, 0);
    load_s(cbeg + kq, sr[0]);
    load_w(cbeg + kq, 1);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < 4; ++f) put_w(0, f);
#pragma unroll
    for (int f = 0; f < 4; ++f) get_w(0, f);
    pk4g_wait_vmcnt<4>();
    __syncthreads();
    dma_x(1);
    __builtin_amdgcn_sched_barrier(0);
    load_w(cbeg + KS + kq, 0);
    load_s(cbeg + KS + kq, sr[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < AH; ++u) read_x(0, u);
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int pp = 0; pp < 4; ++pp) decode(0, f, pp, sr[0]);

    auto chunk = [&](int r, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        const int i = cbeg + KS * r + kq;  // past the slice (a ragged last round): zeros from both streams
#pragma unroll
        for (int u = 0; u < GROUPS; ++u) {
            const int st = u / MT, mt = u % MT;
            if (u == GROUPS - AH) {
                __builtin_amdgcn_sched_barrier(0);
                pk4g_wait_vmcnt<RING>();  // this wave's part of the next round of x (requested before the weights) is in LDS
                __syncthreads();          // and every wave holds its last fragment of this round: the buffer is free
                dma_x(r + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (u + AH < GROUPS) read_x(r, u + AH);
            else read_x(r + 1, u + AH - GROUPS);
            if (st == 0 || st == 2) {  // half 1 of this chunk, half 0 of the next: in LDS, then out as operands
                const int h = st == 0 ? 1 : 0, k = 2 * (mt & 1);
                if (mt < 2) put_w(h, k), put_w(h, k + 1);
                else get_w(h, k), get_w(h, k + 1);
            }
#pragma unroll
            for (int t = 0; t < 16 / MT; ++t) {
                const int k = mt * (16 / MT) + t;
                decode((st + 1) & 3, k >> 2, k & 3, sr[st < 3 ? CUR : CUR ^ 1]);
            }
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                uint32_t am[4] = {a[u & 3][0], a[u & 3][1], a[u & 3][2], a[u & 3][3]};
                acc[mt][f] = Ops::mfma(am, b[st & 1][f], acc[mt][f]);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (st == 0 || st == 2) {
                if (mt < 2) __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
                else __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 16 / MT, 0);
            }
            if (mt == MT - 1 && (st == 0 || st == 2)) {
                __builtin_amdgcn_sched_barrier(0);
                if (st == 0) load_w(i + KS, 1);
                else load_w(i + 2 * KS, 0), load_s(i + 2 * KS, sr[CUR]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    {
        int r = 0;
        for (; r + 1 < NR; r += 2) {
            chunk(r, std::integral_constant<int, 0>{});
            chunk(r + 1, std::integral_constant<int, 1>{});
        }
        if (r < NR) chunk(r, std::integral_constant<int, 0>{});
    }

    f8_gemm_finish<MT, 4, KS>(acc, y, part, M, N, m0, n0, wave, lane, live);
}

// 128 rows, a wave has two strips: a decoded weight serves eight row tiles instead of four (two vector instructions an MFMA), at the
// price of fragments of x that feed two MFMAs.  KS = 1: 256 columns, KS = 2: 128 with K over the two waves of a column group.
// What bounds it: issue.  At 5632 x 5632 and 1024 rows the MFMAs take 55 % of the time, with 2.4 other vector instructions each, and reads
// of LDS 38 %, at the 256 bytes a clock that a loop of 16-byte reads reaches (K over two waves, 640 rows: 43 % and 32 %).
// us, best of the forms of 64 rows -> 128: 5632 x 5632 at 128 / 400 / 640 / 1024 rows 32 / 68 / 70 / 100 -> 24 / 48 / 50 / 75, 4096 x
// 4096 at 640 / 1024 53 / 55 -> 38 / 42, 2048 x 5632 at 640 / 1024 34 / 46 -> 24 / 34.  Bits as f8_gemm_kernel's (KS = 1).
template <int KS>
__global__ __launch_bounds__(512) void f8_gemm128_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ w,
                                                         const float *__restrict__ scales, uint16_t *__restrict__ y,
                                                         float *__restrict__ part, int M, int K, int N, int NG, int RT,
                                                         int cslice, int block_r, int cshift, int s_cols, int s_rows) {
    typedef MfmaOps<BF16Traits> Ops;
    constexpr int MT = 8, NS = 2, SPW = 8 / KS, ROWS = 16 * MT, XBUF = KS * ROWS * 256, XV = ROWS / 4 / SPW, OOB = 0x7FFFFF00;
    constexpr int RING = 6;  // vector loads of weights and scales between two rounds' loads of x
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int ws = wave % SPW, kq = wave / SPW;  // the wave's column group of the workgroup, and its share of K
    int rt, g;
    if constexpr (KS == 1) {
        if ((int)blockIdx.x >= RT * NG) return;  // the whole workgroup, before any barrier
        pk4g_tile_of((int)blockIdx.x, RT, NG, rt, g);
    } else {
        rt = (int)blockIdx.x / NG, g = (int)blockIdx.x % NG;
    }
    const int n0 = 16 * NS * (g * SPW + ws);
    const bool live = n0 < N;
    const int m0 = rt * ROWS;
    const int NC = K >> 7;
    const int cbeg = (int)blockIdx.y * cslice, cend = min(NC, cbeg + cslice);
    const int NR = (cend - cbeg + KS - 1) / KS;
    const int xrows = min(M - m0, ROWS), wrows = live ? min(N - n0, 16 * NS) : 0;

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(w, 0u);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(w + (size_t)(live ? n0 : 0) * K, (uint32_t)wrows * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(scales, (uint32_t)(s_rows * s_cols) * 4u);
    // a chunk of the wave's columns is 4 KB: load q brings rows 8 q + lane / 8 whole, and the wave's own LDS turns them to
    // operands, the 16-byte pieces of row r swapped by r % 8
    int voff_w[4], soff_s[NS];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = 8 * q + (lane >> 3);
        voff_w[q] = r < wrows ? r * K + (lane & 7) * 16 : OOB;
    }
#pragma unroll
    for (int f = 0; f < NS; ++f) soff_s[f] = min((n0 + 16 * f) / block_r, s_rows - 1) * s_cols;
    unsigned char *wslot = pk4_lds + 2 * XBUF + wave * 4096;
    const int w_wr = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    int w_rd[2];  // half h of a chunk: two steps
#pragma unroll
    for (int h = 0; h < 2; ++h) w_rd[h] = ni * 128 + (((4 * h + kb) ^ (ni & 7)) << 4);
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (ws * XV + q) + (lane >> 4);
        xo[q] = r * K * 2 + (((lane & 15) ^ (r & 15)) << 4);
    }
    int a_rd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_rd[st] = ni * 256 + ((pk4_x_chunk<1>(st, kb) ^ ni) << 4);

    u32x4_t wr[4], wq[2][NS];  // as loaded; [half][strip]: as operands
    float sr[2][NS];
    auto dma_x = [&](int r) {
        const int i = cbeg + KS * r + kq;
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_x : rs_none;
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256) + (ws * XV + q) * 1024, xo[q], i * 256);
    };
    auto load_w = [&](int i) {
        const __amdgpu_buffer_rsrc_t rw = i < cend ? rs_w : rs_none;
#pragma unroll
        for (int q = 0; q < 4; ++q) wr[q] = __builtin_amdgcn_raw_buffer_load_b128(rw, voff_w[q], i * 128, 0);
    };
    auto load_s = [&](int i, float (&s)[NS]) {
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_s : rs_none;
#pragma unroll
        for (int f = 0; f < NS; ++f) s[f] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, 0, (soff_s[f] + (i >> cshift)) * 4, 0));
    };
    auto put_w = [&](int q) { *(u32x4_t *)(wslot + q * 1024 + w_wr) = wr[q]; };
    auto get_w = [&](int h, int f) { wq[h][f] = *(const u32x4_t *)(wslot + f * 2048 + w_rd[h]); };

    // The pipeline of f8_gemm_kernel with a group of two products: operands decoded a step ahead, fragments of x read AH groups
    // ahead, the barrier AH groups before the round's end.  The next chunk's weights go into LDS in step 1 (this chunk's were all
    // read before it began) and come out by halves in steps 2 and 3, each behind the last decode from the half it replaces.
    constexpr int GROUPS = 4 * MT, AH = 3;
    u32x4_t a[4];
    uint32_t b[2][NS][4];
    auto read_x = [&](int r, int u) { a[u & 3] = *(const u32x4_t *)(pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256) + (u % MT) * 4096 + a_rd[u / MT]); };
    auto decode = [&](int st, int f, int pp, const float (&sc)[NS]) {
        const uint32_t word = wq[st >> 1][f][2 * (st & 1) + (pp >> 1)];
        const float2_t v = (pp & 1) ? (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)word, true)
                                    : (float2_t)__builtin_amdgcn_cvt_pk_f32_fp8((int)word, false);
        b[st & 1][f][pp] = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{v[0] * sc[f], v[1] * sc[f]}, bf16x2_t));
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
    load_w(cbeg + kq);
    load_s(cbeg + kq, sr[0]);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][NS];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NS; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; ++q) put_w(q);
#pragma unroll
    for (int f = 0; f < NS; ++f) get_w(0, f), get_w(1, f);
    pk4g_wait_vmcnt<0>();
    __syncthreads();
    dma_x(1);
    __builtin_amdgcn_sched_barrier(0);
    load_w(cbeg + KS + kq);
    load_s(cbeg + KS + kq, sr[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < AH; ++u) read_x(0, u);
#pragma unroll
    for (int f = 0; f < NS; ++f)
#pragma unroll
        for (int pp = 0; pp < 4; ++pp) decode(0, f, pp, sr[0]);

    auto chunk = [&](int r, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        const int i = cbeg + KS * r + kq;  // past the slice (a ragged last round): zeros from both streams
#pragma unroll
        for (int u = 0; u < GROUPS; ++u) {
            const int st = u / MT, mt = u % MT;
            if (u == GROUPS - AH) {
                __builtin_amdgcn_sched_barrier(0);
                pk4g_wait_vmcnt<RING>();  // this wave's part of the next round of x (requested before the weights) is in LDS
                __syncthreads();          // and every wave holds its last fragment of this round: the buffer is free
                dma_x(r + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (u + AH < GROUPS) read_x(r, u + AH);
            else read_x(r + 1, u + AH - GROUPS);
            if (st == 1 && mt < 4) put_w(mt);
            if (st == 2 && mt < NS) get_w(0, mt);
            if (st == 3 && mt < NS) get_w(1, mt);
            decode((st + 1) & 3, mt >> 2, mt & 3, sr[st < 3 ? CUR : CUR ^ 1]);
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                uint32_t am[4] = {a[u & 3][0], a[u & 3][1], a[u & 3][2], a[u & 3][3]};
                acc[mt][f] = Ops::mfma(am, b[st & 1][f], acc[mt][f]);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (st == 1 && mt < 4) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            if (st >= 2 && mt < NS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            if (mt == MT - 1 && (st == 1 || st == 2)) {
                __builtin_amdgcn_sched_barrier(0);
                if (st == 1) load_w(i + 2 * KS);
                else load_s(i + 2 * KS, sr[CUR]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    {
        int r = 0;
        for (; r + 1 < NR; r += 2) {
            chunk(r, std::integral_constant<int, 0>{});
            chunk(r + 1, std::integral_constant<int, 1>{});
        }
        if (r < NR) chunk(r, std::integral_constant<int, 0>{});
    }
    f8_gemm_finish<MT, NS, KS>(acc, y, part, M, N, m0, n0, wave, lane, live);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int64_t f8_s_rows(const F8Problem &p) { return p.N / p.block_r; }

static bool f8_shape_ok(const F8Problem &p) {
    return p.K % 128 == 0 && p.block_c % 128 == 0 && (p.block_c & (p.block_c - 1)) == 0 && p.block_r % 16 == 0 &&
           ((uintptr_t)p.x & 15) == 0 && ((uintptr_t)p.w & 15) == 0 && ((uintptr_t)p.scales & 3) == 0 && p.K * 128 < (1ll << 31) &&
           f8_s_rows(p) * p.s_cols * 4 < (1ll << 31);
}

// Which form, by estimated us.  Fitted over nine shapes (512..7168 x 512..7168) at 17..1024 rows; the pick is within 4 %
// of the best of all forms at nearly every one:
//   tiles of 32 rows x 16 columns        2.0 + rounds of 256 workgroups x (0.9 + 1.25 x chunks a wave)
//   tiles of 32 rows x 64 columns        1.4 + rounds x (2.5 + 2.05 x chunks a wave)
//   tiles of 48 rows x 64 columns        1.4 + rounds x (4.4 + 2.15 x chunks a wave)
//   tiles of 32 rows x 32 columns        1.4 + rounds x (1.15 + 1.8 x chunks a wave)
//   tiles of 48 rows x 32 columns        1.4 + rounds x (1.7 + 2.0 x chunks a wave)
// A workgroup's LDS slots leave room for one a CU, so the tile that just fits one round of CUs is ahead; the two of 32
// columns stand between the strips and the 64-column groups (fitted over 512..7168 x 768..7168 at 20..320 rows, 1.15 x the fit:
// ahead at 163 of 480 points, by 1.28 x there, and behind at none).  Us, without them -> with: 3968 x 3456 at 33, 64, 96 rows
// 13.1 -> 9.8, 13.3 -> 10.1, 15.1 -> 11.4; 5632 x 5632 at 33 rows 15.7 -> 12.1; 1408 x 2048 at 96 rows 6.7 -> 4.9.
//   64 rows x 128 columns, K over waves  rounds x (7.5 + 2.45 x rounds of four chunks); K slices add a second launch and
//                                        the partials' traffic
//   128 rows x 128 columns, K over waves 6.4 + rounds x (1.2 + 1.6 x rounds of two chunks) + 0.36 x those, of the CUs in use; K slices likewise
//   64 rows x 512 columns                rounds x (7 + 2.1 x chunks)
//   128 rows x 256 columns               rounds x (7.5 + 1.6 x chunks)
// (The last four fitted again over 40 layers of 512..7168 x 512..7168 at 17..2048 rows, every form forced at each of 160 calls:
// 0.9 % behind the fastest form together, 148 within 5 %, 157 within 12 %.  That of 128 rows x 128 columns, fitted there without a term of
// its own for slices, took 57 of 2592 calls of 520 other layers that a form without 128 rows ends 4 - 38 % earlier, all of long K and few columns
// (7296 x 640 at 218 rows 18.9 / 13.6 us, 7936 x 1792 at 157 21.9 / 17.2); fitted on half of those layers, 5 of 2592, the most 9 %, and 1.7 %
// behind the fastest form together.)
//   the staged tiles of blockq_mm.hip    from 33 rows and up to K = 2048, where a workgroup of eight waves has too little K
//                                        to share: several small workgroups a CU win at some shapes
struct F8Form {
    int kind, ns, slices;  // kind 0: tiles, 4 | 1: KS of the gemm kernel of 64 rows, 2: the gemm kernel of 128, -1: blockq_mm.hip
    int mt = 0;            // tiles of 16 mt rows (0: by the rows at hand); KS of the kernel of 128 rows
};
static F8Form f8_form(const oxq_ctx *ctx, const F8Problem &p) {
    const double cus = ctx->num_cus > 0 ? ctx->num_cus : 256, mn = (double)p.M * (double)p.N;
    const int64_t chunks = p.K / 128, strips = ceil_div(p.N, (int64_t)16), groups = ceil_div(p.N, (int64_t)64);
    const double per_wave = (double)ceil_div(chunks, (int64_t)8);
    const int forced = tune(ctx, OXQ_TUNE_F8_FORM, -1), fs = tune(ctx, OXQ_TUNE_F8_SLICES, 0);
    F8Form best = {0, 1, 1};
    double least = 1e30;
    auto offer = [&](int form, double us, F8Form f) {
        if (forced >= 0 ? form == forced : us < least) least = us, best = f;
    };
    const double tiles = (double)ceil_div(p.M, (int64_t)(p.M > 16 ? 32 : 16));
    offer(0, 2.0 + std::ceil((double)strips * tiles / cus) * (0.9 + 1.25 * per_wave), {0, 1, 1});
    if (p.M <= 16) return best;  // a single row tile is bound by the weights' latency: the most workgroups
    offer(2, 1.4 + std::ceil((double)groups * tiles / cus) * (2.5 + 2.05 * per_wave), {0, 4, 1});
    offer(3, 1.4 + std::ceil((double)groups * (double)ceil_div(p.M, (int64_t)48) / cus) * (4.4 + 2.15 * per_wave), {0, 4, 1, 3});
    const double pairs = (double)ceil_div(strips, (int64_t)2);
    offer(5, 1.4 + std::ceil(pairs * tiles / cus) * (1.15 + 1.8 * per_wave), {0, 2, 1, 2});
    offer(6, 1.4 + std::ceil(pairs * (double)ceil_div(p.M, (int64_t)48) / cus) * (1.7 + 2.0 * per_wave), {0, 2, 1, 3});
    if (p.M <= 32) return best;
    const auto sum = [&](int64_t S, double us, double rate) { return S > 1 ? us + ((double)S * 8.0 + 2.0) * mn / rate : 0.0; };  // the second launch
    const int64_t rt = ceil_div(p.M, (int64_t)64), wgs = ceil_div(groups, (int64_t)2) * rt;
    const int64_t most = p.N % 4 == 0 ? std::min<int64_t>(ceil_div(chunks, (int64_t)4), 32) : 1;
    for (int64_t S = 1; S <= most; ++S) {
        if (fs > 0 && S != std::min<int64_t>(fs, most)) continue;
        const int64_t rounds = ceil_div(ceil_div(chunks, S), (int64_t)4);
        if (ceil_div(chunks, 4 * rounds) != S || (S > 1 && (uint64_t)(S * p.M) * (uint64_t)p.N * 4 > ctx->workspace_bytes)) continue;
        offer(4, std::ceil((double)(wgs * S) / cus) * (7.5 + (double)rounds * 2.45) + sum(S, 2.5, 4e6),
              {4, 1, (int)S});
    }
    offer(1, std::ceil((double)(ceil_div(groups, (int64_t)8) * rt) / cus) * (7.0 + (double)chunks * 2.1), {1, 1, 1});
    if (p.K < (1 << 22)) {  // 128 rows x 256 | 128 columns
        const int64_t rt128 = ceil_div(p.M, (int64_t)128), wgs128 = ceil_div(p.N, (int64_t)128) * rt128;
        offer(9, std::ceil((double)(ceil_div(p.N, (int64_t)256) * rt128) / cus) * (7.5 + (double)chunks * 1.6), {2, 1, 1, 1});
        const int64_t most2 = p.N % 4 == 0 ? std::min<int64_t>(ceil_div(chunks, (int64_t)2), 8) : 1;
        for (int64_t S = 1; S <= most2; ++S) {
            if (fs > 0 && S != std::min<int64_t>(fs, most2)) continue;
            const int64_t rounds = ceil_div(ceil_div(chunks, S), (int64_t)2);
            if (ceil_div(chunks, 2 * rounds) != S || (S > 1 && (uint64_t)(S * p.M) * (uint64_t)p.N * 4 > ctx->workspace_bytes)) continue;
            const double w = (double)(wgs128 * S) / cus;
            offer(10, 6.4 + std::ceil(w) * (1.2 + (double)rounds * 1.6) + w * (double)rounds * 0.36 + sum(S, 1.3, 4.3e6), {2, 1, (int)S, 2});
        }
    }
    if (p.K <= 2048) offer(8, 4.8 + 0.38 * (double)chunks + mn * 1.0e-6 + mn * (double)p.K * 3.5e-9, {-1, 1, 1});
    return best;
}

bool f8_direct_takes(const oxq_ctx *ctx, const F8Problem &p) { return f8_shape_ok(p) && f8_form(ctx, p).kind >= 0; }

template <int MT, int NS, int XQ, int NL>
static int f8_tile_launch(hipStream_t s, dim3 grid, const F8Problem &p) {
    static LdsGrant grant;
    constexpr auto kernel = f8_tile_kernel<MT, NS, 8, XQ, NL>;
    const size_t lds = (size_t)8 * (MT * 4096 + NS * 2048);
    OXQ_HIP_CHECK(grant.ensure((const void *)kernel, lds));
    hipLaunchKernelGGL(kernel, grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w, p.scales, (uint16_t *)p.y,
                       (int)p.M, (int)p.K, (int)p.N, (int)p.block_r, __builtin_ctzll((unsigned long long)p.block_c) - 7, (int)p.s_cols, (int)f8_s_rows(p));
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <int MT, int NS, int XQ>
static int f8_tile_go(hipStream_t s, dim3 grid, const F8Problem &p) {
    const int64_t most = ceil_div(p.K / 128, (int64_t)8);  // chunks a wave
    if (most <= 1) return f8_tile_launch<MT, NS, XQ, 1>(s, grid, p);
    if (most == 2) return f8_tile_launch<MT, NS, XQ, 2>(s, grid, p);
    if constexpr (NS == 1)
        if (most == 3) return f8_tile_launch<MT, NS, XQ, 3>(s, grid, p);
    return f8_tile_launch<MT, NS, XQ, 0>(s, grid, p);
}
template <int KS>
static int f8_gemm_go(hipStream_t s, dim3 grid, const F8Problem &p, float *part, int NG, int RT, int cslice) {
    static LdsGrant grant;
    const size_t lds = (size_t)2 * KS * 64 * 256 + 8 * 4096;
    OXQ_HIP_CHECK(grant.ensure((const void *)f8_gemm_kernel<4, KS>, lds));
    hipLaunchKernelGGL((f8_gemm_kernel<4, KS>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w, p.scales, (uint16_t *)p.y, part,
                       (int)p.M, (int)p.K, (int)p.N, NG, RT, cslice, (int)p.block_r, __builtin_ctzll((unsigned long long)p.block_c) - 7, (int)p.s_cols,
                       (int)f8_s_rows(p));
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

template <int KS>
static int f8_gemm128_go(hipStream_t s, dim3 grid, const F8Problem &p, float *part, int NG, int RT, int cslice) {
    static LdsGrant grant;
    const size_t lds = (size_t)2 * KS * 128 * 256 + 8 * 4096;
    OXQ_HIP_CHECK(grant.ensure((const void *)f8_gemm128_kernel<KS>, lds));
    hipLaunchKernelGGL((f8_gemm128_kernel<KS>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w, p.scales, (uint16_t *)p.y, part,
                       (int)p.M, (int)p.K, (int)p.N, NG, RT, cslice, (int)p.block_r, __builtin_ctzll((unsigned long long)p.block_c) - 7, (int)p.s_cols,
                       (int)f8_s_rows(p));
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

int launch_f8_direct(oxq_ctx *ctx, hipStream_t s, const F8Problem &p) {
    const F8Form form = f8_form(ctx, p);
    char name[64];
    if (form.kind == 0) {
        const int mt = form.mt ? form.mt : p.M > 16 ? 2 : 1;
        dim3 grid((unsigned)ceil_div(p.N, (int64_t)16 * form.ns), 1, (unsigned)ceil_div(p.M, (int64_t)16 * mt));
        if (grid.z > 65535) return fail(OXQ_ERR_UNSUPPORTED, "f8 matmul: m = %lld exceeds the grid", (long long)p.M);
        plan_name(name, sizeof name, "f8_mul_mm_bf16_mt%d%s", mt, form.ns == 4 ? "_n64" : form.ns == 2 ? "_n32" : "");
        set_plan(ctx, name, grid, dim3(512), 1, 1, 0);
        if (ctx->plan_only) return OXQ_OK;
        if (form.ns == 2) return mt == 3 ? f8_tile_go<3, 2, 12>(s, grid, p) : f8_tile_go<2, 2, 8>(s, grid, p);
        if (form.ns == 4) return mt == 3 ? f8_tile_go<3, 4, 12>(s, grid, p) : f8_tile_go<2, 4, 8>(s, grid, p);
        if (p.M > 16) return f8_tile_go<2, 1, 8>(s, grid, p);
        if (p.M > 8) return f8_tile_go<1, 1, 4>(s, grid, p);
        return p.M > 4 ? f8_tile_go<1, 1, 2>(s, grid, p) : f8_tile_go<1, 1, 1>(s, grid, p);
    }
    const bool tall = form.kind == 2;  // 128 rows, 32 columns a wave
    const int ks = tall ? form.mt : form.kind, spw = 8 / ks, rows = tall ? 128 : 64;
    const int64_t NG = ceil_div(ceil_div(p.N, (int64_t)(tall ? 32 : 64)), (int64_t)spw), RT = ceil_div(p.M, (int64_t)rows), chunks = p.K / 128;
    const int64_t wgs = ks == 1 ? pk4g_workgroups(RT, NG) : RT * NG;
    if (wgs > 0x7FFFFFFF) return fail(OXQ_ERR_UNSUPPORTED, "f8 matmul: m = %lld exceeds the grid", (long long)p.M);
    const int cslice = form.slices > 1 ? (int)(ceil_div(ceil_div(chunks, (int64_t)form.slices), (int64_t)ks) * ks) : (int)chunks;
    dim3 grid((unsigned)wgs, (unsigned)form.slices);
    plan_name(name, sizeof name, "f8_mul_mm_bf16_r%dx%d%s", rows, spw, ks == 4 ? "k4" : ks == 2 ? "k2" : "");
    set_plan(ctx, name, grid, dim3(512), form.slices, 1, form.slices > 1 ? (size_t)form.slices * p.M * p.N * 4 : 0);
    if (ctx->plan_only) {
        if (form.slices > 1) add_launch(ctx);
        return OXQ_OK;
    }
    float *part = (float *)ctx->workspace;
    const int rc = tall ? (ks == 2 ? f8_gemm128_go<2>(s, grid, p, part, (int)NG, (int)RT, cslice) : f8_gemm128_go<1>(s, grid, p, part, (int)NG, (int)RT, cslice))
                   : ks == 4 ? f8_gemm_go<4>(s, grid, p, part, (int)NG, (int)RT, cslice) : f8_gemm_go<1>(s, grid, p, part, (int)NG, (int)RT, cslice);
    if (rc != OXQ_OK || form.slices == 1) return rc;
    return launch_splitk_reduce(ctx, s, part, nullptr, p.y, p.M, p.N, form.slices, OXQ_BF16);
}

}  // namespace oxq
