// The checkpoint layouts (AWQ, quant_kernels.metal:3349-3499; GPTQ) at few rows of x on the matrix cores: up to 16, AWQ
// 4-bit in f16 up to 8 (from nine rows its tile kernel has the calls, though not by its time: 4096 x 4096 at 9 / 16 rows, tile kernel /
// this one, 10.5 / 8.7, 12.7 / 9.9 us, 4096 x 14336 13.9 / 12.6, 15.3 / 15.1, 8192 x 1024 11.3 / 8.9, 12.0 / 9.7).
//
// An AWQ word holds 8 (8-bit: 4) columns of one row of K.  A lane takes 16 columns - two (four) neighbouring words - of
// eight consecutive rows: nibble slot s of its words, row by row, is the B operand of one MFMA step for one column, and
// interleaving the 16-bit halves of two rows' words makes a pair of exact 16-bit floats one AND-OR away.  Sixteen lanes
// side by side read 128 (256) contiguous bytes of a row.  A GPTQ word is 8 (4) rows of one column, an operand as it lies
// once x is put in the order of its nibbles: a lane reads four columns of every 64.  A workgroup is 256 columns; its four
// waves take a quarter of its rows of K each, 128 or 64 at a time, and meet in LDS; the slices of K are added in slice
// order by a second launch.
//
// The weight is never rounded: bias and zero point come out through the row sums of x, the scale multiplies the group's
// f32 sum.  (Where a row is not finite, or so large that the biased products could overflow, the zero point leaves the
// integers instead: such sums have a sign.)
//
// What bounds it: the read of the weights plus a launch (the sum).  Every load of a wave's rows is requested before
// the first is waited for - 16 KB a wave, two workgroups a compute unit.  AWQ f16 4096 x 14336 at 4 rows, profiled: 9.0 us and
// 2.7 for the sum; vector issue is 3.3 of the 9.0 (12 instructions an MFMA), the waves wait 40 % of their time.
#include "oxq_device.hpp"
#include "oxq_internal.hpp"
#include "oxq_mfma.hpp"

#include <type_traits>

namespace oxq {

constexpr int SLAB_COLS = 256, SLAB_WAVES = 4;

// B operands hold bias + q: the bias.  It takes bits of the sums: 1024 beside four-bit codes in f16 left errors of small
// outputs three times those of weights multiplied one by one (1e-6 against 3e-7 of the sum of the terms' magnitudes at K =
// 4096), 64 leaves none to be seen; 128 in bf16 four to five times as many results that are not the nearest bf16 (9e-4 of them
// against 2e-4 at 4096 x 14336, 4 rows), 16 fewer (1e-4).  They cost a shift more a word (up to 2 %).  Without
// LOW two forms keep 1024 and 128, no further off than the kernels that took those calls before: f16 AWQ of more than one row (two
// shifts, 4096 x 14336, groups of 32, 13.3 -> 13.6 us), whose weights the tile kernel rounds, and bf16 GPTQ in runs of 128 (5120 x
// 13832, 2 rows, 16.4 -> 17.6 us), where the dot products left 6e-4.
template <typename TT, int BITS, bool GPTQ, bool LOW> __device__ __forceinline__ constexpr float slab_bias(int s) {
    if (TT::DTYPE != F16Traits::DTYPE) return BITS == 8 ? 0.f : GPTQ && !LOW ? 128.f : 16.f;
    return BITS == 8 ? 256.f : GPTQ || LOW || (s & 1) ? 64.f : 1024.f;
}
// bytes 0 and 2 of t, or 1 and 3
template <typename TT> __device__ __forceinline__ uint32_t slab_bytes(uint32_t t, bool high) {
    if constexpr (TT::DTYPE == F16Traits::DTYPE) return ((high ? t >> 6 : t << 2) & 0x03FC03FCu) | 0x5C005C00u;
    const float lo = high ? (float)((t >> 8) & 0xFFu) : (float)(t & 0xFFu), hi = high ? (float)(t >> 24) : (float)((t >> 16) & 0xFFu);
    return perm_b32(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);  // 8 bits: exact
}
// AWQ: slot `s` of a 16-bit half of the four row pairs t
template <typename TT, int BITS, bool LOW>
__device__ __forceinline__ void slab_awq_operand(const uint32_t (&t)[4], int s, const NibbleMasks &nm, uint32_t (&b)[4]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        if constexpr (BITS == 8) {
            b[p] = slab_bytes<TT>(t[p], s & 1);
        } else if constexpr (TT::DTYPE == F16Traits::DTYPE && LOW) {
            b[p] = ((s ? t[p] >> (4 * s - 4) : t[p] << 4) & nm.m1) | 0x54005400u;
        } else if constexpr (TT::DTYPE == F16Traits::DTYPE) {
            const uint32_t u = s < 2 ? t[p] : t[p] >> 8;
            b[p] = s & 1 ? (u & nm.m1) | 0x54005400u : (u & nm.m0) | 0x64006400u;
        } else {
            b[p] = ((s ? t[p] >> (4 * s - 3) : t[p] << 3) & nm.m0) | 0x41804180u;
        }
    }
}
// GPTQ: eight rows of one column, in the order that slab_gptq_x gives x
template <typename TT, int BITS, bool LOW> __device__ __forceinline__ void slab_gptq_operand(uint32_t w0, uint32_t w1, const NibbleMasks &nm, uint32_t (&b)[4]) {
    if constexpr (BITS == 8) {
        b[0] = slab_bytes<TT>(w0, false), b[1] = slab_bytes<TT>(w0, true), b[2] = slab_bytes<TT>(w1, false), b[3] = slab_bytes<TT>(w1, true);
    } else {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            if constexpr (TT::DTYPE == F16Traits::DTYPE) b[n] = ((n ? w0 >> (4 * n - 4) : w0 << 4) & nm.m1) | 0x54005400u;
            else if constexpr (LOW) b[n] = ((n ? w0 >> (4 * n - 3) : w0 << 3) & nm.m0) | 0x41804180u;
            else b[n] = ((w0 >> (4 * n)) & nm.m0) | 0x43004300u;
        }
    }
}
template <int BITS> __device__ __forceinline__ u32x4_t slab_gptq_x(u32x4_t d) {
    if constexpr (BITS == 4) return u32x4_t{pack_lo16(d[0], d[2]), pack_hi16(d[0], d[2]), pack_lo16(d[1], d[3]), pack_hi16(d[1], d[3])};
    return u32x4_t{pack_lo16(d[0], d[1]), pack_hi16(d[0], d[1]), pack_lo16(d[2], d[3]), pack_hi16(d[2], d[3])};
}

// STEPS: MFMA steps (32 rows of K) of a run, which a wave holds at once.  SETS: groups in it (1: a group is a run or more).
// SIGNS: infinite x give signed sums, and very large ones those of the weights themselves.  `blocks`: runs a wave takes.
template <typename TT, int BITS, bool GPTQ, int STEPS, int SETS, bool SIGNS, bool LOW>
__global__ __launch_bounds__(SLAB_WAVES * 64, 2) void wna16_slab_kernel(const uint16_t *__restrict__ x, const uint32_t *__restrict__ qw,
                                                                      const uint32_t *__restrict__ qz, const uint16_t *__restrict__ sc,
                                                                      const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                                      float *__restrict__ ws, int M, int K, int N, int gshift, int blocks) {
    typedef MfmaOps<TT> Ops;
    constexpr bool F16 = TT::DTYPE == F16Traits::DTYPE;
    constexpr int RUN = 32 * STEPS, ST = STEPS / SETS;  // rows of a run, steps of a group in it
    constexpr int W = BITS / 2, CPW = 32 / BITS;  // AWQ: words a lane reads of a row, columns of a word
    constexpr int OOB = 0x7FFFFF00;
    extern __shared__ __attribute__((aligned(16))) unsigned char slab_lds[];
    typedef uint32_t words_t __attribute__((ext_vector_type(GPTQ ? 4 : W)));
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int PW = N / CPW, G = (K + (1 << gshift) - 1) >> gshift;
    // The lane's 16 columns: AWQ c0 .. c0 + 15 (N % 8 == 0: 8 or 16 of them exist), GPTQ four of every 64, c0 + 64 j .. + 3
    const int c0 = (int)blockIdx.x * SLAB_COLS + (GPTQ ? 4 : 16) * ni;

    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(qw, 0u);
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(qw, (uint32_t)K * (uint32_t)PW * 4u);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(qz, (uint32_t)G * (uint32_t)PW * 4u);
    const __amdgpu_buffer_rsrc_t rs_s = make_rsrc(sc, (uint32_t)G * (uint32_t)N * 2u);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, (uint32_t)M * (uint32_t)K * 2u);
    constexpr int WR = GPTQ ? 8 / CPW : 8;  // rows of words that a lane reads a step
    auto exists = [&](int j) { return c0 + (GPTQ ? 64 * j : 0) < N; };
    auto vo_w = [&](int j) { return exists(j) ? GPTQ ? (kb * WR * N + c0 + 64 * j) * 4 : (kb * 8 * PW + c0 / CPW) * 4 : OOB; };
    auto vo_z = [&](int j) { return exists(j) ? (c0 + (GPTQ ? 64 * j : 0)) / CPW * 4 : OOB; };
    auto vo_s = [&](int j) { return exists(j) ? (c0 + (GPTQ ? 64 * j : 0)) * 2 : OOB; };
    const int vo_x = ni < M ? (ni * K + 8 * kb) * 2 : OOB;
    const NibbleMasks nm = F16 || (GPTQ && !LOW) ? nibble_masks() : NibbleMasks{vgpr_const(0x00780078u), 0u};

    float4_t acc[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] = float4_t{0.f, 0.f, 0.f, 0.f};

    const int b0 = ((int)blockIdx.y * SLAB_WAVES + wave) * blocks, b1 = min(b0 + blocks, (K + RUN - 1) / RUN);
    u32x4_t xa[STEPS];
    uint32_t w[STEPS][8 * W], zw[SETS][4], sv[SETS][8];  // words: AWQ [row][word], GPTQ [column][row]; scales in pairs of columns
    auto request = [&](int b) {
        const int k0 = b * RUN;
        // x, then the weights, then what the sums are scaled with; steps past K read zeros of x
#pragma unroll
        for (int st = 0; st < STEPS; ++st)
            xa[st] = __builtin_amdgcn_raw_buffer_load_b128(k0 + 32 * st < K ? rs_x : rs_none, vo_x, (k0 + 32 * st) * 2, 0);
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            const __amdgpu_buffer_rsrc_t rs = k0 + 32 * st < K ? rs_w : rs_none;
            if constexpr (GPTQ) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int r = 0; r < WR; ++r) {
                        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, vo_w(j), ((k0 + 32 * st) / CPW + r) * N * 4, 2);
#pragma unroll
                        for (int i = 0; i < 4; ++i) w[st][(4 * j + i) * WR + r] = v[i];
                    }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    words_t v;
                    if constexpr (W == 2) v = __builtin_bit_cast(words_t, __builtin_amdgcn_raw_buffer_load_b64(rs, vo_w(0), (k0 + 32 * st + j) * PW * 4, 2));
                    else v = __builtin_bit_cast(words_t, __builtin_amdgcn_raw_buffer_load_b128(rs, vo_w(0), (k0 + 32 * st + j) * PW * 4, 2));
#pragma unroll
                    for (int i = 0; i < W; ++i) w[st][j * W + i] = v[i];
                }
            }
        }
#pragma unroll
        for (int set = 0; set < SETS; ++set) {
            const int g = min((k0 + set * (32 * ST)) >> gshift, G - 1);
            if constexpr (GPTQ) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    zw[set][j] = __builtin_amdgcn_raw_buffer_load_b32(rs_z, vo_z(j), g * PW * 4, 0);
                    const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs_s, vo_s(j), g * N * 2, 0));
                    sv[set][2 * j] = v[0], sv[set][2 * j + 1] = v[1];
                }
            } else {
#pragma unroll
                for (int i = 0; i < W; ++i) zw[set][i] = __builtin_amdgcn_raw_buffer_load_b32(rs_z, vo_z(0) + 4 * i, g * PW * 4, 0);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs_s, vo_s(0) + 16 * i, g * N * 2, 0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) sv[set][4 * i + q] = v[q];
                }
            }
        }
    };
    auto multiply = [&] {
        if constexpr (GPTQ) {
#pragma unroll
            for (int st = 0; st < STEPS; ++st) xa[st] = slab_gptq_x<BITS>(xa[st]);
        } else {  // row pairs in place: [j] the low, [4 + j] the high halves of rows 2 j and 2 j + 1
#pragma unroll
            for (int st = 0; st < STEPS; ++st)
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    uint32_t t[8];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t r0 = w[st][2 * j * W + i], r1 = w[st][(2 * j + 1) * W + i];
                        t[j] = pack_lo16(r0, r1), t[4 + j] = pack_hi16(r0, r1);
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) w[st][j * W + i] = t[j];
                }
        }
#pragma unroll
        for (int set = 0; set < SETS; ++set) {
            float4_t rs = float4_t{0.f, 0.f, 0.f, 0.f};  // row sums of x, in the layout of the products
            float4_t sq = float4_t{0.f, 0.f, 0.f, 0.f};  // x times itself transposed: a row's squares on the diagonal
            {
                constexpr uint32_t ONE = F16 ? 0x3C003C00u : 0x3F803F80u;
                const uint32_t ones[4] = {ONE, ONE, ONE, ONE};
#pragma unroll
                for (int st = set * ST; st < set * ST + ST; ++st) {
                    const uint32_t a[4] = {xa[st][0], xa[st][1], xa[st][2], xa[st][3]};
                    rs = Ops::mfma(a, ones, rs);
                    if constexpr (SIGNS) sq = Ops::mfma(a, a, sq);
                }
            }
            // EXACT: the zero point leaves the integers instead of the sums, so that an infinite or very large x gives what it
            // gives where every weight is multiplied by itself.  In bf16 a group's sum of up to 2^15 |x| is kept down by as much
            // until the scale multiplies it.
            auto columns = [&](auto exact) {
                constexpr bool EXACT = decltype(exact)::value;
                constexpr float DOWN = 0x1p-15f;
#pragma unroll
                for (int c = 0; c < 16; ++c) {  // AWQ: slot s of word i; GPTQ: the lane's columns in order
                    const int i = c / CPW, s = c % CPW, HALF = CPW / 2;  // HALF: slots in a 16-bit half
                    const int col = GPTQ ? c : i * CPW + (BITS == 4 ? awq_slot_col(s) : s);
                    const uint32_t zero = GPTQ ? ((zw[set][c >> 2] >> (BITS * ((c0 + (c & 3)) % CPW))) & ((1u << BITS) - 1u)) + 1u
                                               : (zw[set][i] >> (BITS * s)) & ((1u << BITS) - 1u);
                    const float off = -(slab_bias<TT, BITS, GPTQ, LOW>(s % HALF) + (float)zero);
                    float4_t p = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int st = set * ST; st < set * ST + ST; ++st) {
                        const uint32_t a[4] = {xa[st][0], xa[st][1], xa[st][2], xa[st][3]};
                        uint32_t bq[4];
                        if constexpr (GPTQ) {
                            slab_gptq_operand<TT, BITS, LOW>(w[st][c * WR], w[st][c * WR + WR - 1], nm, bq);
                        } else {
                            uint32_t t[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) t[j] = w[st][((s / HALF) * 4 + j) * W + i];
                            slab_awq_operand<TT, BITS, LOW>(t, s % HALF, nm, bq);
                        }
                        if constexpr (EXACT) {  // integers of at most 9 bits, 256 the only one of 9: exact in either type
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                if constexpr (F16) {
                                    const half2_t off2 = {(_Float16)off, (_Float16)off};
                                    bq[j] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, bq[j]) + off2);
                                } else {
                                    const float lo = (__builtin_bit_cast(float, bq[j] << 16) + off) * DOWN, hi = (__builtin_bit_cast(float, bq[j] & 0xFFFF0000u) + off) * DOWN;
                                    bq[j] = perm_b32(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
                                }
                            }
                        }
                        p = Ops::mfma(a, bq, p);
                    }
                    const uint32_t sw = sv[set][col >> 1];
                    const float scale = TT::to_f32((uint16_t)(col & 1 ? sw >> 16 : sw)) * (EXACT && !F16 ? 1.0f / DOWN : 1.0f);
                    if constexpr (!EXACT) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) p[q] = __builtin_fmaf(off, rs[q], p[q]);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[col][q] = __builtin_fmaf(scale, p[q], acc[col][q]);
                }
            };
            if constexpr (SIGNS) {
                // Finite squares: no |x| beyond 2^64, so neither the biased products (at most 2^11 |x|) nor their sums overflow.
                // (The sum of four finite ones may overflow: the exact columns then, for nothing but time.)
                const float sum = (sq[0] + sq[1]) + (sq[2] + sq[3]);
                if (__builtin_expect(__any(!(fabsf(sum) <= 3.4e38f)), 0)) columns(std::true_type{});
                else columns(std::false_type{});
            } else {
                columns(std::false_type{});
            }
        }
    };
    for (int b = b0; b < b1; ++b) {
        request(b);
        __builtin_amdgcn_sched_barrier(0);
        multiply();
    }

    // lane (ni, kb): rows 4 kb + q of its 16 columns.  [wave][column][lane], lanes of rows that exist; wave k adds the
    // four waves' sums of columns 4 k .. 4 k + 3 in order of K.
    const int lanes = 16 * ((M + 3) >> 2);
    if (lane < lanes) {
#pragma unroll
        for (int c = 0; c < 16; ++c) *(float4_t *)(slab_lds + ((wave * 16 + c) * lanes + lane) * 16) = acc[c];
    }
    __syncthreads();
    const int n = c0 + (GPTQ ? 64 : 4) * wave;
    if (lane >= lanes || n >= N) return;
    float4_t sum[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        sum[c] = *(const float4_t *)(slab_lds + ((4 * wave + c) * lanes + lane) * 16);
#pragma unroll
        for (int k = 1; k < SLAB_WAVES; ++k) {
            const float4_t v = *(const float4_t *)(slab_lds + ((k * 16 + 4 * wave + c) * lanes + lane) * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[c][q] += v[q];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = 4 * kb + q;
        if (m >= M) break;
        if (gridDim.y > 1) {
            *(float4_t *)(ws + ((size_t)blockIdx.y * M + m) * N + n) = float4_t{sum[0][q], sum[1][q], sum[2][q], sum[3][q]};
        } else {
            uint32_t o[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float lo = sum[2 * c][q], hi = sum[2 * c + 1][q];
                if (bias) lo += TT::to_f32(bias[n + 2 * c]), hi += TT::to_f32(bias[n + 2 * c + 1]);
                o[c] = (uint32_t)TT::from_f32(lo) | ((uint32_t)TT::from_f32(hi) << 16);
            }
            *(uint2 *)(y + (size_t)m * N + n) = uint2{o[0], o[1]};
        }
    }
}

static int64_t slab_tiles(const Wna16Problem &p) {  // workgroups, at a run of 128 rows a wave
    return ceil_div(p.N, (int64_t)SLAB_COLS) * ceil_div(p.K, (int64_t)128 * SLAB_WAVES);
}

// us before (dot products; f16 4-bit: rows of 16 in 512-column tiles) and here, 4096 x 14336:
//   rows                     1             2             4             8
//   4-bit f16             11.3 / 11.8   15.0 / 12.0   15.6 / 12.4   16.0 / 13.4
//   4-bit bf16            12.2 / 11.8   18.2 / 12.2   21.5 / 12.7   33.7 / 13.6
//   4-bit bf16, group 32  26.2 / 14.8        -        51.4 / 15.3   80.7 / 16.0
//   8-bit f16             16.6 / 18.0   23.1 / 18.3   22.7 / 19.0   44.4 / 20.1
// One row: where there are few workgroups (4096 x 4096 f16 9.6 -> 7.8, 4096 x 8192, as many as compute units, 10.3 -> 9.3, 5120 x
// 8192 10.8 -> 11.5) or the alternative is the generic kernel.  The 512-column tiles stay for layers of so few columns
// that a launch's time is all there is (f16, 4 rows, 2048 x 1024 6.7 / 7.1), the generic AWQ kernel below 2^18 weights
// (8-bit from 9 rows: the copy in the workspace, below 2^20).
// GPTQ where gptq_tile.hip's rules exclude a layer (groups of 32 or 64 rows, K no multiple of 128, N none of 64), which then ran the
// generic kernel, or the dot products of groups of 128; 4-bit f16 / 8-bit bf16:
//   rows                           1                         4                         8                       16
//   6144 x 12864, group 32    85.0 / 16.3, 94.5 / 21.4   151 / 17.8, 200 / 22.1   229 / 18.2, 321 / 22.8   57.2 / 19.5, 638 / 24.8
//   4096 x 4096, group 64     10.9 / 7.8, 13.6 / 9.8    19.3 / 8.5, 26.7 / 10.5  28.9 / 9.2, 40.7 / 11.2  18.7 / 10.1, 25.8 / 12.4
//   5120 x 13832, group 128   14.5 / 15.2, 24.9 / 21.5  23.4 / 16.1, 30.8 / 22.4 35.8 / 16.8, 43.9 / 23.2 44.0 / 18.9, 87.2 / 25.4
// One row of groups of 128 stays with the dot products, one and two rows of less than 2^23 weights with the generic kernel
// (1408 x 1664 at one row 5.4 / 6.5, at four 7.6 / 7.0).
bool wna16_slab_takes(const oxq_ctx *ctx, const Wna16Problem &p) {
    const bool gptq = p.pack_dim == OXQ_PACK_IN;
    if ((p.bits != 4 && p.bits != 8) || p.M > (p.bits == 4 && !gptq && p.dtype == OXQ_F16 ? 8 : 16) || p.group_size < 32) return false;
    if (p.K % 32 != 0 || p.N % 8 != 0 || p.group_size % 32 != 0 || p.K * p.N < (p.M <= 8 ? 1 << 18 : 1 << 20)) return false;
    // 32-bit buffer offsets, a last run of rows past K included
    if ((uint64_t)(p.K + 128) * (uint64_t)(p.N * p.bits / 8) >= (1ull << 31)) return false;
    if ((uint64_t)p.M * (uint64_t)p.K * 2 >= (1ull << 30) || (uint64_t)(p.K / 32 + 1) * (uint64_t)p.N * 2 >= (1ull << 31)) return false;
    if (((uintptr_t)p.x | (uintptr_t)p.scales | (uintptr_t)p.y) & 15) return false;
    // a ctx told how the other kernels are to cut K or to add its slices gets those
    if (!tune(ctx, OXQ_TUNE_GEMV_TILE, 1) || tune(ctx, OXQ_TUNE_FORCE_GENERIC, 0) || tune(ctx, OXQ_TUNE_SPLITK_MODE, 0) ||
        tune(ctx, OXQ_TUNE_GEMV_GPW, 0) > 0 || tune(ctx, OXQ_TUNE_GEMV_CFG, -1) >= 0)
        return false;
    const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    if (gptq) {
        if (((uintptr_t)p.qweight & 15) || (gptq_tile_ok(p) && tune(ctx, OXQ_TUNE_GPTQ_TILE, 1))) return false;
        if (p.M == 1 && p.K % 128 == 0 && p.group_size >= 128) return false;
        return p.M >= 3 || p.K * p.N >= (1 << 23);
    }
    // (one row that the dot-product kernel refuses, ragged columns: 4096 x 8200 bf16 4-bit 21.9 -> 13.2 us, 8-bit 30.4 -> 15.3; groups of 64
    // and a short K stay with the generic kernel, 8-bit 960 x 4776 7.7 / 8.5, 320 x 6192 6.9 / 8.3, but 1088 x 3472 8.0 / 7.1)
    if (p.M == 1) return p.group_size < 64 || (!awq_fast_ok(p) && (p.group_size >= 128 || p.K >= 1024)) || (p.bits == 4 && slab_tiles(p) <= cus);
    return p.bits == 8 || p.dtype != OXQ_F16 || p.group_size < 128 || 2 * slab_tiles(p) >= 64;
}

template <typename TT, int BITS, bool GPTQ, int STEPS, int SETS, bool SIGNS = true, bool LOW = false>
static int slab_go(hipStream_t s, dim3 grid, const Wna16Problem &p, float *ws, int blocks) {
    const size_t lds = (size_t)SLAB_WAVES * 16 * 16 * ((p.M + 3) / 4) * 16;
    hipLaunchKernelGGL((wna16_slab_kernel<TT, BITS, GPTQ, STEPS, SETS, SIGNS, LOW>), grid, dim3(SLAB_WAVES * 64), lds, s, (const uint16_t *)p.x, p.qweight,
                       p.qzeros, (const uint16_t *)p.scales, (const uint16_t *)p.bias, (uint16_t *)p.y, ws, (int)p.M, (int)p.K,
                       (int)p.N, p.group_shift, blocks);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <typename TT, bool GPTQ>
static int slab_by_shape(hipStream_t s, dim3 grid, const Wna16Problem &p, float *ws, int blocks, int run) {
    // bf16 AWQ tensors that the dot-product kernel takes, as there: NaN for infinite x (the second path's registers cost 4 rows of
    // 4096 x 14336 12.7 -> 13.3 us).  Others (their address counts too) keep the signs that the generic kernel gives.
    if constexpr (TT::DTYPE != F16Traits::DTYPE && !GPTQ) {
        if (awq_fast_ok(p) && (p.M <= 8 || p.bits == 8))  // (more rows of 4 bits: the tile kernel's, which keeps the signs)
            return p.bits == 8 ? slab_go<TT, 8, GPTQ, 2, 1, false>(s, grid, p, ws, blocks)
                   : run == 64 ? slab_go<TT, 4, GPTQ, 2, 1, false>(s, grid, p, ws, blocks)
                               : slab_go<TT, 4, GPTQ, 4, 1, false>(s, grid, p, ws, blocks);
    }
    const bool g32 = p.group_size < 64;
    if constexpr (TT::DTYPE == F16Traits::DTYPE && !GPTQ) {
        if (p.bits == 4 && p.M == 1)  // more rows: the tile kernel's
            return g32        ? slab_go<TT, 4, GPTQ, 2, 2, true, true>(s, grid, p, ws, blocks)
                   : run == 64 ? slab_go<TT, 4, GPTQ, 2, 1, true, true>(s, grid, p, ws, blocks)
                               : slab_go<TT, 4, GPTQ, 4, 1, true, true>(s, grid, p, ws, blocks);
    }
    if (p.bits == 8) return g32 ? slab_go<TT, 8, GPTQ, 2, 2>(s, grid, p, ws, blocks) : slab_go<TT, 8, GPTQ, 2, 1>(s, grid, p, ws, blocks);
    if (run == 128) return slab_go<TT, 4, GPTQ, 4, 1>(s, grid, p, ws, blocks);
    return g32 ? slab_go<TT, 4, GPTQ, 2, 2, true, GPTQ>(s, grid, p, ws, blocks) : slab_go<TT, 4, GPTQ, 2, 1, true, GPTQ>(s, grid, p, ws, blocks);
}

int launch_wna16_slab(oxq_ctx *ctx, hipStream_t s, const Wna16Problem &p) {
    const int64_t tiles = ceil_div(p.N, (int64_t)SLAB_COLS), cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    // Runs of 64 registers of words; 4-bit layers whose workgroups come to five eighths of the compute units or less, half of
    // that (f16, 4 rows, 4096 x 4096 9.0 -> 8.3 us, 2 rows 1280 x 12736 9.4 -> 8.0; 4096 x 6144, six eighths, 9.1 -> 9.9).
    const int run = p.bits == 8 || p.group_size < 128 || slab_tiles(p) <= cus * 5 / 8 ? 64 : 128;
    const int64_t NB = ceil_div(p.K, (int64_t)run);
    // one run a wave while two workgroups a compute unit hold them all, else as many as bring that about (5120 x 13824, 1 row,
    // two runs, 14.6 us; half as long ones with the next requested meanwhile 17.5)
    int64_t blocks = std::max<int64_t>(1, ceil_div(tiles * ceil_div(NB, (int64_t)SLAB_WAVES), 2 * cus));
    while (ceil_div(NB, SLAB_WAVES * blocks) > 1 && (uint64_t)ceil_div(NB, SLAB_WAVES * blocks) * p.M * p.N * 4 > ctx->workspace_bytes) ++blocks;
    const int S = (int)ceil_div(NB, SLAB_WAVES * blocks);
    dim3 grid((unsigned)tiles, (unsigned)S);
    const uint64_t ws_bytes = S > 1 ? (uint64_t)S * p.M * p.N * 4 : 0;
    const bool f16 = p.dtype == OXQ_F16, gptq = p.pack_dim == OXQ_PACK_IN;
    char name[64];
    plan_name(name, sizeof name, "%s%d_gemv_fast_%s_m%d_slab%d%s", gptq ? "gptq" : "awq", p.bits, f16 ? "f16" : "bf16", (int)p.M, run,
             p.group_size >= 128 ? "" : p.group_size == 64 ? "_g64" : "_g32");
    set_plan(ctx, name, grid, dim3(SLAB_WAVES * 64), S, 1, ws_bytes);
    if (!ctx->plan_only) {
        float *ws = (float *)ctx->workspace;
        const int rc = gptq ? (f16 ? slab_by_shape<F16Traits, true>(s, grid, p, ws, (int)blocks, run) : slab_by_shape<BF16Traits, true>(s, grid, p, ws, (int)blocks, run))
                            : (f16 ? slab_by_shape<F16Traits, false>(s, grid, p, ws, (int)blocks, run) : slab_by_shape<BF16Traits, false>(s, grid, p, ws, (int)blocks, run));
        if (rc != OXQ_OK) return rc;
    }
    return S > 1 ? launch_splitk_reduce(ctx, s, (const float *)ctx->workspace, p.bias, p.y, p.M, p.N, S, p.dtype) : OXQ_OK;
}

}  // namespace oxq
