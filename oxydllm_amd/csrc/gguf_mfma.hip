// Resident GGUF layers for 16-bit activations: a copy of the blocks laid out for the matrix cores, and the
// matmul that reads it at any number of rows (linear.rs:197-284 GgufFastPath: forward_decode up to 8 rows,
// forward_prefill above; kernels quant_kernels.metal:792-870, 1097-1221 and the mul_mm strips).
//
// The rotated copy of gguf_res.hip gives a lane one unit of 32 elements and multiplies on the vector ALU: the
// work grows with every row of x.  Here a strip of 16 output columns and a unit of 32 elements of K are one
// v_mfma_f32_16x16x32_bf16 whose 16 rows are rows of x, so 1 to 16 rows cost the same instructions:
//
//   strip j (16 columns), chunk c (128 elements of K = 4 units), lane l = (ni = l % 16, kb = l / 16):
//   word t of the lane's quants = elements 8 kb .. 8 kb + 7 of unit 4 c + t of column 16 j + ni, which is the B
//   operand of the unit's MFMA once the integers are 16-bit floats; A = the same 8 elements of row ni of x.
//
//   Q4_0  chunk = [64 lanes][16 B] nibbles (element 2 pp in nibble pp, 2 pp + 1 in nibble pp + 4 of word t, so
//                 that one AND-OR per pair yields 128 + q as two bf16) + [16 columns][4 units] f16 d    1152 B
//   Q8_0  chunk = 2 x [64 lanes][16 B] (plane h = units 2 h, 2 h + 1; bytes of a word: elements 0, 2, 1, 3 of
//                 its four, stored as q + 128) + [16 columns][4 units] f16 d                             2176 B
//   Q4_1  as Q4_0, the unit headers are {d, m} pairs                                                     1280 B
//   Q5_0  as Q4_0 + [64 lanes][4 B] of fifth bits: the bit of element 2 pp (2 pp + 1) of unit t in bit
//         ggm_bit_at(t, pp) of the low (high) half: one shift puts a pair's bits at positions 4 and 20, or those of
//         pairs 0 and 2 (1 and 3) at bit 4 of the four bytes that hold their nibbles                        1408 B
//   Q5_1  as Q5_0 with {d, m} pairs                                                                      1536 B
//   Q5_K  as Q4_K with the plane of fifth bits in every chunk                                            2816 B
//   Q4_K  block = 2 chunks of [64 lanes][16 B] nibbles as Q4_0 + [16 columns] the super-block's first 16
//                 bytes (d, dmin, 12 scale bytes)                                                        2304 B
//   Q6_K  block = 2 chunks of { [64 lanes][16 B] low nibbles, [64 lanes][8 B] high bit pairs, [16 columns][8]
//                 int8 scales } + [16 columns] f16 d.  A scale covers 16 elements, so a step is a sub-block of 16
//                 and v_mfma_f32_16x16x16_bf16: step s of the chunk takes elements 16 s + 4 kb .. + 3; their
//                 nibbles sit in word s / 2 as Q4_0's pairs 2 (s % 2) and 2 (s % 2) + 1, their bit pairs in
//                 word s / 4 of the second plane, bit ggm_pair_at(2 (s % 4) + pair) of each 16-bit half   3360 B
//   Q2_K  block = 2 chunks of { [64 lanes][8 B] bit pairs, [16 columns][8] scale bytes } + [16 columns] {d, dmin}.  Steps as
//                 Q6_K's; pair p of steps 2 t and 2 t + 1 is field 2 (t % 2) + p of the bytes of word t / 2: bytes 0, 1 the
//                 step of 16 before, 2, 3 the one behind                                                  1344 B
//   Q3_K  block = 2 chunks of { [64 lanes][8 B] bit pairs as Q2_K, [64 lanes][4 B] third bits (bit 2 t + p of the same byte),
//                 [16 columns][8] int8 scales } + [16 columns] f16 d (the file packs its six-bit scales)     1824 B
//
// Exactly the file's bytes per weight (Q3_K: 114 for 110).  The integers stay integers: the MFMA accumulates x * (bias + q) in f32
// (products of 8-bit significands are exact), a second MFMA against the constant -(bias + offset) takes the
// bias and the format's offset out in the same accumulator, and the unit's scale multiplies the sum once per
// output, in f32, as the reference's GEMV does (d * sum of q * x, quant_kernels.metal:1097-1221).
//
// A workgroup is one strip; its 16 (8) waves split the strip's chunks and stage their own rows of x through
// LDS (no barrier before the epilogue); the partial tiles meet in LDS in wave order.
#include "gguf_decode.hpp"
#include "pk4_common.hpp"

namespace oxq {

template <int FMT> struct GgmFmt;
// WQ: 16-byte quant planes a chunk; CH: chunks a block; UH: bytes of unit headers a chunk and column;
// BH: bytes of block header a column; NEG: the constant that takes bias and offset out (as a bf16 pair)
template <> struct GgmFmt<OXQ_GGUF_Q4_0> { static constexpr int WQ = 1, CH = 1, UH = 8, BH = 0; static constexpr uint32_t NEG = 0xC308C308u; };  // -136
template <> struct GgmFmt<OXQ_GGUF_Q8_0> { static constexpr int WQ = 2, CH = 1, UH = 8, BH = 0; static constexpr uint32_t NEG = 0xC300C300u; };  // -128
template <> struct GgmFmt<OXQ_GGUF_Q4_1> { static constexpr int WQ = 1, CH = 1, UH = 16, BH = 0; static constexpr uint32_t NEG = 0xC300C300u; };  // -128
template <> struct GgmFmt<OXQ_GGUF_Q5_0> { static constexpr int WQ = 1, CH = 1, UH = 8, BH = 0; static constexpr uint32_t NEG = 0xC310C310u; };  // -144
template <> struct GgmFmt<OXQ_GGUF_Q5_1> { static constexpr int WQ = 1, CH = 1, UH = 16, BH = 0; static constexpr uint32_t NEG = 0xC300C300u; };  // -128
template <> struct GgmFmt<OXQ_GGUF_Q5_K> { static constexpr int WQ = 1, CH = 2, UH = 0, BH = 16; static constexpr uint32_t NEG = 0xC300C300u; };  // -128
template <> struct GgmFmt<OXQ_GGUF_Q4_K> { static constexpr int WQ = 1, CH = 2, UH = 0, BH = 16; static constexpr uint32_t NEG = 0xC300C300u; };  // -128
template <> struct GgmFmt<OXQ_GGUF_Q6_K> { static constexpr int WQ = 1, CH = 2, UH = 8, BH = 2; static constexpr uint32_t NEG = 0xC320C320u; };  // -160
template <> struct GgmFmt<OXQ_GGUF_Q2_K> { static constexpr int WQ = 0, CH = 2, UH = 8, BH = 4; static constexpr uint32_t NEG = 0x3F803F80u; };  // 1: no bias
template <> struct GgmFmt<OXQ_GGUF_Q3_K> { static constexpr int WQ = 0, CH = 2, UH = 8, BH = 2; static constexpr uint32_t NEG = 0x3F803F80u; };

// formats of two and three bits: 16-element scales as Q6_K, no plane of nibbles
template <int FMT> constexpr bool ggm_narrow = FMT == OXQ_GGUF_Q2_K || FMT == OXQ_GGUF_Q3_K;
template <int FMT> constexpr bool ggm_k16 = FMT == OXQ_GGUF_Q6_K || ggm_narrow<FMT>;  // a scale covers 16 elements
// formats with a fifth bit; with a term that multiplies the sum of x: a minimum beside the scale, or Q3_K's offset
template <int FMT> constexpr bool ggm_fifth_bit = FMT == OXQ_GGUF_Q5_0 || FMT == OXQ_GGUF_Q5_1 || FMT == OXQ_GGUF_Q5_K;
template <int FMT> constexpr bool ggm_has_min = FMT == OXQ_GGUF_Q4_K || FMT == OXQ_GGUF_Q5_K || FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q5_1 || ggm_narrow<FMT>;

// Place in its 16-bit half of the fifth bit of pair pp of unit t, and of the bit pair of field f (Q6_K): pairs 0, 1 of a unit in the
// low byte, 2, 3 in the high one.
__device__ constexpr int ggm_bit_at(int t, int pp) { return 2 * t + (pp & 1) + 8 * (pp >> 1); }
__device__ constexpr int ggm_pair_at(int f) { return 2 * (2 * (f >> 2) + (f & 1)) + 8 * ((f >> 1) & 1); }

template <int FMT> struct GgmLayout {
    typedef GgmFmt<FMT> F;
    static constexpr int H_OFF = F::WQ * 1024;                                  // Q6_K: the plane of bit pairs; fifth bits
    static constexpr int UH_OFF = F::WQ * 1024 + (ggm_k16<FMT> ? 512 : 0) + (ggm_fifth_bit<FMT> || FMT == OXQ_GGUF_Q3_K ? 256 : 0);
    static constexpr int CHB = UH_OFF + 16 * F::UH;
    static constexpr int BH_OFF = F::CH * CHB;
    static constexpr int BLKB = F::CH * CHB + 16 * F::BH;
    static_assert(BLKB == 16 * (128 * F::CH / GgufFmt<FMT>::BE) * (GgufFmt<FMT>::BB + (FMT == OXQ_GGUF_Q3_K ? 4 : 0)), "the copy has the file's size");
};

// ---------------------------------------------------------------------------
// repack: one thread per (strip, chunk, lane)
// ---------------------------------------------------------------------------
// Resident column -> row of the file.  A fused gate|up layer (half = N / 2 gate rows followed by as many up rows)
// keeps, in every strip of 16, 8 gate columns followed by the 8 up columns they are multiplied with, so that one
// workgroup holds both factors of its outputs.
__device__ __forceinline__ int ggm_src_row(int c, int half) {
    if (!half) return c;
    const int j = c >> 4, cc = c & 15;
    return cc < 8 ? 8 * j + cc : half + 8 * j + (cc - 8);
}

template <int FMT>
__global__ __launch_bounds__(256) void ggm_repack_kernel(const uint8_t *__restrict__ w, uint8_t *__restrict__ pw, int K,
                                                         int N, int half) {
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    const int nch = K >> 7;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)((N + 15) >> 4) * nch * 64) return;
    const int lane = (int)(idx & 63), c = (int)((idx >> 6) % nch), strip = (int)((idx >> 6) / nch);
    const int ni = lane & 15, kb = lane >> 4;
    if (16 * strip + ni >= N) {  // the last strip of a layer whose rows end inside it: zero weights, zero scales
        uint8_t *zb = pw + ((size_t)strip * (nch / F::CH) + c / F::CH) * L::BLKB, *zc = zb + (c % F::CH) * L::CHB;
#pragma unroll
        for (int pl = 0; pl < F::WQ; ++pl) *(u32x4_t *)(zc + pl * 1024 + lane * 16) = u32x4_t{0u, 0u, 0u, 0u};
        if constexpr (ggm_k16<FMT>) *(uint2 *)(zc + L::H_OFF + lane * 8) = uint2{0u, 0u};
        if constexpr (FMT == OXQ_GGUF_Q3_K) *(uint32_t *)(zc + 512 + lane * 4) = 0u;
        if constexpr (ggm_fifth_bit<FMT>) *(uint32_t *)(zc + L::H_OFF + lane * 4) = 0u;
        for (int b = kb; b < F::UH; b += 4) zc[L::UH_OFF + ni * F::UH + b] = 0;
        if (c % F::CH == 0)
            for (int b = kb; b < F::BH; b += 4) zb[L::BH_OFF + ni * F::BH + b] = 0;
        return;
    }
    const size_t row_bytes = (size_t)(K / GgufFmt<FMT>::BE) * GgufFmt<FMT>::BB;
    const uint8_t *row = w + (size_t)ggm_src_row(16 * strip + ni, half) * row_bytes;
    uint8_t *blk = pw + ((size_t)strip * (nch / F::CH) + c / F::CH) * L::BLKB;
    uint8_t *chunk = blk + (c % F::CH) * L::CHB;
    if constexpr (FMT == OXQ_GGUF_Q4_0) {
        uint32_t q[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint8_t *p = row + (size_t)(4 * c + t) * 18;
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int e = 8 * kb + i;  // element e of the unit: low nibble of byte e (e < 16), high of byte e - 16
                const uint32_t nib = e < 16 ? (p[2 + e] & 0xFu) : (p[2 + e - 16] >> 4);
                v |= nib << (4 * (i >> 1) + 16 * (i & 1));
            }
            q[t] = v;
            if (t == kb) *(uint16_t *)(chunk + L::UH_OFF + ni * 8 + t * 2) = ld16(p);
        }
        *(u32x4_t *)(chunk + lane * 16) = u32x4_t{q[0], q[1], q[2], q[3]};
    } else if constexpr (FMT == OXQ_GGUF_Q8_0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t q[4];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const int t = 2 * h + tt;
                const uint8_t *p = row + (size_t)(4 * c + t) * 34;
#pragma unroll
                for (int d = 0; d < 2; ++d) {  // word d of the step: elements 4 d .. 4 d + 3 of the lane's 8
                    const uint8_t *e = p + 2 + 8 * kb + 4 * d;
                    q[2 * tt + d] = ((uint32_t)(e[0] ^ 0x80u)) | ((uint32_t)(e[2] ^ 0x80u) << 8) |
                                    ((uint32_t)(e[1] ^ 0x80u) << 16) | ((uint32_t)(e[3] ^ 0x80u) << 24);
                }
                if (t == kb) *(uint16_t *)(chunk + L::UH_OFF + ni * 8 + t * 2) = ld16(p);
            }
            *(u32x4_t *)(chunk + h * 1024 + lane * 16) = u32x4_t{q[0], q[1], q[2], q[3]};
        }
    } else if constexpr (FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q5_0 || FMT == OXQ_GGUF_Q5_1) {
        // quant_kernels.metal:709-790, 872-1036: {d (, m)} (, 32 fifth bits), 16 bytes of nibbles as Q4_0
        constexpr bool MIN = FMT != OXQ_GGUF_Q5_0, FIFTH = FMT != OXQ_GGUF_Q4_1;
        constexpr int BB = GgufFmt<FMT>::BB, QS = (MIN ? 4 : 2) + (FIFTH ? 4 : 0);
        uint32_t q[4], hb = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint8_t *p = row + (size_t)(4 * c + t) * BB;
            const uint32_t qh = FIFTH ? (ld16(p + QS - 4) | (ld16(p + QS - 2) << 16)) : 0u;
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int e = 8 * kb + i;
                const uint32_t nib = e < 16 ? (p[QS + e] & 0xFu) : (p[QS + e - 16] >> 4);
                v |= nib << (4 * (i >> 1) + 16 * (i & 1));
                hb |= ((qh >> e) & 1u) << (ggm_bit_at(t, i >> 1) + 16 * (i & 1));
            }
            q[t] = v;
            if (t == kb) {
                if constexpr (MIN) *(uint32_t *)(chunk + L::UH_OFF + ni * 16 + t * 4) = ld16(p) | (ld16(p + 2) << 16);
                else *(uint16_t *)(chunk + L::UH_OFF + ni * 8 + t * 2) = ld16(p);
            }
        }
        *(u32x4_t *)(chunk + lane * 16) = u32x4_t{q[0], q[1], q[2], q[3]};
        if constexpr (FIFTH) *(uint32_t *)(chunk + L::H_OFF + lane * 4) = hb;
    } else if constexpr (FMT == OXQ_GGUF_Q4_K || FMT == OXQ_GGUF_Q5_K) {
        // quant_kernels.metal:2438-2482: sub-block sb of the super-block reads byte (sb / 2) * 32 + e of qs, low
        // nibble if sb is even; Q5_K (1438-1680): its fifth bit is bit sb of byte e of qh
        constexpr bool FIFTH = FMT == OXQ_GGUF_Q5_K;
        const uint8_t *p = row + (size_t)(c >> 1) * GgufFmt<FMT>::BB;
        const uint8_t *qs = p + (FIFTH ? 48 : 16);
        uint32_t q[4], hb = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int sb = 4 * (c & 1) + t;
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t byte = qs[(sb >> 1) * 32 + 8 * kb + i];
                v |= ((sb & 1) ? (byte >> 4) : (byte & 0xFu)) << (4 * (i >> 1) + 16 * (i & 1));
                if constexpr (FIFTH) hb |= (((uint32_t)p[16 + 8 * kb + i] >> sb) & 1u) << (ggm_bit_at(t, i >> 1) + 16 * (i & 1));
            }
            q[t] = v;
        }
        *(u32x4_t *)(chunk + lane * 16) = u32x4_t{q[0], q[1], q[2], q[3]};
        if constexpr (FIFTH) *(uint32_t *)(chunk + L::H_OFF + lane * 4) = hb;
        if ((c & 1) == 0 && kb < 4) *(uint32_t *)(blk + L::BH_OFF + ni * 16 + kb * 4) = ld32a2(p + 4 * kb);
    } else if constexpr (FMT == OXQ_GGUF_Q6_K) {
        // quant_kernels.metal:2518-2554: element j of the super-block, h = j / 128, q = (j % 128) / 32, l = j % 32:
        // low nibble from ql[64 h + (q & 1) * 32 + l] (high nibble of the byte if q >= 2), bit pair 2 q of qh[32 h + l]
        const uint8_t *p = row + (size_t)(c >> 1) * 210;
        const int h = c & 1;
        uint32_t lw[4] = {0u, 0u, 0u, 0u}, hw[2] = {0u, 0u};
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int jj = 16 * s2 + 4 * kb + i;  // element of this half of the super-block
                const int qq = jj >> 5, l = jj & 31;
                const uint32_t lb = p[64 * h + (qq & 1) * 32 + l];
                const uint32_t lo = qq < 2 ? (lb & 0xFu) : (lb >> 4);
                const uint32_t hi = (p[128 + 32 * h + l] >> (2 * qq)) & 3u;
                const int pair = i >> 1, half = i & 1;
                lw[s2 >> 1] |= lo << (4 * (2 * (s2 & 1) + pair) + 16 * half);
                hw[s2 >> 2] |= hi << (ggm_pair_at(2 * (s2 & 3) + pair) + 16 * half);
            }
        *(u32x4_t *)(chunk + lane * 16) = u32x4_t{lw[0], lw[1], lw[2], lw[3]};
        *(uint2 *)(chunk + L::H_OFF + lane * 8) = uint2{hw[0], hw[1]};
        if (kb < 2) *(uint32_t *)(chunk + L::UH_OFF + ni * 8 + kb * 4) = ld32a2(p + 192 + 8 * h + 4 * kb);
        if (h == 0 && kb == 0) *(uint16_t *)(blk + L::BH_OFF + ni * 2) = ld16(p + 208);
    } else if constexpr (ggm_narrow<FMT>) {
        // quant_kernels.metal:2556-2680: element j of the super-block, h = j / 128, q = (j % 128) / 32, l = j % 32: bit pair
        // 2 q of qs[32 h + l]; Q3_K's third bit is bit 4 h + q of hmask[l]
        constexpr bool THREE = FMT == OXQ_GGUF_Q3_K;
        const uint8_t *p = row + (size_t)(c >> 1) * GgufFmt<FMT>::BB;
        const int h = c & 1;
        const uint8_t *qs = p + (THREE ? 32 : 16) + 32 * h;
        uint32_t w2[2] = {0u, 0u}, w3 = 0u;
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int jj = 16 * s2 + 4 * kb + i, qq = jj >> 5, l = jj & 31;
                const int t = s2 >> 1, pr = i >> 1, byte = 2 * (s2 & 1) + (i & 1);
                w2[t >> 1] |= (((uint32_t)qs[l] >> (2 * qq)) & 3u) << (8 * byte + 4 * (t & 1) + 2 * pr);
                if constexpr (THREE) w3 |= (((uint32_t)p[l] >> (4 * h + qq)) & 1u) << (8 * byte + 2 * t + pr);
            }
        *(uint2 *)(chunk + lane * 8) = uint2{w2[0], w2[1]};
        if constexpr (THREE) *(uint32_t *)(chunk + 512 + lane * 4) = w3;
        // two scales of the chunk's eight a lane group
#pragma unroll
        for (int b = 2 * kb; b < 2 * kb + 2; ++b)
            chunk[L::UH_OFF + ni * 8 + b] = THREE ? (uint8_t)(int8_t)q3k_scale(p + 96, 8 * h + b) : p[8 * h + b];
        if (h == 0 && kb == 0) {
            if constexpr (THREE) *(uint16_t *)(blk + L::BH_OFF + ni * 2) = ld16(p + 108);
            else *(uint32_t *)(blk + L::BH_OFF + ni * 4) = ld16(p + 80) | (ld16(p + 82) << 16);
        }
    }
}

// dense [N, K] f32 from the copy, with the arithmetic of the file-layout dequant (pins the repack bit for bit)
template <int FMT>
__global__ __launch_bounds__(256) void ggm_dequant_kernel(const uint8_t *__restrict__ pw, float *__restrict__ out, int K,
                                                          int N, int half) {
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    const int nch = K >> 7;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)((N + 15) >> 4) * nch * 64) return;
    const int lane = (int)(idx & 63), c = (int)((idx >> 6) % nch), strip = (int)((idx >> 6) / nch);
    const int ni = lane & 15, kb = lane >> 4;
    if (16 * strip + ni >= N) return;
    const uint8_t *blk = pw + ((size_t)strip * (nch / F::CH) + c / F::CH) * L::BLKB;
    const uint8_t *chunk = blk + (c % F::CH) * L::CHB;
    const size_t orow = (size_t)ggm_src_row(16 * strip + ni, half);
    float *o = out + orow * K + (size_t)c * 128 + 8 * kb;
    if constexpr (FMT == OXQ_GGUF_Q4_0) {
        const u32x4_t q = *(const u32x4_t *)(chunk + lane * 16);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float d = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)(chunk + L::UH_OFF + ni * 8 + t * 2));
#pragma unroll
            for (int i = 0; i < 8; ++i)
                o[32 * t + i] = (float)((int)((q[t] >> (4 * (i >> 1) + 16 * (i & 1))) & 0xFu) - 8) * d;
        }
    } else if constexpr (FMT == OXQ_GGUF_Q8_0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const u32x4_t q = *(const u32x4_t *)(chunk + h * 1024 + lane * 16);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const int t = 2 * h + tt;
                const float d = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)(chunk + L::UH_OFF + ni * 8 + t * 2));
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int byte = ((i & 3) >> 1) | ((i & 1) << 1);  // elements 0, 2, 1, 3 in bytes 0 .. 3
                    o[32 * t + i] = (float)((int)((q[2 * tt + (i >> 2)] >> (8 * byte)) & 0xFFu) - 128) * d;
                }
            }
        }
    } else if constexpr (FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q5_0 || FMT == OXQ_GGUF_Q5_1) {
        constexpr bool MIN = FMT != OXQ_GGUF_Q5_0, FIFTH = FMT != OXQ_GGUF_Q4_1;
        const u32x4_t q = *(const u32x4_t *)(chunk + lane * 16);
        const uint32_t hb = FIFTH ? *(const uint32_t *)(chunk + L::H_OFF + lane * 4) : 0u;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint8_t *uh = chunk + L::UH_OFF + ni * (MIN ? 16 : 8) + t * (MIN ? 4 : 2);
            const float d = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)uh);
            const float m = MIN ? (float)__builtin_bit_cast(_Float16, *(const uint16_t *)(uh + 2)) : 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t v = ((q[t] >> (4 * (i >> 1) + 16 * (i & 1))) & 0xFu) |
                                   (((hb >> (ggm_bit_at(t, i >> 1) + 16 * (i & 1))) & 1u) << 4);
                o[32 * t + i] = MIN ? (float)v * d + m : (float)((int)v - 16) * d;
            }
        }
    } else if constexpr (FMT == OXQ_GGUF_Q4_K || FMT == OXQ_GGUF_Q5_K) {
        const u32x4_t q = *(const u32x4_t *)(chunk + lane * 16);
        const uint32_t hb = FMT == OXQ_GGUF_Q5_K ? *(const uint32_t *)(chunk + L::H_OFF + lane * 4) : 0u;
        const uint8_t *hd = blk + L::BH_OFF + ni * 16;
        const float d = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)hd);
        const float dmin = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)(hd + 2));
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t scv, mnv;
            k4_scale_min(hd + 4, 4 * (c & 1) + t, scv, mnv);
            const float d1 = d * (float)scv, m1 = dmin * (float)mnv;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                o[32 * t + i] = d1 * (float)(((q[t] >> (4 * (i >> 1) + 16 * (i & 1))) & 0xFu) |
                                             (((hb >> (ggm_bit_at(t, i >> 1) + 16 * (i & 1))) & 1u) << 4)) - m1;
        }
    } else if constexpr (FMT == OXQ_GGUF_Q6_K) {
        const u32x4_t lw = *(const u32x4_t *)(chunk + lane * 16);
        const uint2 hw = *(const uint2 *)(chunk + L::H_OFF + lane * 8);
        const float d = (float)__builtin_bit_cast(_Float16, *(const uint16_t *)(blk + L::BH_OFF + ni * 2));
        float *o6 = out + orow * K + (size_t)c * 128 + 4 * kb;
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2) {
            const float ds = d * (float)(int)*(const int8_t *)(chunk + L::UH_OFF + ni * 8 + s2);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int pair = i >> 1, half = i & 1;
                const uint32_t lo = (lw[s2 >> 1] >> (4 * (2 * (s2 & 1) + pair) + 16 * half)) & 0xFu;
                const uint32_t hi = ((s2 < 4 ? hw.x : hw.y) >> (ggm_pair_at(2 * (s2 & 3) + pair) + 16 * half)) & 3u;
                o6[16 * s2 + i] = ds * (float)((int)(lo | (hi << 4)) - 32);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// the matmul
// ---------------------------------------------------------------------------
// bytes 0 and 2 (1 and 3) of a word as a pair of bf16: through f32, exact for 0 .. 255
__device__ __forceinline__ uint32_t ggm_bytes02(uint32_t w) {
    const float lo = (float)(w & 0xFFu), hi = (float)((w >> 16) & 0xFFu);
    return pack_hi16(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}
__device__ __forceinline__ uint32_t ggm_bytes13(uint32_t w) {
    const float lo = (float)((w >> 8) & 0xFFu), hi = (float)(w >> 24);
    return pack_hi16(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float ggm_f16(uint32_t bits) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits); }

// The registers of one chunk: its quants and headers as requested, and what turns them into MFMA operands and
// the factors of a step.  A step's sum t = sum over the step's elements of x * q', q' = q minus the format's
// offset (exact integers); y += f0(step) * t + f1(step) * (sum of x) where the format has a minimum.
template <int FMT> struct GgmChunk {
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    static constexpr int NSTEP = ggm_k16<FMT> ? 8 : 4;
    static constexpr bool HAS_MIN = ggm_has_min<FMT>;
    // vector loads of one request()
    static constexpr int LOADS = (F::UH ? 1 : 0) + (F::BH ? 1 : 0) + F::WQ + ((ggm_k16<FMT> || ggm_fifth_bit<FMT>) ? 1 : 0) + (FMT == OXQ_GGUF_Q3_K ? 1 : 0);
    u32x4_t q[F::WQ ? F::WQ : 1];
    uint32_t qh[FMT == OXQ_GGUF_Q3_K ? 3 : ggm_k16<FMT> ? 2 : 1];  // Q2_K, Q3_K: two words of bit pairs, one of third bits
    uint32_t uh[F::UH == 16 ? 4 : F::UH ? 2 : 1];   // unit headers of the column: four f16 d or {d, m} pairs, eight int8 scales (Q6_K)
    uint32_t bh[F::BH == 16 ? 4 : 1];  // block header of the column

    // c: the chunk's index in its strip
    template <typename RS>
    __device__ __forceinline__ void request(const RS &rs, int lane, int ni, int c, int strip_off) {
        const int blk = strip_off + (c / F::CH) * L::BLKB, soff = blk + (c % F::CH) * L::CHB;
        // headers first: the factors and the minimum's term are worked out while the quants are on their way
        if constexpr (F::UH == 8) {
            const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rs, ni * 8, soff + L::UH_OFF, 2);
            uh[0] = v[0], uh[1] = v[1];
        } else if constexpr (F::UH == 16) {
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, ni * 16, soff + L::UH_OFF, 2);
            uh[0] = v[0], uh[1] = v[1], uh[2] = v[2], uh[3] = v[3];
        }
        if constexpr (F::BH == 16) {
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, ni * 16, blk + L::BH_OFF, 0);
            bh[0] = v[0], bh[1] = v[1], bh[2] = v[2], bh[3] = v[3];
        } else if constexpr (F::BH == 2) {
            bh[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (ni >> 1) * 4, blk + L::BH_OFF, 0);
        } else if constexpr (F::BH == 4) {
            bh[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, ni * 4, blk + L::BH_OFF, 0);
        }
#pragma unroll
        for (int pl = 0; pl < F::WQ; ++pl) q[pl] = __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, soff + pl * 1024, 2);
        if constexpr (ggm_k16<FMT>) {
            const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rs, lane * 8, soff + L::H_OFF, 2);
            qh[0] = v[0], qh[1] = v[1];
            if constexpr (FMT == OXQ_GGUF_Q3_K) qh[2] = __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4, soff + 512, 2);
        } else if constexpr (ggm_fifth_bit<FMT>) {
            qh[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4, soff + L::H_OFF, 2);
        }
    }
    // The factors of the chunk's steps, once per chunk when its registers have arrived; half = c % 2 (wave-uniform).
    // f0[st] multiplies the step's sum, f1[st] (formats with a minimum) the bias term -128 sum(x).
    __device__ __forceinline__ void factors(int half, int ni, float (&f0)[NSTEP], float (&f1)[NSTEP]) const {
        if constexpr (FMT == OXQ_GGUF_Q4_K || FMT == OXQ_GGUF_Q5_K) {
            // get_scale_min_k4 (quant_kernels.metal:2438-2450) for the chunk's four sub-blocks at once, a byte each
            // (selected by mask: as a branch on the chunk's parity the two sides kept twice the registers alive)
            const uint32_t hm = half ? 0xFFFFFFFFu : 0u;
            const uint32_t sc4 = (((bh[3] & 0x0F0F0F0Fu) | ((bh[1] >> 2) & 0x30303030u)) & hm) | (bh[1] & 0x3F3F3F3Fu & ~hm);
            const uint32_t mn4 = ((((bh[3] >> 4) & 0x0F0F0F0Fu) | ((bh[2] >> 2) & 0x30303030u)) & hm) | (bh[2] & 0x3F3F3F3Fu & ~hm);
            const float d = ggm_f16(bh[0] & 0xFFFFu), dm = ggm_f16(bh[0] >> 16) * 0.0078125f;  // dmin / 128
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f0[t] = d * (float)((sc4 >> (8 * t)) & 0xFFu);
                f1[t] = dm * (float)((mn4 >> (8 * t)) & 0xFFu);
            }
        } else if constexpr (FMT == OXQ_GGUF_Q6_K) {
            const float d = ggm_f16((ni & 1) ? (bh[0] >> 16) : (bh[0] & 0xFFFFu));
#pragma unroll
            for (int st = 0; st < 8; ++st) f0[st] = d * (float)(int)(int8_t)((uh[st >> 2] >> (8 * (st & 3))) & 0xFFu), f1[st] = 0.f;
        } else if constexpr (FMT == OXQ_GGUF_Q3_K) {  // w = f0 (q + 4) - 4 f0
            const float d = ggm_f16((ni & 1) ? (bh[0] >> 16) : (bh[0] & 0xFFFFu));
#pragma unroll
            for (int st = 0; st < 8; ++st) f0[st] = d * (float)(int)(int8_t)((uh[st >> 2] >> (8 * (st & 3))) & 0xFFu), f1[st] = f0[st] * 0.03125f;
        } else if constexpr (FMT == OXQ_GGUF_Q2_K) {
            const float d = ggm_f16(bh[0] & 0xFFFFu), dm = ggm_f16(bh[0] >> 16) * 0.0078125f;  // dmin / 128
#pragma unroll
            for (int st = 0; st < 8; ++st) {
                f0[st] = d * (float)((uh[st >> 2] >> (8 * (st & 3))) & 0xFu);
                f1[st] = dm * (float)((uh[st >> 2] >> (8 * (st & 3) + 4)) & 0xFu);
            }
        } else if constexpr (F::UH == 16) {  // w = d q + m: the minimum times sum(x) = -m / 128 times the bias term
#pragma unroll
            for (int st = 0; st < 4; ++st) f0[st] = ggm_f16(uh[st] & 0xFFFFu), f1[st] = ggm_f16(uh[st] >> 16) * -0.0078125f;
        } else {
#pragma unroll
            for (int st = 0; st < 4; ++st) f0[st] = ggm_f16((st & 1) ? (uh[st >> 1] >> 16) : (uh[st >> 1] & 0xFFFFu)), f1[st] = 0.f;
        }
    }
    // The five- and six-bit integers of 32 elements, a byte each: bytes 0, 2 of lo, hi pairs 0, 1; bytes 1, 3 pairs 2, 3
    __device__ __forceinline__ void bytes(int st, uint32_t &lo, uint32_t &hi) const {
        const int at = FMT == OXQ_GGUF_Q6_K ? ggm_pair_at(4 * (st & 1)) : ggm_bit_at(st, 0), next = FMT == OXQ_GGUF_Q6_K ? 2 : 1;
        constexpr uint32_t MASK = FMT == OXQ_GGUF_Q6_K ? 0x30303030u : 0x10101010u;
        const uint32_t w = q[0][st], h = FMT == OXQ_GGUF_Q6_K ? qh[st >> 1] : qh[0];
        auto moved = [&](int a) { return a < 4 ? h << (4 - a) : h >> (a - 4); };
        lo = (moved(at) & MASK) | (w & 0x0F0F0F0Fu), hi = (moved(at + next) & MASK) | ((w >> 4) & 0x0F0F0F0Fu);
    }
    // Q2_K, Q3_K: the unsigned integers of 32 elements, a byte each: lo pair 0, hi pair 1; bytes 0, 1 of step 2 st, 2, 3 of 2 st + 1
    __device__ __forceinline__ void bytes2(int st, uint32_t &lo, uint32_t &hi) const {
        const uint32_t w = qh[st >> 1] >> (4 * (st & 1));
        lo = w & 0x03030303u, hi = (w >> 2) & 0x03030303u;
        if constexpr (FMT == OXQ_GGUF_Q3_K) {
            auto third = [&](int at) { return (at < 2 ? qh[2] << (2 - at) : qh[2] >> (at - 2)) & 0x04040404u; };
            lo |= third(2 * st), hi |= third(2 * st + 1);
        }
    }
    // Formats with scales of 16 elements, the way rows of x lie: elements 8 kb .. + 7 of unit st, four bytes each in v0 and v1, all of
    // sub-block 2 st + kb / 2.  The copy gives lane group kb elements 4 kb .. + 3 of both sub-blocks; two exchanges of
    // lane groups turn one into the other.
    __device__ __forceinline__ void in_order(int st, uint32_t &v0, uint32_t &v1) const {
        uint32_t lo, hi, even, odd;  // of sub-block 2 st, 2 st + 1
        if constexpr (ggm_narrow<FMT>) {
            bytes2(st, lo, hi);
            even = pack_lo16(lo, hi), odd = pack_hi16(lo, hi);
        } else {
            bytes(st, lo, hi);
            even = perm_b32(hi, lo, 0x06040200u), odd = perm_b32(hi, lo, 0x07050301u);
        }
        const auto halves = __builtin_amdgcn_permlane32_swap(even, odd, false, false);           // {e0 e1 o0 o1}, {e2 e3 o2 o3}
        const auto rows = __builtin_amdgcn_permlane16_swap(halves[0], halves[1], false, false);  // {e0 e2 o0 o2}, {e1 e3 o1 o3}
        v0 = rows[0], v1 = rows[1];
    }
    // w = f0 q + c of the lane's elements of unit st in that order (q: the unsigned integer)
    __device__ __forceinline__ void factors_in_order(int ni, int kb, float (&f0)[4], float (&c)[4]) const {
        const int sh = 8 * (kb >> 1);
        const uint32_t u[2] = {uh[0] >> sh, uh[1] >> sh};
        const float d = ggm_f16(FMT == OXQ_GGUF_Q2_K || !(ni & 1) ? bh[0] & 0xFFFFu : bh[0] >> 16), dm = ggm_f16(bh[0] >> 16);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const uint32_t b = u[st >> 1] >> (16 * (st & 1));
            if constexpr (FMT == OXQ_GGUF_Q2_K) f0[st] = d * (float)(b & 0xFu), c[st] = -dm * (float)((b >> 4) & 0xFu);
            else f0[st] = d * (float)(int)(int8_t)(b & 0xFFu), c[st] = f0[st] * (FMT == OXQ_GGUF_Q3_K ? -4.0f : -32.0f);
        }
    }
    // B operand of step st: bias + q as bf16 pairs (four for a step of 32 elements, two for one of 16)
    __device__ __forceinline__ void operand(int st, uint32_t (&b)[4], const NibbleMasks &nm) const {
        if constexpr (FMT == OXQ_GGUF_Q4_0 || FMT == OXQ_GGUF_Q4_K || FMT == OXQ_GGUF_Q4_1) {
#pragma unroll
            for (int pp = 0; pp < 4; ++pp) b[pp] = BF16Traits::unpack1(q[0][st], pp, nm);
        } else if constexpr (ggm_fifth_bit<FMT>) {  // nibble | fifth bit << 4; m1: the bits' mask, in a register
#pragma unroll
            for (int pp = 0; pp < 4; ++pp) {
                const int sft = ggm_bit_at(st, pp) - 4;
                const uint32_t hs = sft < 0 ? (qh[0] << -sft) : (qh[0] >> sft);
                b[pp] = (hs & nm.m1) | BF16Traits::unpack1(q[0][st], pp, nm);
            }
        } else if constexpr (FMT == OXQ_GGUF_Q8_0) {
            const uint32_t w0 = q[st >> 1][2 * (st & 1)], w1 = q[st >> 1][2 * (st & 1) + 1];
            b[0] = ggm_bytes02(w0), b[1] = ggm_bytes13(w0), b[2] = ggm_bytes02(w1), b[3] = ggm_bytes13(w1);
        } else if constexpr (ggm_narrow<FMT>) {  // 0 .. 7 as f8 codes (512ths): no bias
            uint32_t lo, hi;
            bytes2(st >> 1, lo, hi);
            b[0] = __builtin_bit_cast(uint32_t, (st & 1) ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true)
                                                         : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
            b[1] = __builtin_bit_cast(uint32_t, (st & 1) ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true)
                                                         : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
            b[2] = b[3] = 0u;
        } else {  // Q6_K: nibble | bit pair << 4, 128 + (0 .. 63) is exact in bf16
            const uint32_t lw = q[0][st >> 1], hw = qh[st >> 2];
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {
                const int at = ggm_pair_at(2 * (st & 3) + pr);
                const uint32_t hs = at < 4 ? (hw << (4 - at)) : (hw >> (at - 4));
                b[pr] = (hs & nm.m1) | BF16Traits::unpack1(lw, 2 * (st & 1) + pr, nm);  // m1: the bit pairs' mask, in a register
            }
            b[2] = b[3] = 0u;
        }
    }
};

// The B operand with the smallest bias that leaves the integers exact, for f32 activations: 16 + q (4-bit formats), 32 + q
// (5-bit), 64 + q (Q6_K).  The bias and the format's offset come out in the same f32 accumulator, and the rounding of what
// is taken out there grows with its size: with 128 + q the sums carry seven times that of the integers' own products.  With
// these the 2-norm error is 0.3 - 0.93 x that of the vector kernels over K of 1024 - 14336 in every format (0.7e-7 - 1.5e-7
// of the result against 1e-7 - 3e-7).  Bytes (Q8_0) have no bias.  A pair is built as for 128 + q, with the bits moved to
// the mantissa position that the exponent asks for: as many instructions.
//
// Q4_1 and Q5_1, d q + m with q >= 0: no bias at all - nibbles widened as f8 codes, five-bit bytes through f32 - and the row's
// sum against ones.  Nothing is taken out, so an infinite x gives the infinity that the vector kernels give (in the other
// formats the offset or the subtracted minimum makes it NaN there and here).  Widened through f32 Q4_1 took up to 1.25 x as
// long; Q5_1 at 3 - 16 rows is at 1.03 - 1.13 x the biased operand's time.
template <int FMT> struct GgmSmallBias {
    static constexpr bool PLAIN = FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q5_1 || ggm_narrow<FMT>;
    static constexpr bool FOURS = FMT == OXQ_GGUF_Q4_1;  // pair i of the operand holds elements i and i + 4, else 2 i and 2 i + 1
    static constexpr bool NIB = FMT == OXQ_GGUF_Q4_0 || FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q4_K;
    static constexpr float BIAS = NIB ? 16.f : ggm_fifth_bit<FMT> ? 32.f : FMT == OXQ_GGUF_Q6_K ? 64.f : 0.f;
    // the constant that takes bias and offset out (the minimum's term divides by it)
    static constexpr float NEG = PLAIN ? 1.f : -(BIAS + (FMT == OXQ_GGUF_Q4_0 ? 8.f : FMT == OXQ_GGUF_Q5_0 ? 16.f : FMT == OXQ_GGUF_Q6_K ? 32.f : FMT == OXQ_GGUF_Q8_0 ? 128.f : 0.f));
    static constexpr uint32_t NEG_PAIR = (__builtin_bit_cast(uint32_t, NEG) >> 16) | (__builtin_bit_cast(uint32_t, NEG) & 0xFFFF0000u);
    static constexpr int AT = NIB ? 3 : ggm_fifth_bit<FMT> ? 2 : 1;  // mantissa bit of the nibble's lowest
    static constexpr uint32_t EXP = NIB ? 0x41804180u : ggm_fifth_bit<FMT> ? 0x42004200u : 0x42804280u;
    static constexpr uint32_t M0 = (0xFu << AT) * 0x10001u, M1 = (ggm_fifth_bit<FMT> ? 0x40u : 0x60u) * 0x10001u;
    __device__ static __forceinline__ uint32_t move(uint32_t v, int left) { return left >= 0 ? v << left : v >> -left; }
    __device__ static __forceinline__ void operand(const GgmChunk<FMT> &w, int st, uint32_t (&b)[4], const NibbleMasks &nm) {
        if constexpr (FMT == OXQ_GGUF_Q4_1) {  // nibbles as f8 codes (pk4g_widen): elements (0, 4), (1, 5), (2, 6), (3, 7)
            const uint32_t lo = w.q[0][st] & 0x0F0F0F0Fu, hi = (w.q[0][st] >> 4) & 0x0F0F0F0Fu;
            b[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
            b[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
            b[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
            b[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
        } else if constexpr (PLAIN && !ggm_narrow<FMT>) {  // bytes 0, 2 hold pair 0 or 1, bytes 1, 3 pair 2 or 3
            uint32_t lo, hi;
            w.bytes(st, lo, hi);
            b[0] = ggm_bytes02(lo), b[1] = ggm_bytes02(hi), b[2] = ggm_bytes13(lo), b[3] = ggm_bytes13(hi);
        } else if constexpr (NIB) {
#pragma unroll
            for (int pp = 0; pp < 4; ++pp) b[pp] = (move(w.q[0][st], AT - 4 * pp) & nm.m0) | EXP;
        } else if constexpr (ggm_fifth_bit<FMT>) {  // the bit of pair pp -> 6
#pragma unroll
            for (int pp = 0; pp < 4; ++pp)
                b[pp] = (move(w.qh[0], 6 - ggm_bit_at(st, pp)) & nm.m1) | ((move(w.q[0][st], AT - 4 * pp) & nm.m0) | EXP);
        } else if constexpr (FMT == OXQ_GGUF_Q6_K) {  // the bit pair of field f -> 5, 6
#pragma unroll
            for (int pr = 0; pr < 2; ++pr)
                b[pr] = (move(w.qh[st >> 2], 5 - ggm_pair_at(2 * (st & 3) + pr)) & nm.m1) |
                        ((move(w.q[0][st >> 1], AT - 4 * (2 * (st & 1) + pr)) & nm.m0) | EXP);
            b[2] = b[3] = 0u;
        } else {
            w.operand(st, b, nm);
        }
    }
};

typedef short short4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4_t ggm_mfma16(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4_t, u32x2_t{a0, a1}),
                                                     __builtin_bit_cast(short4_t, u32x2_t{b0, b1}), c, 0, 0, 0);
}

// Epilogue of a fused gate|up layer (ffn.rs:386-400 runs gated_silu_fused / gated_gelu_tanh_fused on the fused
// projection's output): the waves' partial tiles meet in LDS as in pk4n_epilogue; a thread then owns (row, gate
// column p of a strip and its up column p + 8), adds the waves in order, rounds both factors to bf16 as the
// projection's own output would be, and writes act(gate) * up to y [M, N / 2].
template <int MT, int NS, int NW>
__device__ __forceinline__ void ggm_epilogue_act(const float4_t (&acc)[MT][NS], const uint16_t *__restrict__ bias,
                                                 uint16_t *__restrict__ y, int M, int N, int j, int m0, int act,
                                                 int wave, int lane) {
    typedef BF16Traits TT;
    constexpr int NT = NW * 64, ROWS = 16 * MT;
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float *dst = (float *)(pk4_lds + (size_t)wave * MT * 4096) + ((mt * 4 + e) * 64 + lane) * NS;
#pragma unroll
            for (int f = 0; f < NS; ++f) dst[f] = acc[mt][f][e];
        }
    __syncthreads();
    const int half = N >> 1;
    for (int t = threadIdx.x; t < ROWS * 8 * NS; t += NT) {
        const int p = t & 7, f = (t >> 3) % NS, ml = t / (8 * NS);
        if (m0 + ml >= M) continue;
        const int mt = ml >> 4, r = ml & 15, kb = r >> 2, e = r & 3;
        float g = 0.f, u = 0.f;
#pragma unroll
        for (int s = 0; s < NW; ++s) {
            const float *src = (const float *)(pk4_lds + (size_t)s * MT * 4096) + ((mt * 4 + e) * 64 + kb * 16 + p) * NS + f;
            g += src[0];
            u += src[8 * NS];
        }
        const int n = 8 * (NS * j + f) + p;
        if (bias) {
            g += TT::to_f32(bias[n]);
            u += TT::to_f32(bias[half + n]);
        }
        g = TT::to_f32(TT::from_f32(g));
        u = TT::to_f32(TT::from_f32(u));
        y[(size_t)(m0 + ml) * half + n] = TT::from_f32(mul_f32_rn(act == 1 ? silu_f32(g) : gelu_tanh_f32(g), u));
    }
}

// Epilogue of the f32 form: tile row 4 p + m holds piece p of row m of x.  The waves' partial tiles meet in LDS; a wave
// takes a row of x, lane (p, ni) adds piece p's sums over the waves in pairs, and the three pieces' lanes meet, the
// smallest piece first.
template <int MT, int NS, int NW>
__device__ __forceinline__ void ggm_epilogue_f32(const float4_t (&acc)[MT][NS], const float *__restrict__ bias, float *__restrict__ y,
                                                 int M, int N, int j, int m0, int wave, int lane) {
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float *dst = (float *)(pk4_lds + (size_t)wave * MT * 4096) + ((mt * 4 + e) * 64 + lane) * NS;
#pragma unroll
            for (int f = 0; f < NS; ++f) dst[f] = acc[mt][f][e];
        }
    __syncthreads();
    for (int ml = wave; ml < 4 * MT && m0 + ml < M; ml += NW)
#pragma unroll
        for (int f = 0; f < NS; ++f) {
            float w[NW];
#pragma unroll
            for (int s = 0; s < NW; ++s) w[s] = ((const float *)(pk4_lds + (size_t)s * MT * 4096))[(ml * 64 + lane) * NS + f];
#pragma unroll
            for (int d = 1; d < NW; d *= 2)
#pragma unroll
                for (int s = 0; s < NW; s += 2 * d) w[s] += w[s + d];
            const float v = w[0] * (lane < 16 ? 1.0f : lane < 32 ? 0x1p-8f : 0x1p-16f), v1 = __shfl_down(v, 16), v2 = __shfl_down(v, 32);
            const int n = 16 * (NS * j + f) + lane;
            if (lane < 16 && n < N) {
                const float tot = (v2 + v1) + v;
                y[(size_t)(m0 + ml) * N + n] = bias ? tot + bias[n] : tot;
            }
        }
}
// f32 as three bf16 pieces, exactly: truncated to 8 significant bits, 2^8 times the rest truncated, 2^16 times the rest of
// that (at most 8 bits); the epilogue divides the pieces' sums again.  Unscaled, the second and third piece of values
// below 1e-34 fall below bf16's normal range, where they lose bits (values around 1e-36: 5e-5 of the result).  INF: an infinity is its first piece alone (formats whose sums can keep one).
template <bool INF> __device__ __forceinline__ void ggm_split3_pair(uint32_t a, uint32_t b, uint32_t (&p)[3]) {
    float ra = __builtin_bit_cast(float, a) - __builtin_bit_cast(float, a & 0xFFFF0000u);
    float rb = __builtin_bit_cast(float, b) - __builtin_bit_cast(float, b & 0xFFFF0000u);
    if constexpr (INF) {
        if (__builtin_isinf(__builtin_bit_cast(float, a))) ra = 0.f;
        if (__builtin_isinf(__builtin_bit_cast(float, b))) rb = 0.f;
    }
    ra *= 256.0f, rb *= 256.0f;
    const uint32_t am = __builtin_bit_cast(uint32_t, ra), bm = __builtin_bit_cast(uint32_t, rb);
    const float sa = 256.0f * (ra - __builtin_bit_cast(float, am & 0xFFFF0000u)), sb = 256.0f * (rb - __builtin_bit_cast(float, bm & 0xFFFF0000u));
    p[0] = pack_hi16(a, b), p[1] = pack_hi16(am, bm);
    p[2] = pack_hi16(__builtin_bit_cast(uint32_t, sa), __builtin_bit_cast(uint32_t, sb));
}
template <bool INF, bool FOURS> __device__ __forceinline__ void ggm_split3(const u32x4_t &v0, const u32x4_t &v1, u32x4_t (&p)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t t[3];
        if constexpr (FOURS) ggm_split3_pair<INF>(v0[i], v1[i], t);
        else ggm_split3_pair<INF>(i < 2 ? v0[2 * i] : v1[2 * i - 4], i < 2 ? v0[2 * i + 1] : v1[2 * i - 3], t);
        p[0][i] = t[0], p[1][i] = t[1], p[2][i] = t[2];
    }
}

// Q2_K, Q3_K: row x times column n weight by weight, in f32.  5 - 8 bf16 rows ran on the tile matmul with unrounded weights,
// where an infinity times a weight keeps its sign and a row of 1e37 has finite sums; with the integers in front of the scale, and the
// minimum or offset behind them, both are NaN.  A sum that is not finite is made again so (up to 4 rows ran on the vector kernel,
// which splits the weight in the same way), 2^24 smaller, so that it overflows only where the result does.  x: the row, 16-byte aligned.
template <int FMT>
__device__ __forceinline__ float ggm_narrow_dot(const uint8_t *__restrict__ pw, const uint16_t *__restrict__ x, int n, int K) {
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    constexpr bool THREE = FMT == OXQ_GGUF_Q3_K;
    const int ni = n & 15;
    const uint8_t *blk = pw + (size_t)(n >> 4) * (K >> 8) * L::BLKB;
    float sum = 0.f;
#pragma unroll 1
    for (int b = 0; b < K >> 8; ++b, blk += L::BLKB) {
        const float d = ggm_f16(*(const uint16_t *)(blk + L::BH_OFF + ni * F::BH));
        const float dm = THREE ? 0.f : ggm_f16(*(const uint16_t *)(blk + L::BH_OFF + ni * F::BH + F::BH - 2));
#pragma unroll 1
        for (int s = 0; s < 16; ++s) {  // sixteen elements: step s % 8 of chunk s / 8
            const uint8_t *chunk = blk + (s >> 3) * L::CHB;
            const int s2 = s & 7, t = s2 >> 1;
            const uint32_t sc = chunk[L::UH_OFF + ni * 8 + s2];
            const float f = d * (THREE ? (float)(int)(int8_t)sc : (float)(sc & 0xFu)), g = dm * (float)(sc >> 4);
            const u32x4_t xv[2] = {*(const u32x4_t *)(x + b * 256 + s * 16), *(const u32x4_t *)(x + b * 256 + s * 16 + 8)};
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const int lane = 16 * kb + ni, at = 16 * (s2 & 1);
                const uint32_t w = *(const uint32_t *)(chunk + lane * 8 + 4 * (t >> 1)) >> (at + 4 * (t & 1));
                const uint32_t w3 = THREE ? *(const uint32_t *)(chunk + 512 + lane * 4) >> (at + 2 * t) : 0u;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int bit = 8 * (i & 1) + (i >> 1);  // byte of the word, pair of the byte
                    const int q = (int)((w >> (bit + (i >> 1))) & 3u) | (THREE ? (int)((w3 >> bit) & 1u) << 2 : 0);
                    const float v = THREE ? f * (float)(q - 4) : f * (float)q - g;
                    const uint32_t pair = xv[kb >> 1][2 * (kb & 1) + (i >> 1)];
                    sum = __builtin_fmaf(v, __builtin_bit_cast(float, i & 1 ? pair & 0xFFFF0000u : pair << 16) * 0x1p-24f, sum);
                }
            }
        }
    }
    return sum * 0x1p24f;
}

// Waves a SIMD that an instantiation's registers have to leave room for.  Two workgroups of eight waves a compute unit are what
// hides the waits of one to four rows on layers of more than one round of strips; Q6_K came out two registers over that (a row,
// us, without / with room: 1024 x 9216 6.5 / 5.5, 4096 x 8704 12.3 / 10.8, 5632 x 7168 10.7 / 10.0).
template <int FMT, int MT, int XQ, int NW, int NS, bool XF32>
constexpr int ggm_waves = FMT == OXQ_GGUF_Q6_K && MT == 1 && XQ == 1 && NW == 8 && NS == 1 && !XF32 ? 4 : 1;

// XF32: f32 activations and results.  An f32 value is the sum of three bf16 pieces, so four rows of x are twelve rows of
// a matrix-core tile (piece p of row m in tile row 4 p + m) and the products stay exact; MT tiles take 4 MT rows of x,
// XQ = 2 MT loads bring them.  The vector-ALU kernel on the rotated copy does the same work once per row.  XQ = 1: a single
// row, whose chunk the whole wave fetches and splits, two elements a lane.
// f32 results keep what the sums hold, so a chunk's steps are summed by themselves before they join the wave's sum: added to it
// one by one, 4 - 16 roundings a chunk at the size of the whole sum, the formats with a minimum were 1.4 - 1.8 x as far from
// 64 bits as the vector kernels at K = 14336 (Q4_K at 8 rows 1.7e-7 against 1.25e-7; now 1.0e-7, at up to 2.5 % of the time).
// NL > 0 (ggm_short_kernel): no wave has more than NL chunks, all of them requested at once; 0: a loop.
template <int FMT, int MT, int XQ, int NW, int NS, bool XF32, int NL>
__device__ __forceinline__ void ggm_body(const uint16_t *__restrict__ x, const uint8_t *__restrict__ pw, const uint16_t *__restrict__ bias,
                                         uint16_t *__restrict__ y, float *__restrict__ ws, int M, int K, int N, int cslice, int act) {
    constexpr bool ONE = XF32 && XQ == 1;
    static_assert(!XF32 || XQ == 2 * MT || (ONE && MT == 1), "two loads a lane bring four rows' chunk of f32");
    constexpr int TROWS = XF32 ? 4 * MT : 16 * MT;  // rows of x a tile takes
    typedef BF16Traits TT;
    typedef MfmaOps<TT> Ops;
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    typedef GgmChunk<FMT> C;
    constexpr int ROWS = 16 * MT, AQ = XQ, SLOT = ROWS * 256, OOB = 0x7FFFFF00, NSTEP = C::NSTEP;
    // chunks in flight a wave: three (4096 x 4096 at one row, Q8_0: 5.06 us with three, 5.87 with two); two
    // where a workgroup takes four strips, whose quants are four times the registers
    constexpr int RD = NL > 0 ? NL : NS > 1 ? 2 : 3;
    constexpr bool K16 = NSTEP == 8;  // steps of 16 elements
    extern __shared__ __attribute__((aligned(16))) unsigned char pk4_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ni = lane & 15, kb = lane >> 4;
    const int j = blockIdx.x;
    const int m0 = blockIdx.z * TROWS;
    const int NC = K >> 7;
    const int sc0 = blockIdx.y * cslice;
    const int SC = min(NC, sc0 + cslice) - sc0;
    const int cbase = SC / NW, crem = SC % NW;
    const int nloc = cbase + (wave < crem ? 1 : 0);
    const int cc0 = sc0 + wave * cbase + min(wave, crem);
    unsigned char *slot = pk4_lds + wave * SLOT;

    // the workgroup's NS neighbouring strips behind one descriptor (NS * strip_bytes < 2^31: checked on the host)
    const uint32_t strip_bytes = (uint32_t)(NC / F::CH) * (uint32_t)L::BLKB;
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(pw + (size_t)j * NS * strip_bytes, NS * strip_bytes);
    const int xrows = min(M - m0, TROWS);
    constexpr int XB = XF32 ? 4 : 2;  // bytes of an element of x
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc((const uint8_t *)x + (size_t)m0 * K * XB, (uint32_t)xrows * (uint32_t)K * XB);
    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    int voff_a[AQ];
#pragma unroll
    for (int q = 0; q < AQ; ++q) {
        const int r = ONE ? 0 : XF32 ? 4 * (q >> 1) + kb : 4 * q + kb;
        const int at = ONE ? ni * 32 + kb * (GgmSmallBias<FMT>::FOURS ? 4 : 8) : XF32 ? r * K * 4 + ni * 32 + (q & 1) * 16 : r * K * 2 + ni * 16;
        voff_a[q] = r < xrows ? at : OOB;
    }
    // x in LDS: row r of the tile at r * 256, its sixteen 16-byte pieces XOR-swizzled by the row
    int a_wr[4];
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) a_wr[qq] = kb * 256 + (((ni ^ kb) ^ (qq << 2)) << 4);
    // step st of the chunk: elements 32 st + 8 kb .. + 7 of row ni (16 st + 4 kb .. + 3 for steps of 16)
    int a_rd[NSTEP];
#pragma unroll
    for (int st = 0; st < NSTEP; ++st)
        a_rd[st] = K16 ? ni * 256 + (((2 * st + (kb >> 1)) ^ ni) << 4) + (kb & 1) * 8 : ni * 256 + (((4 * st + kb) ^ ni) << 4);
    // both masks in registers: v_and_or_b32 takes one literal, and the exponent pattern is it
    const NibbleMasks nm = XF32 ? NibbleMasks{vgpr_const(GgmSmallBias<FMT>::M0), vgpr_const(GgmSmallBias<FMT>::M1)} : FMT == OXQ_GGUF_Q6_K ? NibbleMasks{vgpr_const(0x000F000Fu), vgpr_const(0x00300030u)}
                           : ggm_fifth_bit<FMT> ? NibbleMasks{vgpr_const(0x000F000Fu), vgpr_const(0x00100010u)} : nibble_masks();
#pragma unroll
    for (int q = XF32 ? 0 : AQ; q < 4 * MT; ++q) {  // rows no call of this instantiation brings stay zero
        if (XF32 && !ONE && (q & 3) != 3) continue;
        const int row = 4 * q + kb;
        *(u32x4_t *)(slot + row * 256 + ((ni ^ (row & 15)) << 4)) = u32x4_t{0u, 0u, 0u, 0u};
    }

    C wr[RD][NS];
    u32x4_t ar[RD][AQ];
    auto request = [&](int i, C (&w)[NS], u32x4_t (&a)[AQ]) {
        const bool live = i < nloc;  // wave-uniform
        const __amdgpu_buffer_rsrc_t rx = live ? rs_x : rs_none, rw = live ? rs_w : rs_none;
        const int c = cc0 + i;
#pragma unroll
        for (int q = 0; q < AQ; ++q) {
            if constexpr (ONE && GgmSmallBias<FMT>::FOURS) {
                a[0][0] = __builtin_amdgcn_raw_buffer_load_b32(rx, voff_a[0], c * 512, 0);
                a[0][1] = __builtin_amdgcn_raw_buffer_load_b32(rx, voff_a[0], c * 512 + 16, 0);
            } else if constexpr (ONE) {
                const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rx, voff_a[0], c * 512, 0);
                a[0][0] = v[0], a[0][1] = v[1];
            } else {
                a[q] = __builtin_amdgcn_raw_buffer_load_b128(rx, voff_a[q], c * (128 * XB), 0);
            }
        }
#pragma unroll
        for (int f = 0; f < NS; ++f) w[f].request(rw, lane, ni, c, (int)(f * strip_bytes));
        __builtin_amdgcn_sched_barrier(0);  // chunks are requested in the order they are used
    };
    if constexpr (NL > 0) {  // the last chunk has the last set, whatever their number
#pragma unroll
        for (int d = 0; d < RD; ++d)
            if (nloc - RD + d >= 0) request(nloc - RD + d, wr[d], ar[d]);
    } else {
#pragma unroll
        for (int d = 0; d < RD; ++d) request(d, wr[d], ar[d]);
    }

    float4_t acc[MT][NS];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NS; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    constexpr bool FOURS = XF32 && GgmSmallBias<FMT>::FOURS;
    constexpr bool PLAIN = (XF32 || ggm_narrow<FMT>) && GgmSmallBias<FMT>::PLAIN;  // the integers without a bias: their sums start from zero
    constexpr uint32_t NEGP = XF32 ? GgmSmallBias<FMT>::NEG_PAIR : F::NEG;
    const uint32_t neg[4] = {NEGP, NEGP, NEGP, NEGP};
    // the minimum's factor is per 128 (factors()); here the bias term is smaller
    constexpr float MINF = (XF32 || ggm_narrow<FMT>) && C::HAS_MIN ? 128.0f / -GgmSmallBias<FMT>::NEG : 1.0f;
    auto operand = [&](const C &w, int st, uint32_t (&b)[4], const NibbleMasks &k) {
        if constexpr (XF32) GgmSmallBias<FMT>::operand(w, st, b, k);
        else w.operand(st, b, k);
    };
    const float4_t zero4 = float4_t{0.f, 0.f, 0.f, 0.f};

    // A operand of step st, row tile mt
    auto load_a = [&](int st, int mt, uint32_t (&a)[4]) {
        if constexpr (K16) {
            const uint2 av = *(const uint2 *)(slot + mt * 4096 + a_rd[st]);
            a[0] = av.x, a[1] = av.y, a[2] = 0u, a[3] = 0u;
        } else {
            const u32x4_t av = *(const u32x4_t *)(slot + mt * 4096 + a_rd[st]);
            a[0] = av[0], a[1] = av[1], a[2] = av[2], a[3] = av[3];
        }
    };
    auto mma = [&](const uint32_t (&a)[4], const uint32_t (&b)[4], float4_t c) -> float4_t {
        if constexpr (K16) return ggm_mfma16(a[0], a[1], b[0], b[1], c);
        else return Ops::mfma(a, b, c);
    };

    auto chunk = [&](int i, auto cur_c, bool more) {
        constexpr int CUR = decltype(cur_c)::value;
        if constexpr (ONE) {
            uint32_t part[3];
            ggm_split3_pair<PLAIN>(ar[CUR][0][0], ar[CUR][0][1], part);
#pragma unroll
            for (int p = 0; p < 3; ++p) *(uint32_t *)(slot + p * 1024 + ((ni ^ (4 * p)) << 4) + kb * 4) = part[p];
        } else if constexpr (XF32) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                u32x4_t part[3];
                ggm_split3<PLAIN, FOURS>(ar[CUR][2 * t], ar[CUR][2 * t + 1], part);
#pragma unroll
                for (int p = 0; p < 3; ++p) *(u32x4_t *)(slot + (4 * t + p) * 1024 + a_wr[p]) = part[p];
            }
        } else {
#pragma unroll
            for (int q = 0; q < AQ; ++q) *(u32x4_t *)(slot + q * 1024 + a_wr[q & 3]) = ar[CUR][q];
        }
        float f0[NSTEP], f1[NSTEP];
        if constexpr (MT == 1) {
            // what depends on x alone first (x is requested ahead of the chunk's quants): the operands and the
            // bias term of four steps, so that one MFMA a step and strip is left when the quants arrive
#pragma unroll
            for (int g = 0; g < NSTEP; g += 4) {
                uint32_t a[4][4];
                float4_t tn[4];
#pragma unroll
                for (int s4 = 0; s4 < 4; ++s4) {
                    load_a(g + s4, 0, a[s4]);
                    tn[s4] = mma(a[s4], neg, zero4);
                }
#pragma unroll
                for (int f = 0; f < NS; ++f) {
                    const C &w = wr[CUR][f];
                    if (g == 0 || NS > 1) w.factors((cc0 + i) & 1, ni, f0, f1);
                    float4_t own = XF32 ? zero4 : acc[0][f];
                    if constexpr (C::HAS_MIN) {
#pragma unroll
                        for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                            for (int e = 0; e < 4; ++e) own[e] = fmaf(f1[g + s4] * MINF, tn[s4][e], own[e]);
                    }
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        uint32_t b[4];
                        operand(w, g + s4, b, nm);
                        const float4_t t = mma(a[s4], b, PLAIN ? zero4 : tn[s4]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) own[e] = fmaf(f0[g + s4], t[e], own[e]);
                    }
                    if constexpr (XF32) acc[0][f] += own;
                    else acc[0][f] = own;
                    if constexpr (NS > 1) __builtin_amdgcn_sched_barrier(0);  // one strip's operands at a time
                }
            }
        } else {  // more row tiles: step by step, the registers do not hold a chunk's operands
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                const C &w = wr[CUR][f];
                w.factors((cc0 + i) & 1, ni, f0, f1);
                float4_t own[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) own[mt] = XF32 ? zero4 : acc[mt][f];
#pragma unroll
                for (int st = 0; st < NSTEP; ++st) {
                    uint32_t b[4];
                    operand(w, st, b, nm);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        uint32_t a[4];
                        load_a(st, mt, a);
                        const float4_t tn = mma(a, neg, zero4);
                        const float4_t t = mma(a, b, PLAIN ? zero4 : tn);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            own[mt][e] = fmaf(f0[st], t[e], own[mt][e]);
                            if constexpr (C::HAS_MIN) own[mt][e] = fmaf(f1[st] * MINF, tn[e], own[mt][e]);
                        }
                    }
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    if constexpr (XF32) acc[mt][f] += own[mt];
                    else acc[mt][f] = own[mt];
                }
                if constexpr (NS > 1) __builtin_amdgcn_sched_barrier(0);  // one strip's operands at a time
            }
        }
        if (more) request(i + RD, wr[CUR], ar[CUR]);
        __builtin_amdgcn_sched_barrier(0);  // one chunk's operands in the registers at a time
    };
    // A load that brings nothing (past a wave's last chunk) takes its turn in the address unit as any other: none but at the loop's
    // start.  us, the last round of chunks in the loop -> behind it: 6144 x 4096 at 1 / 6 / 16 rows Q4_K 5.9 / 6.7 / 11.4 -> 5.3 / 5.8 / 7.6, Q6_K
    // 8.1 / 8.5 / 15.0 -> 6.8 / 7.1 / 9.2, 3072 x 8192 at 6 / 24 Q4_K 6.6 / 15.2 -> 5.8 / 12.3, Q8_0 9.1 / 16.5 -> 7.2 / 13.3; four strips, 2048 x 16384
    // at 1 / 32 Q4_K 8.2 / 13.1 -> 7.4 / 11.5, 4096 x 14336 at 1 / 32 11.2 / 19.1 -> 10.7 / 18.3.
    const std::integral_constant<int, 0> c0;
    const std::integral_constant<int, 1> c1;
    const std::integral_constant<int, 2> c2;
    if constexpr (NL > 0) {
        static_assert(NL <= 2, "two chunks at most");
        if constexpr (NL == 2) {
            if (nloc > 1) chunk(nloc - 2, c0, false);
        }
        if (nloc > 0) chunk(nloc - 1, std::integral_constant<int, NL - 1>{}, false);
    } else {
        int i = 0;
        if constexpr (RD == 2) {
            for (; i + 2 < nloc; i += 2) {
                chunk(i, c0, true);
                chunk(i + 1, c1, true);
            }
            if (i < nloc) chunk(i, c0, false);
            if (i + 1 < nloc) chunk(i + 1, c1, false);
        } else {
            for (; i + 3 < nloc; i += 3) {
                chunk(i, c0, true);
                chunk(i + 1, c1, true);
                chunk(i + 2, c2, true);
            }
            if (i < nloc) chunk(i, c0, false);
            if (i + 1 < nloc) chunk(i + 1, c1, false);
            if (i + 2 < nloc) chunk(i + 2, c2, false);
        }
    }
    if constexpr (XF32) ggm_epilogue_f32<MT, NS, NW>(acc, (const float *)bias, (float *)y, M, N, j, m0, wave, lane);
    else if (act) ggm_epilogue_act<MT, NS, NW>(acc, bias, y, M, N, j, m0, act, wave, lane);
    else if constexpr (ggm_narrow<FMT> && XQ > 1)
        pk4n_epilogue<TT, MT, NS, NW, true>(acc, bias, y, ws, M, N, j, m0, wave, lane, [&](float v, int m, int n) {
            return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) == 0x7F800000u ? ggm_narrow_dot<FMT>(pw, x + (size_t)m * K, n, K) : v;
        });
    else pk4n_epilogue<TT, MT, NS, NW, true>(acc, bias, y, ws, M, N, j, m0, wave, lane);
}

template <int FMT, int MT, int XQ, int NW, int NS, bool XF32 = false>
__global__ __launch_bounds__(NW * 64, (ggm_waves<FMT, MT, XQ, NW, NS, XF32>)) void ggm_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ pw, const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
    float *__restrict__ ws, int M, int K, int N, int cslice, int act) {
    ggm_body<FMT, MT, XQ, NW, NS, XF32, 0>(x, pw, bias, y, ws, M, K, N, cslice, act);
}
// The same for up to NL chunks a wave, without the loop's code to jump over: a kernel's instructions come from memory anew at each launch.
template <int FMT, int MT, int XQ, int NW, int NS, bool XF32, int NL>
__global__ __launch_bounds__(NW * 64, (ggm_waves<FMT, MT, XQ, NW, NS, XF32>)) void ggm_short_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ pw, const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
    float *__restrict__ ws, int M, int K, int N, int cslice, int act) {
    ggm_body<FMT, MT, XQ, NW, NS, XF32, NL>(x, pw, bias, y, ws, M, K, N, cslice, act);
}

// ---------------------------------------------------------------------------
// prefill: the decomposition of pk4n_gemm_kernel on the matrix-core copy
// ---------------------------------------------------------------------------
// More rows than the integer kernel above should take (every 32 of them read the weights again, and the scale is
// applied per unit and output) run the tile arithmetic of the reference's mul_mm (quant_kernels.metal strips,
// linear.rs:270-284 forward_prefill): B = the dequantized weight rounded once to bf16, f32 accumulation.  A
// workgroup takes 64 rows of x and eight waves x four neighbouring strips (512 columns); a chunk (128 elements of
// K) of the rows goes from global memory straight into LDS once for all eight waves (two buffers, one barrier a
// chunk); a wave rings its four strips' chunks in two halves, turns a step's integers into the weight with one
// fma each (two where a five-bit format has a minimum) from the integer kernel's own factors, and keeps the whole
// K in its accumulators: one launch, no partial tiles.
// KS = 4: two waves of 64 columns a workgroup and the four waves of a column group take every fourth chunk, as in
// pk4_gemm_kernel - the form for 33 to a few hundred rows of a wide layer.  A layer of few columns does not fill the chip
// with such workgroups: gridDim.y slices of `cslice` chunks each then write their f32 tiles to `part` and a second
// launch adds them in slice order.  half: a fused gate|up layer without its activation - columns go back to the
// file's order (ggm_src_row).
// NS = 2, MT = 8: 128 rows, a wave has two strips.  What bounds the form above is the conversion's vector instructions, 5 - 7 an
// MFMA at four row tiles a weight; here a weight serves eight (Q4_K 4.1, Q6_K 4.8 an MFMA; the MFMAs take 45 and 37 % of the time),
// at the price of LDS, whose fragment then feeds two MFMAs instead of four (reads, without conflicts: 22 and 19 %).  (Four strips do
// not fit: 128 accumulators beside two ring halves.)  KS = 1: 256 columns, 143 - 161 registers; KS = 2: 128
// columns, the two waves of a column group take every other chunk and finish four row tiles each - for launches that 256 columns
// leave CUs idle in.  us, best of the forms of 64 rows -> 128: Q4_K 4096 x 4096 at 520 / 1024 / 2048 rows 55 / 56 / 91 -> 39 / 42 / 71,
// 4096 x 14336 at 256 / 1024 / 2048 56 / 179 / 345 -> 41 / 136 / 262, 14336 x 4096 at 777 164 -> 122; Q8_0 4096 x 14336 at 2048
// 344 -> 275; Q6_K 435 -> 312; Q3_K 405 -> 281.
// What bounds it: the conversion's vector instructions beside the MFMAs.  The five- and six-bit formats join nibble and plane bits
// four weights at a time into bytes (GgmChunk::bytes), 3.4 instructions a weight; pair by pair as the integer kernel's operand
// they took 4.3, and 5.3 with a minimum added behind the fma (Q6_K / Q5_K / Q5_1 / Q5_0 4096 x 4096 at 2048 rows 127 / 130 /
// 123 / 108 -> 113 / 105 / 96 / 95 us in the 64-row form).  Q6_K multiplies its two scales of a 32-element step into one MFMA's
// operand (of 16 elements each before).
// Formats with scales of 16 elements: at 128 rows the integers go into the order of the rows of x (GgmChunk::in_order): one scale a
// lane and step, half of the factors, and whole 16-byte reads of x instead of two of 8 bytes that met in the banks (3 - 7 cycles a
// read): Q6_K 4096 x 14336 at 2048 rows 395 -> 312 us.  At 64 rows, where a fragment serves four strips, the exchanges
// cost what the reads save (439 / 435), and more at 48 (14336 x 4096 at 33 22.1 / 22.5): those keep elements 4 kb .. + 3 of both halves.
// NS: strips of a wave.
template <int FMT, int MT, int KS, int NS = 4>
__global__ __launch_bounds__(512) void ggm_gemm_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ pw,
                                                       const uint16_t *__restrict__ bias, uint16_t *__restrict__ y,
                                                       float *__restrict__ part, int M, int K, int N, int NG, int RT, int act,
                                                       int cslice, int half) {
    typedef BF16Traits TT;
    typedef MfmaOps<TT> Ops;
    typedef GgmFmt<FMT> F;
    typedef GgmLayout<FMT> L;
    typedef GgmChunk<FMT> C;
    static_assert(KS == 1 || KS >= MT || MT % KS == 0, "the waves of a column group finish as many row tiles each");
    constexpr int SPW = 8 / KS;  // waves of 16 NS columns a workgroup
    constexpr int ROWS = 16 * MT, XBUF = KS * ROWS * 256, XV = ROWS / 4 / SPW;
    constexpr bool K16 = ggm_k16<FMT> && NS == 4;    // scales of 16 elements: an MFMA takes two of them, four elements a lane each
    constexpr bool ORDER = ggm_k16<FMT> && NS != 4;  // in the order of the rows of x: a lane's eight are within one
    constexpr int NSTEP = K16 ? C::NSTEP : 4;
    constexpr int RING = NS * C::LOADS;  // vector loads of a chunk's weights: younger than the chunk's loads of x
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
    const int j = g * SPW + ws;  // the wave's columns: strips NS j .. NS j + NS - 1
    const int strips = (N + 15) >> 4;
    const bool live = NS * j < strips;
    const int m0 = rt * ROWS;
    const int NC = K >> 7;
    const int cbeg = (int)blockIdx.y * cslice, cend = min(NC, cbeg + cslice);  // the slice's chunks
    const int NR = (cend - cbeg + KS - 1) / KS;                                // rounds of KS chunks
    const int xrows = min(M - m0, ROWS);

    const uint32_t strip_bytes = (uint32_t)(NC / F::CH) * (uint32_t)L::BLKB;
    const __amdgpu_buffer_rsrc_t rs_none = make_rsrc(pw, 0u);
    const __amdgpu_buffer_rsrc_t rs_wl = make_rsrc(pw + (size_t)(live ? NS * j : 0) * strip_bytes, (uint32_t)min(NS, live ? strips - NS * j : NS) * strip_bytes);
    const __amdgpu_buffer_rsrc_t rs_w = live ? rs_wl : rs_none;
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x + (size_t)m0 * K, (uint32_t)xrows * (uint32_t)K * 2u);
    // x: load q of a wave brings rows 4 (XV wave + q) .. + 3 of the chunk, lane l the 16 bytes that belong at
    // position l % 16 of row l / 16 (piece (l % 16) ^ (row % 16): the swizzle the fragment reads undo); rows past
    // M lie beyond the descriptor and arrive as zeros
    int xo[XV];
#pragma unroll
    for (int q = 0; q < XV; ++q) {
        const int r = 4 * (ws * XV + q) + (lane >> 4);
        xo[q] = r * K * 2 + (((lane & 15) ^ (r & 15)) << 4);
    }
    int a_rd[NSTEP];
#pragma unroll
    for (int st = 0; st < NSTEP; ++st)
        a_rd[st] = K16 ? ni * 256 + (((2 * st + (kb >> 1)) ^ ni) << 4) + (kb & 1) * 8 : ni * 256 + (((4 * st + kb) ^ ni) << 4);
    constexpr float NEGF = __builtin_bit_cast(float, (F::NEG & 0xFFFFu) << 16);
    constexpr bool NIB = FMT == OXQ_GGUF_Q4_0 || FMT == OXQ_GGUF_Q4_1 || FMT == OXQ_GGUF_Q4_K;

    C wr[2][NS];
    auto dma_x = [&](int r) {  // round r: the wave's chunk is KS r + kq, its tile of x at kq ROWS 256 of the round's buffer
        const int i = cbeg + KS * r + kq;
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_x : rs_none;
#pragma unroll
        for (int q = 0; q < XV; ++q)
            pk4g_load_lds16(rs, pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256) + (ws * XV + q) * 1024, xo[q], i * 256);
    };
    auto request = [&](int i, C (&w)[NS]) {
        const __amdgpu_buffer_rsrc_t rs = i < cend ? rs_w : rs_none;
#pragma unroll
        for (int f = 0; f < NS; ++f) w[f].request(rs, lane, ni, i, (int)(f * strip_bytes));
    };

    dma_x(0);
    __builtin_amdgcn_sched_barrier(0);  // requests keep this order: the wait counts rely on it
    request(cbeg + kq, wr[0]);
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc[MT][NS];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NS; ++f) acc[mt][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    pk4g_wait_vmcnt<RING>();
    __syncthreads();

    auto chunk = [&](int r, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        const int i = cbeg + KS * r + kq;  // past the slice (a ragged last round): zeros from both streams
        dma_x(r + 1);
        __builtin_amdgcn_sched_barrier(0);
        request(i + KS, wr[CUR ^ 1]);
        __builtin_amdgcn_sched_barrier(0);  // not sunk to the chunk's end, where the next chunk would wait for them
        const unsigned char *buf = pk4_lds + (r & 1) * XBUF + kq * (ROWS * 256);
        // w = f0 q' + c2 with q' = q minus the format's offset and c2 = -(minimum): exact products, one rounding -
        // the bits of the dense dequant (ggm_dequant_kernel), so the tile the matrix cores see is the reference's
        float f0[NS][NSTEP], c2[NS][C::HAS_MIN || ORDER ? NSTEP : 1];
#pragma unroll
        for (int f = 0; f < NS; ++f) {
            if constexpr (ORDER) {
                wr[CUR][f].factors_in_order(ni, kb, f0[f], c2[f]);
            } else {
                float f1[NSTEP];
                wr[CUR][f].factors(i & 1, ni, f0[f], f1);
                if constexpr (C::HAS_MIN) {
#pragma unroll
                    for (int st = 0; st < NSTEP; ++st) c2[f][st] = -128.0f * f1[st];
                }
            }
        }
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            uint32_t a[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if constexpr (K16) {
                    const uint2 a0 = *(const uint2 *)(buf + mt * 4096 + a_rd[2 * st]), a1 = *(const uint2 *)(buf + mt * 4096 + a_rd[2 * st + 1]);
                    a[mt][0] = a0.x, a[mt][1] = a0.y, a[mt][2] = a1.x, a[mt][3] = a1.y;
                } else {
                    const u32x4_t av = *(const u32x4_t *)(buf + mt * 4096 + a_rd[st]);
                    a[mt][0] = av[0], a[mt][1] = av[1], a[mt][2] = av[2], a[mt][3] = av[3];
                }
            }
#pragma unroll
            for (int f = 0; f < NS; ++f) {
                uint32_t b[4];
                const float sc = f0[f][st];
                if constexpr (K16 && ggm_narrow<FMT>) {
                    uint32_t lo, hi;
                    wr[CUR][f].bytes2(st, lo, hi);
                    float ql[4], qu[4];
                    pk4g_widen(lo, ql), pk4g_widen(hi, qu);
                    const Pk4gBf16 c0 = {f0[f][2 * st], c2[f][2 * st]}, c1 = {f0[f][2 * st + 1], c2[f][2 * st + 1]};
                    b[0] = c0.pair(ql[0], ql[1]), b[1] = c0.pair(qu[0], qu[1]), b[2] = c1.pair(ql[2], ql[3]), b[3] = c1.pair(qu[2], qu[3]);
                } else if constexpr (K16) {
                    uint32_t lo, hi;
                    wr[CUR][f].bytes(st, lo, hi);
                    Pk4gBf16 c0, c1;
                    c0.set(f0[f][2 * st], -32.0f), c1.set(f0[f][2 * st + 1], -32.0f);
                    b[0] = c0.template bytes<0>(lo), b[1] = c0.template bytes<0>(hi), b[2] = c1.template bytes<1>(lo), b[3] = c1.template bytes<1>(hi);
                } else if constexpr (ORDER) {
                    uint32_t v0, v1;
                    wr[CUR][f].in_order(st, v0, v1);
                    const Pk4gBf16 cv = {sc, c2[f][st]};
                    if constexpr (ggm_narrow<FMT>) {
                        float q0[4], q1[4];
                        pk4g_widen(v0, q0), pk4g_widen(v1, q1);
                        b[0] = cv.pair(q0[0], q0[1]), b[1] = cv.pair(q0[2], q0[3]), b[2] = cv.pair(q1[0], q1[1]), b[3] = cv.pair(q1[2], q1[3]);
                    } else {
                        b[0] = cv.pair((float)(v0 & 0xFFu), (float)((v0 >> 8) & 0xFFu)), b[1] = cv.pair((float)((v0 >> 16) & 0xFFu), (float)(v0 >> 24));
                        b[2] = cv.pair((float)(v1 & 0xFFu), (float)((v1 >> 8) & 0xFFu)), b[3] = cv.pair((float)((v1 >> 16) & 0xFFu), (float)(v1 >> 24));
                    }
                } else if constexpr (NIB) {
                    // plain nibbles (pair pp = nibble pp of each 16-bit half)
                    Pk4gBf16 cv;
                    cv.s = sc, cv.c = C::HAS_MIN ? c2[f][st] : (NEGF + 128.0f) * sc;
                    cv.rows(wr[CUR][f].q[0][st], b);
                } else if constexpr (FMT == OXQ_GGUF_Q8_0) {
                    // bytes q + 128, elements 0, 2, 1, 3 of a word's four: pairs in bytes (0, 2) and (1, 3)
                    const uint32_t w0 = wr[CUR][f].q[st >> 1][2 * (st & 1)], w1 = wr[CUR][f].q[st >> 1][2 * (st & 1) + 1];
                    Pk4gBf16 cv;
                    cv.s = sc, cv.c = -128.0f * sc;
                    b[0] = cv.template bytes<0>(w0), b[1] = cv.template bytes<1>(w0);
                    b[2] = cv.template bytes<0>(w1), b[3] = cv.template bytes<1>(w1);
                } else {  // five bits
                    uint32_t lo, hi;
                    wr[CUR][f].bytes(st, lo, hi);
                    Pk4gBf16 cv;
                    cv.s = sc, cv.c = C::HAS_MIN ? c2[f][st] : (NEGF + 128.0f) * sc;
                    b[0] = cv.template bytes<0>(lo), b[1] = cv.template bytes<0>(hi), b[2] = cv.template bytes<1>(lo), b[3] = cv.template bytes<1>(hi);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][f] = Ops::mfma(a[mt], b, acc[mt][f]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        pk4g_wait_vmcnt<RING>();  // this wave's part of the next chunk of x is in LDS
        __syncthreads();
    };
    {
        int r = 0;
        for (; r + 1 < NR; r += 2) {
            chunk(r, std::integral_constant<int, 0>{});
            chunk(r + 1, std::integral_constant<int, 1>{});
        }
        if (r < NR) {
            chunk(r, std::integral_constant<int, 0>{});
            // no weights are requested past this round, so RING counts loads that are not there: the zeros requested for
            // the round after it must be in LDS before the sum uses the place
            pk4g_wait_vmcnt<0>();
            __syncthreads();
        }
    }

    // the finished tile rows of this wave: all of them (KS = 1), or row tiles FT kq .. + FT - 1 summed over the column group's waves
    constexpr int FT = KS == 1 ? MT : (MT + KS - 1) / KS;
    float4_t fin[FT][NS];
    if constexpr (KS == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < NS; ++f) fin[mt][f] = acc[mt][f];
    } else {
        // slot of wave w: [mt][e][lane] x NS floats; the last round's barrier has freed the buffers
        typedef float part_t __attribute__((ext_vector_type(NS)));
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
            for (int k = 0; k < KS; ++k)  // K order: the same sum whatever the timing
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const part_t v = red[(((k * SPW + ws) * MT + min(FT * kq + t, MT - 1)) * 4 + e) * 64 + lane];
#pragma unroll
                    for (int f = 0; f < NS; ++f) fin[t][f][e] += v[f];
                }
        }
    }
    if (!live || (KS > MT && kq >= MT)) return;
    // 128 rows: stores of four columns (a quad of lanes turns its 4 x 4 values; four neighbours of the copy are neighbours of y,
    // ggm_src_row) where rows of y begin on 8 bytes, not of one: Q4_K 1024 x 8192 at 300 / 2048 rows 14.9 -> 14.3 / 49.4 -> 47.6 us, 4096 x
    // 14336 at 2048 270 -> 268.  With one row tile a wave, as in the forms of 64 rows, they gain nothing (Q6_K 4096 x 4096 at 300 33.0 / 34.3).
    const bool by4 = NS == 2 && ((uintptr_t)y & 7) == 0 && N % 4 == 0;
    const int quad = ni & 3;
    if (act) {
        // Fused gate|up layer (ggm_src_row): strip NS j + f holds gate columns 8 (NS j + f) .. + 7 in lanes ni < 8 and
        // the up columns they meet in lanes ni + 8.  The two lanes of a pair exchange their values (row_ror:8) and finish
        // half of the outputs each; both factors rounded to bf16 first, as in ggm_epilogue_act.  y is [M, N / 2].
        const int hc = N >> 1, p = ni & 7;
        const bool low = ni < 8;
        float bv[NS] = {};
        if (bias) {
#pragma unroll
            for (int f = 0; f < NS; ++f) bv[f] = TT::to_f32(bias[(low ? 0 : hc) + 8 * (NS * j + f) + p]);
        }
#pragma unroll
        for (int t = 0; t < FT; ++t) {
            uint32_t o4[4];  // NS = 2
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + e;
                float mine[NS], other[NS];
#pragma unroll
                for (int f = 0; f < NS; ++f) {
                    mine[f] = TT::to_f32(TT::from_f32(fin[t][f][e] + bv[f]));
                    other[f] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, mine[f]), 0x128, 0xF, 0xF, false));
                }
#pragma unroll
                for (int q = 0; q < NS / 2; ++q) {
                    const int f = low ? q : NS / 2 + q;
                    const float gq = low ? mine[q] : other[NS / 2 + q], uq = low ? other[q] : mine[NS / 2 + q];
                    const uint16_t o = TT::from_f32(mul_f32_rn(act == 1 ? silu_f32(gq) : gelu_tanh_f32(gq), uq));
                    if constexpr (NS == 2) o4[e] = o;
                    if (row < M && !by4) y[(size_t)row * hc + 8 * (NS * j + f) + p] = o;
                }
            }
            if constexpr (NS == 2) {
                const uint2 v = quad_turn16(o4[0] | (o4[1] << 16), o4[2] | (o4[3] << 16), lane);
                const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + quad;
                if (row < M && by4) *(uint2 *)(y + (size_t)row * hc + 8 * (NS * j + (low ? 0 : 1)) + p - quad) = v;
            }
        }
        return;
    }
    // row 16 mt + 4 kb + e, column 16 (NS j + f) + ni (of the copy)
    int col[NS];
#pragma unroll
    for (int f = 0; f < NS; ++f) {
        const int c = 16 * (NS * j + f) + ni;
        col[f] = c < N ? ggm_src_row(c, half) : -1;
    }
    if (gridDim.y > 1) {
#pragma unroll
        for (int t = 0; t < FT; ++t) {
            if constexpr (NS == 2) {  // (K slices are a choice of N % 4 == 0 only)
                const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + quad;
#pragma unroll
                for (int f = 0; f < NS; ++f) {
                    const float4_t v = quad_turn32(fin[t][f], lane);
                    if (row < M && col[f] >= 0) *(float4_t *)(part + ((size_t)blockIdx.y * M + row) * N + col[f] - quad) = v;
                }
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + e;
                if (row >= M) continue;
#pragma unroll
                for (int f = 0; f < NS; ++f)
                    if (col[f] >= 0) part[((size_t)blockIdx.y * M + row) * N + col[f]] = fin[t][f][e];
            }
        }
        return;
    }
    float bv[NS] = {};
    if (bias) {
#pragma unroll
        for (int f = 0; f < NS; ++f) bv[f] = col[f] >= 0 ? TT::to_f32(bias[col[f]]) : 0.f;
    }
    if constexpr (NS == 2) {
        if (by4) {
#pragma unroll
            for (int t = 0; t < FT; ++t)
#pragma unroll
                for (int f = 0; f < NS; ++f) {
                    uint32_t o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = TT::from_f32(fin[t][f][e] + bv[f]);
                    const uint2 v = quad_turn16(o[0] | (o[1] << 16), o[2] | (o[3] << 16), lane);
                    const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + quad;
                    if (row < M && col[f] >= 0) *(uint2 *)(y + (size_t)row * N + col[f] - quad) = v;
                }
            return;
        }
    }
#pragma unroll
    for (int t = 0; t < FT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + 16 * (KS == 1 ? t : FT * kq + t) + 4 * kb + e;
            if (row >= M) continue;
#pragma unroll
            for (int f = 0; f < NS; ++f)
                if (col[f] >= 0) y[(size_t)row * N + col[f]] = TT::from_f32(fin[t][f][e] + bv[f]);
        }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static bool ggm_format(int quant) {
    return quant == OXQ_GGUF_Q4_0 || quant == OXQ_GGUF_Q8_0 || quant == OXQ_GGUF_Q4_K || quant == OXQ_GGUF_Q6_K ||
           quant == OXQ_GGUF_Q4_1 || quant == OXQ_GGUF_Q5_0 || quant == OXQ_GGUF_Q5_1 || quant == OXQ_GGUF_Q5_K;
}
static bool ggm_narrow_format(int quant) { return quant == OXQ_GGUF_Q2_K || quant == OXQ_GGUF_Q3_K; }
static const char *ggm_name(int q) {
    switch (q) {
    case OXQ_GGUF_Q4_0: return "q4_0";
    case OXQ_GGUF_Q8_0: return "q8_0";
    case OXQ_GGUF_Q4_K: return "q4k";
    case OXQ_GGUF_Q4_1: return "q4_1";
    case OXQ_GGUF_Q5_0: return "q5_0";
    case OXQ_GGUF_Q5_1: return "q5_1";
    case OXQ_GGUF_Q5_K: return "q5k";
    case OXQ_GGUF_Q2_K: return "q2k";
    case OXQ_GGUF_Q3_K: return "q3k";
    default: return "q6k";
    }
}

bool gguf_mfma_eligible(const oxq_ctx *ctx, int quant, int64_t K, int64_t N) {
    if (!ggm_format(quant) || tune(ctx, OXQ_TUNE_GGUF_MFMA, 1) == 0) return false;
    // Rows that end inside a strip of 16 (a tensor-parallel shard, a padded vocabulary): from 2^20 weights on; below
    // the file-layout kernels take a launch's time as well.
    if (N % 16 != 0 && N * K < (1 << 20)) return false;
    return gguf_res_eligible(quant, K, (N + 15) & ~(int64_t)15);  // the same strips, chunks and 32-bit offsets
}
// Whether a layer of these activations holds the matrix-core copy.  bf16: always where it exists.  f32: from 2^20
// weights, beside the rotated copy of the vector GEMV; on smaller layers that one takes a launch's time.
// Q2_K and Q3_K layers hold it beside the rotated copy, which stays ahead at one row and on smaller layers.
bool gguf_mfma_layer(const oxq_ctx *ctx, int quant, int64_t K, int64_t N, int act_dtype) {
    if (ggm_narrow_format(quant))
        return tune(ctx, OXQ_TUNE_GGUF_MFMA, 1) != 0 && N * K >= (1 << 20) && gguf_res_eligible(quant, K, N) &&
               (act_dtype == OXQ_BF16 || act_dtype == OXQ_F32);
    return gguf_mfma_eligible(ctx, quant, K, N) && (act_dtype == OXQ_BF16 || (act_dtype == OXQ_F32 && N * K >= (1 << 20)));
}
// Whether such a layer does without the rotated copy: bf16, and f32 where OXQ_GGUF_MFMA is 2 (one copy fewer; what one and two
// rows then take stands below: up to 8 % more on layers of one round of strips).
bool gguf_mfma_alone(const oxq_ctx *ctx, int quant, int act_dtype) {
    return !ggm_narrow_format(quant) && (act_dtype == OXQ_BF16 || tune(ctx, OXQ_TUNE_GGUF_MFMA, 1) == 2);
}
// f32 rows of a layer that has both copies: the vector GEMV's arithmetic grows with the rows, and it is slow on many short strips, on
// a K that leaves its sixteen waves little or three chunks each, of which it works off four; the matrix cores take four rows as
// one.  us on the rotated / the matrix-core copy, Q4_K, 1 / 2 / 4 / 8 rows: 4096 x 4096 4.5 / 5.2 / 6.5 / 12.7 against 4.7 / 5.6 / 5.9 / 8.7,
// 14336 x 4096 11.5 / 14.1 / 17.8 / 35.2 against 11.0 / 13.7 / 15.1 / 22.0.  1 / 2 rows: 1024 x 4096 4.4 / 5.2 against 3.3 / 3.3 (Q6_K 4.5 / 5.5 against
// 3.6 / 3.7), 1536 x 4096 4.4 / 5.2 against 3.5 / 3.7, 2048 x 4096 4.3 / 5.0 against 4.0 / 4.3 (Q6_K 4.4 / 5.2 against 4.5 / 4.8, Q4_1 4.0 / 4.8
// against 4.5 / 4.5), 3072 x 8192 7.2 / 8.9 against 5.9 / 7.0, 4096 x 8192 7.6 / 9.3 against 7.3 / 8.7 (Q6_K 8.7 against 9.5), 6144 x 4096
// 6.7 / 8.2 against 5.7 / 7.0 (Q6_K 7.9 / 8.8 against 7.1 / 8.4), 5120 x 4096 5.6 / 6.8 against 5.3 / 6.3 (Q4_1 5.3 / 6.3 against 5.8 / 6.3).
bool gguf_f32_on_mfma(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N) {
    if (M >= 3) return true;
    const bool many = ceil_div(N, (int64_t)16) > (ctx->num_cus > 0 ? ctx->num_cus : 256), three = K > 4096 && K <= 6144;
    const bool pairs = quant == OXQ_GGUF_Q4_1 || quant == OXQ_GGUF_Q5_1;
    if (M == 2) return many || K <= 2048 || K >= 8192 || (three && !pairs);
    return K < 2048 || (many && K <= 3072) || ((K == 2048 || three) && quant != OXQ_GGUF_Q6_K && !pairs) || (three && K > 5120);
}
// Rows of a layer that holds both copies: whether they run on the matrix-core one.  Q2_K and Q3_K, us on the rotated / the
// matrix-core copy: 4096 x 4096 bf16 3 rows 6.7 / 5.2, 2 rows 5.0 / 5.2 (Q3_K 5.6 / 5.4), 1024 x 5056 2 rows 7.2 / 3.8, 14336 x 4096
// 14.3 / 12.5, 6144 x 4096 8.4 / 6.5, 2048 x 4096 5.1 / 4.1; f32 3 rows 6.5 / 6.5, 18.2 / 15.9 at 14336 x 4096, 8 rows 12.8 / 9.6, 36 / 26, but
// 2 rows 12.6 / 15.9.
bool gguf_rows_on_mfma(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N, int act_dtype) {
    const bool many = ceil_div(N, (int64_t)16) > (ctx->num_cus > 0 ? ctx->num_cus : 256);
    if (ggm_narrow_format(quant)) return act_dtype == OXQ_BF16 ? M >= 3 || (M == 2 && (many || K <= 3072 || K > 4096 || quant == OXQ_GGUF_Q3_K)) : M >= 3 && M <= 8;
    return act_dtype == OXQ_BF16 || gguf_f32_on_mfma(ctx, quant, M, K, N);
}
size_t gguf_mfma_bytes(int quant, int64_t K, int64_t N) {
    if (quant == OXQ_GGUF_Q3_K) return (size_t)N * (size_t)(K / 256) * 114;  // its scales are a byte each
    return gguf_res_bytes(quant, K, (N + 15) & ~(int64_t)15);
}

int launch_gguf_mfma_repack(oxq_ctx *ctx, hipStream_t s, int quant, const uint8_t *w, void *pw, int64_t K, int64_t N,
                            int64_t gate_half) {
    const size_t threads = (size_t)ceil_div(N, 16) * (K / 128) * 64;
    dim3 grid((unsigned)ceil_div((int64_t)threads, 256)), block(256);
    char name[64];
    plan_name(name, sizeof name, "gguf_%s_mfma_repack", ggm_name(quant));
    set_plan(ctx, name, grid, block, 1, 1, 0);
    if (ctx->plan_only) return OXQ_OK;
    switch (quant) {
    case OXQ_GGUF_Q4_0: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q4_0>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q8_0: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q8_0>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q4_K: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q4_K>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q6_K: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q6_K>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q4_1: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q4_1>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_0: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q5_0>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_1: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q5_1>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_K: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q5_K>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q2_K: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q2_K>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q3_K: hipLaunchKernelGGL((ggm_repack_kernel<OXQ_GGUF_Q3_K>), grid, block, 0, s, w, (uint8_t *)pw, (int)K, (int)N, (int)gate_half); break;
    default: return fail(OXQ_ERR_UNSUPPORTED, "gguf repack: format %d has no matrix-core layout", quant);
    }
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

int launch_gguf_mfma_dequant(oxq_ctx *ctx, hipStream_t s, int quant, const void *pw, int64_t K, int64_t N, float *out_nk,
                             int64_t gate_half) {
    const size_t threads = (size_t)ceil_div(N, 16) * (K / 128) * 64;
    dim3 grid((unsigned)ceil_div((int64_t)threads, 256)), block(256);
    char name[64];
    plan_name(name, sizeof name, "gguf_%s_mfma_dequant", ggm_name(quant));
    set_plan(ctx, name, grid, block, 1, 1, 0);
    if (ctx->plan_only) return OXQ_OK;
    switch (quant) {
    case OXQ_GGUF_Q4_0: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q4_0>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q8_0: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q8_0>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q4_K: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q4_K>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q6_K: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q6_K>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q4_1: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q4_1>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_0: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q5_0>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_1: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q5_1>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    case OXQ_GGUF_Q5_K: hipLaunchKernelGGL((ggm_dequant_kernel<OXQ_GGUF_Q5_K>), grid, block, 0, s, (const uint8_t *)pw, out_nk, (int)K, (int)N, (int)gate_half); break;
    default: return fail(OXQ_ERR_UNSUPPORTED, "gguf dequant: format %d has no matrix-core layout", quant);
    }
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

template <int FMT, int MT, int XQ, int NW, int NS, bool XF32, int NL>
static int ggm_launch(hipStream_t s, dim3 grid, const GgufProblem &p, float *ws, int cslice) {
    static LdsGrant lds_grant;  // one per instantiation
    constexpr auto kernel = [] {
        if constexpr (NL > 0) return &ggm_short_kernel<FMT, MT, XQ, NW, NS, XF32, NL>;
        else return &ggm_kernel<FMT, MT, XQ, NW, NS, XF32>;
    }();
    const size_t lds = (size_t)NW * MT * 4096;
    OXQ_HIP_CHECK(lds_grant.ensure((const void *)kernel, lds));
    hipLaunchKernelGGL(kernel, grid, dim3(NW * 64), lds, s, (const uint16_t *)p.x, p.w, (const uint16_t *)p.bias, (uint16_t *)p.y, ws,
                       (int)p.M, (int)p.K, (int)p.N, cslice, p.act);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <int FMT, int MT, int XQ, int NW, int NS, bool XF32 = false>
static int ggm_go(hipStream_t s, dim3 grid, const GgufProblem &p, float *ws, int cslice) {
    if (cslice <= NW) return ggm_launch<FMT, MT, XQ, NW, NS, XF32, 1>(s, grid, p, ws, cslice);
    if (cslice <= 2 * NW) return ggm_launch<FMT, MT, XQ, NW, NS, XF32, 2>(s, grid, p, ws, cslice);
    return ggm_launch<FMT, MT, XQ, NW, NS, XF32, 0>(s, grid, p, ws, cslice);
}
template <int FMT, int MT, int XQ, int NW, int NS>
static int ggm_f32_go(hipStream_t s, dim3 grid, const GgufProblem &p, int cslice) {
    return ggm_go<FMT, MT, XQ, NW, NS, true>(s, grid, p, nullptr, cslice);
}
template <int FMT>
static int ggm_f32_by_shape(hipStream_t s, dim3 grid, const GgufProblem &p, int cslice, int mt, int ns) {
    if constexpr (ggm_narrow<FMT>) {
        if (ns == 4) return mt == 2 ? ggm_f32_go<FMT, 2, 4, 8, 4>(s, grid, p, cslice) : ggm_f32_go<FMT, 1, 2, 8, 4>(s, grid, p, cslice);
        return mt == 2 ? ggm_f32_go<FMT, 2, 4, 8, 1>(s, grid, p, cslice) : ggm_f32_go<FMT, 1, 2, 8, 1>(s, grid, p, cslice);
    } else {
    if (ns == 4) {
        if (p.M == 1) return ggm_f32_go<FMT, 1, 1, 8, 4>(s, grid, p, cslice);
        return mt == 2 ? ggm_f32_go<FMT, 2, 4, 8, 4>(s, grid, p, cslice) : ggm_f32_go<FMT, 1, 2, 8, 4>(s, grid, p, cslice);
    }
    if (mt == 2) return ggm_f32_go<FMT, 2, 4, 8, 1>(s, grid, p, cslice);
    return p.M == 1 ? ggm_f32_go<FMT, 1, 1, 8, 1>(s, grid, p, cslice) : ggm_f32_go<FMT, 1, 2, 8, 1>(s, grid, p, cslice);
    }
}

template <int FMT>
static int ggm_by_shape(hipStream_t s, dim3 grid, const GgufProblem &p, float *ws, int cslice, int mt, int xq, int nw, int ns) {
    if constexpr (ggm_narrow<FMT>) {  // 2 - 8 rows (gguf_mfma_takes)
        if (ns == 4) return xq == 1 ? ggm_go<FMT, 1, 1, 8, 4>(s, grid, p, ws, cslice) : ggm_go<FMT, 1, 2, 8, 4>(s, grid, p, ws, cslice);
        if (nw == 8) return xq == 1 ? ggm_go<FMT, 1, 1, 8, 1>(s, grid, p, ws, cslice) : ggm_go<FMT, 1, 2, 8, 1>(s, grid, p, ws, cslice);
        return xq == 1 ? ggm_go<FMT, 1, 1, 16, 1>(s, grid, p, ws, cslice) : ggm_go<FMT, 1, 2, 16, 1>(s, grid, p, ws, cslice);
    } else {
    if (ns == 4) {  // 8 waves: four strips' quants in flight take the registers of two waves of a 16-wave workgroup
        if (mt == 2) return ggm_go<FMT, 2, 8, 8, 4>(s, grid, p, ws, cslice);
        if (xq == 1) return ggm_go<FMT, 1, 1, 8, 4>(s, grid, p, ws, cslice);
        if (xq == 2) return ggm_go<FMT, 1, 2, 8, 4>(s, grid, p, ws, cslice);
        return ggm_go<FMT, 1, 4, 8, 4>(s, grid, p, ws, cslice);
    }
    if (mt == 2) return ggm_go<FMT, 2, 8, 8, 1>(s, grid, p, ws, cslice);
    if (nw == 8) {
        if (xq == 1) return ggm_go<FMT, 1, 1, 8, 1>(s, grid, p, ws, cslice);
        if (xq == 2) return ggm_go<FMT, 1, 2, 8, 1>(s, grid, p, ws, cslice);
        return ggm_go<FMT, 1, 4, 8, 1>(s, grid, p, ws, cslice);
    }
    if (xq == 1) return ggm_go<FMT, 1, 1, 16, 1>(s, grid, p, ws, cslice);
    if (xq == 2) return ggm_go<FMT, 1, 2, 16, 1>(s, grid, p, ws, cslice);
    return ggm_go<FMT, 1, 4, 16, 1>(s, grid, p, ws, cslice);
    }
}

// A wide layer (768 strips or more) gives a workgroup four neighbouring strips: every strip of a workgroup re-reads
// the rows of x, which outweighs the weights from a few rows on, and 224 workgroups of 64 columns fill the chip
// as 896 of 16 do not (three and a half rounds).
static int ggm_strips(const oxq_ctx *ctx, int64_t N) {
    const int v = tune(ctx, OXQ_TUNE_GGUF_MFMA_NS, 0);
    const int64_t strips = ceil_div(N, 16);
    if (v == 1 || v == 4) return strips % v == 0 ? v : 1;
    return (strips >= 768 && strips % 4 == 0) ? 4 : 1;
}

// rows of x a launch of the matrix-core kernel takes (more go to the tile matmul on the file layout)
bool gguf_mfma_takes(const oxq_ctx *ctx, int quant, int64_t M, int64_t, int act_dtype) {
    // the decode range, whose weights stay unrounded; more rows go to the prefill kernel, whose rounded weights the tile
    // matmul on the file layout has
    if (ggm_narrow_format(quant)) return M >= 1 && M <= 8;
    if (act_dtype == OXQ_F32) return M >= 1;  // row tiles of eight: there is no other kernel for more f32 rows
    return act_dtype == OXQ_BF16 && M >= 1 && M <= tune(ctx, OXQ_TUNE_GGUF_MFMA_MAX_M, 32);
}

// p.w is the matrix-core copy; p.act: 0, or 1 + the gated activation of a fused gate|up layer, whose y is [M, N / 2].
// More rows than gguf_mfma_takes allows run as row tiles of the grid (every tile reads the weights again: the
// callers send such calls elsewhere where they can).
int launch_gguf_mfma(oxq_ctx *ctx, hipStream_t s, const GgufProblem &p) {
    const bool f32 = p.act_dtype == OXQ_F32;
    const int tile = f32 ? 4 : 16;  // rows of x a matrix-core tile takes
    if (p.M > 65535 * 2 * tile) {  // more row tiles than a grid dimension has: that many at a time
        const int64_t most = 65535 * 2 * tile, elem = f32 ? 4 : 2;
        uint32_t launches = 0;
        for (int64_t m0 = 0; m0 < p.M; m0 += most) {
            GgufProblem q = p;
            q.M = std::min(most, p.M - m0);
            q.x = (const uint8_t *)p.x + m0 * p.K * elem;
            q.y = (uint8_t *)p.y + m0 * (p.act ? p.N / 2 : p.N) * elem;
            const int rc = launch_gguf_mfma(ctx, s, q);
            if (rc != OXQ_OK) return rc;
            ++launches;
        }
        ctx->plan.launches = launches;
        return OXQ_OK;
    }
    const int ns = ggm_strips(ctx, p.N);
    const int mt = p.M > tile ? 2 : 1;
    const int rows = (int)std::min<int64_t>(p.M, tile * mt);
    const int xq = rows <= 4 ? 1 : rows <= 8 ? 2 : 4;
    // 16 waves split a strip's chunks where that leaves a wave two to three of them; from 64 chunks on 8 waves with
    // twice the run each measured 3 - 8 % faster (8192 x 4096 at one row, Q4_0 / Q4_K / Q6_K: 5.38 / 5.89 / 7.61
    // against 5.87 / 6.30 / 8.11 us).  Two row tiles or four strips need more than the 128 registers a wave of a
    // 16-wave workgroup has.
    const int64_t chunks = p.K / 128;
    // 16-wave workgroups are one a CU: more strips than CUs would take a second round of them (2048 x 8192 at one row
    // of bf16 / f32, Q4_K: 6.3 / 6.1 -> 4.4 / 4.7 us).  f32 rows: 8 waves are as fast or faster everywhere.
    const bool one_round = ceil_div(p.N, (int64_t)16) <= (ctx->num_cus > 0 ? ctx->num_cus : 256);
    const int nw = (chunks < 16 || chunks >= 64 || mt == 2 || ns == 4 || f32 || !one_round || tune(ctx, OXQ_TUNE_GGR_WAVES, 16) == 8) ? 8 : 16;
    dim3 grid((unsigned)ceil_div(p.N, (int64_t)16 * ns), 1, (unsigned)ceil_div(p.M, (int64_t)tile * mt));
    char name[64];
    plan_name(name, sizeof name, "gguf_%s_mfma_%s_mt%d%s%s", ggm_name(p.quant), f32 ? "f32" : "bf16", mt, ns == 4 ? "_n64" : "", p.act ? "_act" : "");
    set_plan(ctx, name, grid, dim3(nw * 64), 1, 1, 0);
    if (ctx->plan_only) return OXQ_OK;
    if (!f32 && p.act_dtype != OXQ_BF16) return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: activations must be BF16 or F32");
    if (ggm_narrow_format(p.quant) && (p.act || !gguf_mfma_takes(ctx, p.quant, p.M, p.N, p.act_dtype)))
        return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: %s takes up to 8 rows", ggm_name(p.quant));
    if (f32 && p.act) return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: a fused activation needs BF16");
    if ((uintptr_t)p.x & 15) return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: x must be 16-byte aligned");
    if ((uint64_t)16 * mt * (uint64_t)p.K * 2 >= (1ull << 31)) return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: K too large");
    if (gguf_res_bytes(p.quant, p.K, 16) * (uint64_t)ns >= (1ull << 31)) return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: K too large");
    const int cslice = (int)(p.K / 128);
#define OXQ_GGM(F) \
    case F: return f32 ? ggm_f32_by_shape<F>(s, grid, p, cslice, mt, ns) : ggm_by_shape<F>(s, grid, p, nullptr, cslice, mt, xq, nw, ns)
    switch (p.quant) {
        OXQ_GGM(OXQ_GGUF_Q4_0);
        OXQ_GGM(OXQ_GGUF_Q8_0);
        OXQ_GGM(OXQ_GGUF_Q4_K);
        OXQ_GGM(OXQ_GGUF_Q6_K);
        OXQ_GGM(OXQ_GGUF_Q4_1);
        OXQ_GGM(OXQ_GGUF_Q5_0);
        OXQ_GGM(OXQ_GGUF_Q5_1);
        OXQ_GGM(OXQ_GGUF_Q5_K);
        OXQ_GGM(OXQ_GGUF_Q2_K);
        OXQ_GGM(OXQ_GGUF_Q3_K);
    default: return fail(OXQ_ERR_UNSUPPORTED, "gguf matrix-core matmul: format %d", p.quant);
    }
#undef OXQ_GGM
}

// How a bf16 layer's matrix-core copy runs more rows than one launch of the integer kernel's two row tiles takes (33 and
// more): ks = 1 | 4: the prefill kernel, eight | two waves of 64 columns a workgroup (4: K split inside it, and over
// `slices` workgroups); ks = -1: the integer kernel in row tiles of 32; 0: the tile matmul on the file layout (gguf_mm).
//
// From 2^20 weights the cheapest of these by estimate, in us (fitted on one box to 4096 x 4096, 14336 x 4096, 5120 x
// 1408, 3072 x 7424, 2048 x 1024, 4096 x 14336 and 4096 x 28672 at 33 - 512 rows in Q4_K, Q6_K and Q8_0; the five- and six-bit
// formats' rounds again at 512 and 2048 rows of 4096 x 4096 when their conversion changed):
//   integer row tiles   2.6 + chunks a wave x `chunk` x rounds of 256 workgroups (four strips each: 2.5 x).  Ahead where the
//                       tiles fit one round: 2048 x 1024 at 128 rows 9.7 -> 5.3 us, 5120 x 1408 at 64 rows 12.0 -> 10.5
//   two waves           rounds of workgroups x (4.5 + K rounds of four chunks x `round`), and with K slices a second launch of
//                       3.5 us + the partials' bytes at 4.2 TB/s.  14336 x 4096 Q4_K at 33 / 128 / 256 rows 31.8 / 57.8 / 86 ->
//                       20.9 / 30.7 / 53 us (7, 4 and 2 slices), 4096 x 14336 at 64 rows 28.5 -> 23.5 (2 slices)
//   eight waves         rounds of workgroups (a last one on at most three quarters of the CUs 0.95) x chunks x `wide` + 5
//   128 rows            rounds of workgroups x (7 + chunks x `wide128`), and of 128 columns x (7 + K rounds of two chunks x `pair128`) with the
//                       sum of K slices as above; fitted to 4096 x 4096, 4096 x 14336, 14336 x 4096, 2560 x 3072 and 1536 x 6400 at 128 -
//                       2048 rows in Q4_K, Q8_0, Q6_K and Q3_K.  On 45 other layers of ten formats at 65 - 4000 rows, every form forced
//                       (130 calls): within 4 % of the fastest at 117, within 10 % at 125; the others are Q2_K and Q3_K calls that
//                       stay on the file layout
// (The rounds of eight waves are older than the numbering of tiles without gaps.  With column groups that are no multiple of eight, 36 layers of six
// formats, 180 calls of 256 - 4000 rows: within 3 % of the faster form at 167, within 8 % at 179.)
// The file layout's matmul is not ahead of all of these there.  It is for some calls of Q2_K and Q3_K, whose 9 - 32 rows come
// here too: where it has 400 tiles of 64 x 64 and more it runs at 400 T/s (Q3_K 15 % less) behind 6 us; with fewer it is ahead
// where K or the layer is short (Q2_K, us, file layout / here: 1024 x 5056 at 16 rows 6.9 / 8.8, 4096 x 1024 6.9 / 8.1, 2816 x
// 6528 10.7 / 11.1; elsewhere 4096 x 4096 at 16, 48, 101, 512 rows 10.0 / 9.2, 15.5 / 13.0, 24 / 17.6, 46 / 32,
// 14336 x 4096 23 / 16, 38 / 22, 68 / 33, 149 / 99, 9984 x 21056 at 16 rows 61 / 42, Q3_K 79 / 42).  On 71 other layers (K 1024 -
// 14336, N 512 - 19200, 9 - 2000 rows, 497 calls, every form of 64 rows forced): 0.79 x the file layout's time, none of the 342 calls that
// come here behind it by 3 %.  With the forms of 128 rows it is ahead from fewer weights above 512 rows (Q3_K 5888 x 512 at 779 rows
// 30 / 21.5, Q2_K 3072 x 1152 at 656 31.5 / 21.2, Q3_K 2816 x 704 at 704 19.2 / 20.0) and by the bare estimate at 400 tiles (Q2_K
// 1536 x 5504 at 346 24.6 / 20.8); 31 layers, 124 calls at 49 - 4000 rows: 1.7 % behind the fastest form together, 3.4 % before.
// Smaller layers compare it with the unsliced forms only, in rounds of 256 workgroups of 64 rows x 512 columns: 0.17 + 1.45 w
// (1.3 w for the five- and six-bit formats).
// OXQ_GGUF_GEMM_MIN_M: unset = by cost, 0 = never, n = the eight-wave form from n rows on whatever the cost;
// OXQ_GGUF_GEMM_KS = 4 | 1: always | never the two-wave form, 8 | 2: the form of 128 rows and 256 | 128 columns;
// OXQ_GGUF_GEMM_SLICES = n: that many slices of the two-wave form.
struct GgmGemmForm {
    int ks, slices;
    int rows = 64;  // of a workgroup
};
struct GgmCost {
    double chunk, round, wide, wide128, pair128;
};
static GgmCost ggm_cost(int quant) {
    switch (quant) {
    case OXQ_GGUF_Q4_0: case OXQ_GGUF_Q4_1: case OXQ_GGUF_Q4_K: return {1.45, 2.9, 2.6, 1.80, 1.94};
    case OXQ_GGUF_Q8_0: return {1.6, 2.9, 2.9, 1.78, 1.90};
    case OXQ_GGUF_Q6_K: return {1.75, 3.6, 3.4, 2.15, 2.38};
    case OXQ_GGUF_Q2_K: case OXQ_GGUF_Q3_K: return {0.0, 3.5, 3.2, 1.90, 2.25};  // `round`: of 64 rows, below of fewer
    default: return {1.6, 3.3, 3.0, 1.85, 2.04};  // Q5_0, Q5_1, Q5_K
    }
}
// sliced: whether the caller can take K slices, whose partial sums a second launch adds from the workspace.  One that cannot (a copy
// that lies there itself) chooses among whole sums of 128 rows; slices of 64 rows still win over them, and it then takes another kernel.
static GgmGemmForm gguf_gemm_form(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N, int act_dtype, bool sliced) {
    const int64_t v = tune(ctx, OXQ_TUNE_GGUF_GEMM_MIN_M, -1);
    const bool narrow = ggm_narrow_format(quant);
    if (v == 0 || act_dtype != OXQ_BF16 || !(narrow ? M > 8 : ggm_format(quant) && M > 32)) return {0, 1};
    const int ks = tune(ctx, OXQ_TUNE_GGUF_GEMM_KS, 0);
    if (ks == 4) return {N % 64 == 0 ? 4 : 0, 1};
    if (ks == 2 || ks == 8) return {ks == 2 ? 2 : 1, 1, 128};
    if (v > 0) return {N % 64 == 0 && M >= v ? 1 : 0, 1};
    const double cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    const int64_t row_tiles = ceil_div(M, (int64_t)64), groups = ceil_div(N, (int64_t)64), chunks = K / 128;
    const double w64 = (double)(ceil_div(groups, (int64_t)8) * row_tiles) / cus;
    const double whole = std::floor(w64), rest = w64 - whole;
    double r64 = whole + (rest <= 0.0 ? 0.0 : rest <= 0.75 ? 0.95 : 1.0);
    const int64_t mid_wgs = ceil_div(groups, (int64_t)2) * row_tiles;
    if (N * K < (1 << 20)) {
        if (N % 64 != 0) return {0, 1};
        const bool light = quant == OXQ_GGUF_Q4_0 || quant == OXQ_GGUF_Q4_1 || quant == OXQ_GGUF_Q4_K || quant == OXQ_GGUF_Q8_0;
        const double c_mid = ks == 1 ? 1e30 : std::ceil((double)mid_wgs / cus) * 0.31;
        // (Q8_0's 34-byte blocks make the file layout's matmul 1.2 - 1.35 x the 4-bit formats' at the same shape)
        const double c_file = 0.17 + (quant == OXQ_GGUF_Q8_0 ? 1.75 : light ? 1.45 : 1.3) * w64;
        if (c_file <= std::min(r64, c_mid)) return {0, 1};
        return {c_mid < r64 ? 4 : 1, 1};
    }
    GgmCost c = ggm_cost(quant);
    // whole rounds of the workgroups that have a tile (us, idle ones counted / not: Q3_K 2816 x 2304 at 2871 rows, file layout, 113 / 76, Q2_K
    // 4352 x 12544 at 576 140 / 110, Q3_K 3840 x 8576 at 1718, two strips, 251 / 198)
    if (narrow) r64 = std::ceil(w64);
    if (narrow && M <= 48) c.round = M <= 16 ? 2.2 : M <= 32 ? 2.7 : 3.1;
    GgmGemmForm best = {1, 1};
    double least = r64 * ((double)chunks * c.wide + 5.0);
    if (ks != 1) {
        const int64_t given = tune(ctx, OXQ_TUNE_GGUF_GEMM_SLICES, 0);
        const int64_t most = N % 4 == 0 ? std::min<int64_t>(ceil_div(chunks, (int64_t)4), 64) : 1;  // (the second launch adds four columns a thread)
        for (int64_t S = 1; S <= most; ++S) {
            if (given > 0 && S != std::min(given, most)) continue;
            const int64_t rounds = ceil_div(ceil_div(chunks, S), (int64_t)4);
            if (ceil_div(chunks, 4 * rounds) != S || (S > 1 && (uint64_t)(S * M) * (uint64_t)N * 4 > ctx->workspace_bytes)) continue;
            double t = std::ceil((double)(mid_wgs * S) / cus) * (4.5 + (double)rounds * c.round);
            if (S > 1) t += 3.5 + ((double)S * 8.0 + 2.0) * (double)M * (double)N / 4.2e6;
            if (t < least || given > 0) least = given > 0 ? 0.0 : t, best = {4, (int)S};
        }
    }
    // 128 rows x 256 | 128 columns a workgroup
    if (!tune_given(ctx, OXQ_TUNE_GGUF_GEMM_SLICES) && ks == 0 && K < (1 << 22)) {
        const int64_t row_tiles128 = ceil_div(M, (int64_t)128);
        const double t8 = std::ceil((double)(ceil_div(N, (int64_t)256) * row_tiles128) / cus) * (7.0 + (double)chunks * c.wide128);
        if (t8 < least) least = t8, best = {1, 1, 128};
        const int64_t wgs = ceil_div(N, (int64_t)128) * row_tiles128, most = sliced && N % 4 == 0 ? std::min<int64_t>(ceil_div(chunks, (int64_t)2), 8) : 1;
        for (int64_t S = 1; S <= most; ++S) {
            const int64_t rounds = ceil_div(ceil_div(chunks, S), (int64_t)2);
            if (ceil_div(chunks, 2 * rounds) != S || (S > 1 && (uint64_t)(S * M) * (uint64_t)N * 4 > ctx->workspace_bytes)) continue;
            double t = std::ceil((double)(wgs * S) / cus) * (7.0 + (double)rounds * c.pair128);
            if (S > 1) t += 3.5 + ((double)S * 8.0 + 2.0) * (double)M * (double)N / 4.2e6;
            if (t < least) least = t, best = {2, (int)S, 128};
        }
    }
    if (narrow) {
        if (v > 0 || ks || tune(ctx, OXQ_TUNE_GGUF_GEMM_SLICES, 0) > 0) return best;
        const int64_t size = N * K;
        const double file = 6.0 + (double)(row_tiles * 64) * (double)size / 2e8 * (quant == OXQ_GGUF_Q3_K ? 1.15 : 1.0) * (M <= 16 ? 0.55 : M <= 32 ? 0.67 : 1.0);
        bool ahead;
        if (row_tiles * groups >= 400) ahead = least < file;
        else if (M > 64) ahead = size >= (M > 512 ? 1 << 21 : M > 128 ? 1 << 22 : 1 << 23);
        else ahead = K >= 3072 && (size >= 1 << 24 || (size >= 1 << 23 && (K >= 7168 || M > 32)));
        return ahead ? best : GgmGemmForm{0, 1};
    }
    const int ns = ggm_strips(ctx, N);
    const double int_wgs = (double)(ceil_div(N, (int64_t)16 * ns) * ceil_div(M, (int64_t)32));
    const double int_rounds = std::ceil(int_wgs / cus);
    if (2.6 + (double)ceil_div(chunks, (int64_t)8) * c.chunk * (ns == 4 ? 2.5 : 1.0) * (int_rounds > 1.0 ? 1.15 * int_rounds : 1.0) < least) best = {-1, 1};
    return best;
}
bool gguf_gemm_takes(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N, int act_dtype, bool sliced) {
    const GgmGemmForm f = gguf_gemm_form(ctx, quant, M, K, N, act_dtype, sliced);
    return f.ks > 0 && (sliced || f.slices == 1);
}
// A fused gate|up layer: the plain layer's form, which keeps its bits - but for slices of 64 rows, whose calls stay in the integer
// kernel's row tiles (few rows, weights not rounded).  The launch that adds slices of 128 rows runs the activation.
bool gguf_gemm_takes_act(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N, int act_dtype) {
    const GgmGemmForm f = gguf_gemm_form(ctx, quant, M, K, N, act_dtype, true);
    return N % 64 == 0 && f.ks > 0 && (f.slices == 1 || f.rows == 128);
}
// rows beyond gguf_mfma_takes that the integer kernel takes in row tiles
bool gguf_mfma_tiles(const oxq_ctx *ctx, int quant, int64_t M, int64_t K, int64_t N, int act_dtype) {
    return gguf_gemm_form(ctx, quant, M, K, N, act_dtype, true).ks < 0;
}

// Adds the K slices of a fused gate|up layer and runs its activation: columns n and hc + n of a row (file order), summed and rounded
// as splitk_reduce_kernel does it, then act(gate) * up as oxq_gated_activation.  What bounds it: the partials' bytes, as there.  A
// thread has four outputs.  The fused call, us, whole sums in one launch (which are not the plain layer's bits) -> slices and this: Q4_K
// 8192 x 4096 at 300 / 512 rows 49.1 / 49.6 -> 42.1 / 46.4, 6144 x 10752 at 74 38.4 -> 29.1, Q6_K 8192 x 4096 at 400 59.9 -> 50.2.
// hc is a multiple of 32, and the 8 S M hc bytes of partials fit the workspace: the index fits 32 bits.
__global__ __launch_bounds__(256) void ggm_act_reduce_kernel(const float *__restrict__ part, const uint16_t *__restrict__ bias,
                                                             uint16_t *__restrict__ y, unsigned quads, int hc, size_t total, int S, int act) {
    typedef BF16Traits TT;
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= quads) return;
    const unsigned row = i / (unsigned)(hc >> 2), n = (i - row * (unsigned)(hc >> 2)) * 4;
    const float *from = part + (size_t)row * 2 * hc + n;
    float4_t g = {0.f, 0.f, 0.f, 0.f}, u = g;
    for (int s0 = 0; s0 < S; s0 += 4) {
        float4_t vg[4], vu[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float *at = from + (size_t)(s0 + k) * total;
            vg[k] = s0 + k < S ? *(const float4_t *)at : float4_t{0.f, 0.f, 0.f, 0.f};
            vu[k] = s0 + k < S ? *(const float4_t *)(at + hc) : float4_t{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) g += vg[k], u += vu[k];  // slice order
    }
    uint32_t o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float a = g[c], b = u[c];
        if (bias) a += TT::to_f32(bias[n + c]), b += TT::to_f32(bias[hc + n + c]);
        a = TT::to_f32(TT::from_f32(a)), b = TT::to_f32(TT::from_f32(b));
        o[c] = TT::from_f32(mul_f32_rn(act == 1 ? silu_f32(a) : gelu_tanh_f32(a), b));
    }
    uint16_t *to = y + (size_t)row * hc + n;
    if (((uintptr_t)y & 7) == 0) {
        *(uint2 *)to = uint2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) to[c] = (uint16_t)o[c];
    }
}

template <int FMT, int MT, int KS, int NS = 4>
static int ggm_gemm_go(hipStream_t s, dim3 grid, const GgufProblem &p, float *part, int NG, int RT, int cslice) {
    static LdsGrant grant;  // one per instantiation
    const size_t lds = (size_t)2 * KS * 16 * MT * 256;
    OXQ_HIP_CHECK(grant.ensure((const void *)ggm_gemm_kernel<FMT, MT, KS, NS>, lds));
    hipLaunchKernelGGL((ggm_gemm_kernel<FMT, MT, KS, NS>), grid, dim3(512), lds, s, (const uint16_t *)p.x, p.w, (const uint16_t *)p.bias,
                       (uint16_t *)p.y, part, (int)p.M, (int)p.K, (int)p.N, NG, RT, p.act, cslice, (int)p.gate_half);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}
template <int FMT>
static int ggm_gemm_go_form(hipStream_t s, dim3 grid, const GgufProblem &p, float *part, int NG, int RT, int ks, int cslice, int rows) {
    if (rows == 128) return ks == 2 ? ggm_gemm_go<FMT, 8, 2, 2>(s, grid, p, part, NG, RT, cslice) : ggm_gemm_go<FMT, 8, 1, 2>(s, grid, p, part, NG, RT, cslice);
    if (ks == 1) return ggm_gemm_go<FMT, 4, 1>(s, grid, p, part, NG, RT, cslice);
    // up to 48 rows: the 64-row tile without its fourth row tile of MFMAs, and of x (14336 x 4096 at 48 rows, us: Q4_K 21.4 ->
    // 20.3, Q6_K 25.9 -> 24.5, Q8_0 23.3 -> 22.2)
    if constexpr (ggm_narrow<FMT>) {
        if (p.M <= 16) return ggm_gemm_go<FMT, 1, 4>(s, grid, p, part, NG, RT, cslice);
        if (p.M <= 32) return ggm_gemm_go<FMT, 2, 4>(s, grid, p, part, NG, RT, cslice);
    }
    return p.M <= 48 ? ggm_gemm_go<FMT, 3, 4>(s, grid, p, part, NG, RT, cslice) : ggm_gemm_go<FMT, 4, 4>(s, grid, p, part, NG, RT, cslice);
}

// p.w is the matrix-core copy; p.act as for launch_gguf_mfma; p.gate_half: the copy of a fused gate|up layer whose
// activation this call leaves out
int launch_gguf_gemm(oxq_ctx *ctx, hipStream_t s, const GgufProblem &problem, bool sliced) {
    GgufProblem p = problem;
    GgmGemmForm form = gguf_gemm_form(ctx, p.quant, p.M, p.K, p.N, p.act_dtype, sliced);
    if (form.ks <= 0) form = {1, 1};  // a caller that asks for this kernel gets it
    if (!sliced) form.slices = 1;
    const int act_after = form.slices > 1 ? p.act : 0;  // (gguf_gemm_takes_act)
    if (act_after) p.act = 0, p.gate_half = p.N / 2;
    const int ks = form.ks, spw = 8 / ks, rows = form.rows;
    const int64_t NG = ceil_div(ceil_div(p.N, (int64_t)(rows == 128 ? 32 : 64)), (int64_t)spw), RT = ceil_div(p.M, (int64_t)rows);
    const int64_t wgs = ks == 1 ? pk4g_workgroups(RT, NG) : RT * NG;
    if (wgs > 0x7FFFFFFF) return fail(OXQ_ERR_UNSUPPORTED, "gguf prefill matmul: m = %lld exceeds the grid", (long long)p.M);
    const int64_t chunks = p.K / 128;
    const int cslice = form.slices > 1 ? (int)(ceil_div(ceil_div(chunks, (int64_t)form.slices), (int64_t)ks) * ks) : (int)chunks;
    dim3 grid((unsigned)wgs, (unsigned)form.slices);
    // rows x column groups of the workgroup, and the waves that share K inside it
    char name[64], slices[16] = "";
    if (form.slices > 1) snprintf(slices, sizeof slices, "_s%d", form.slices);
    plan_name(name, sizeof name, "gguf_%s_gemm_bf16_r%dx%d%s%s%s", ggm_name(p.quant), rows, spw, ks == 4 ? "k4" : ks == 2 ? "k2" : "", slices,
             problem.act == 1 ? "_silu" : problem.act == 2 ? "_gelu" : "");
    set_plan(ctx, name, grid, dim3(512), form.slices, 1, form.slices > 1 ? (size_t)form.slices * p.M * p.N * 4 : 0);
    if (ctx->plan_only) {
        if (form.slices > 1) add_launch(ctx);
        return OXQ_OK;
    }
    if (p.act_dtype != OXQ_BF16) return fail(OXQ_ERR_UNSUPPORTED, "gguf prefill matmul: activations must be BF16");
    if ((uint64_t)rows * (uint64_t)p.K * 2 >= (1ull << 31)) return fail(OXQ_ERR_UNSUPPORTED, "gguf prefill matmul: K too large");
    if (((uintptr_t)p.x & 15) || ((uintptr_t)p.y & 1)) return fail(OXQ_ERR_UNSUPPORTED, "gguf prefill matmul: x must be 16-byte aligned");
    float *part = (float *)ctx->workspace;
    int rc;
#define OXQ_GGM(F) \
    case F: rc = ggm_gemm_go_form<F>(s, grid, p, part, (int)NG, (int)RT, ks, cslice, rows); break
    switch (p.quant) {
        OXQ_GGM(OXQ_GGUF_Q4_0);
        OXQ_GGM(OXQ_GGUF_Q8_0);
        OXQ_GGM(OXQ_GGUF_Q4_K);
        OXQ_GGM(OXQ_GGUF_Q6_K);
        OXQ_GGM(OXQ_GGUF_Q4_1);
        OXQ_GGM(OXQ_GGUF_Q5_0);
        OXQ_GGM(OXQ_GGUF_Q5_1);
        OXQ_GGM(OXQ_GGUF_Q5_K);
        OXQ_GGM(OXQ_GGUF_Q2_K);
        OXQ_GGM(OXQ_GGUF_Q3_K);
    default: return fail(OXQ_ERR_UNSUPPORTED, "gguf prefill matmul: format %d has no matrix-core layout", p.quant);
    }
#undef OXQ_GGM
    if (rc != OXQ_OK || form.slices == 1) return rc;
    if (!act_after) return launch_splitk_reduce(ctx, s, part, p.bias, p.y, p.M, p.N, form.slices, OXQ_BF16);
    add_launch(ctx);
    const unsigned quads = (unsigned)(p.M * (p.N / 8));
    hipLaunchKernelGGL(ggm_act_reduce_kernel, dim3((unsigned)ceil_div((int64_t)quads, (int64_t)256)), dim3(256), 0, s, part, (const uint16_t *)p.bias,
                       (uint16_t *)p.y, quads, (int)(p.N / 2), (size_t)p.M * p.N, form.slices, act_after);
    OXQ_HIP_CHECK(hipGetLastError());
    return OXQ_OK;
}

}  // namespace oxq
