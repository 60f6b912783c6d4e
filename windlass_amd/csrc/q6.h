// q6.h — f32 rows in six 6-bit floating-point pieces, the operands of the
// routed experts' GEMMs on gfx950's scaled matrix instruction (batched_gemm.h).
//
// v_mfma_scale_f32_16x16x128_f8f6f4 takes the MXFP4 weights as they lie in the
// native block (a lane's 16 bytes are its 32 values, its E8M0 byte the scale
// operand), so nothing is converted. The f32 activations run as 6-bit
// floating-point pieces (E2M3) per block of 32 values, x = sum of p_i 2^s_i:
// s_1 puts the block's largest value in (3.75, 7.5], each piece takes the
// nearest E2M3 value of what the pieces before it left, and the scales fall by
// 4, then 5 powers of two a piece, which is what a piece's rounding leaves (at
// most 1/4 after the first, 1/8 of its scale after the others). Six pieces leave
// at most 2^-29 of the block's largest value: full f32 precision down to 1/32 of
// it, 21 bits down to 1/256.
//
// That is enough for a block whose values are of one size. Where most lie far below
// a few, as beside the outlier channels of a trained model, weights that are zero at
// those few (MXFP4 rounds many to zero) leave a sum of the small ones alone; with five
// pieces such sums were off by 3e-6 of the largest output at 100 times, 1e-3 at 30000
// times, and six leave a 32nd of that. A row in which this may count therefore has
// two further pieces per block, in records of their own that the GEMMs run against
// the same weights, into the same sums: 2^-39 of the largest value, full f32
// precision down to 1/32768 of it. It may count where what six pieces leave of the
// wide blocks, some 2^-31 of the largest for each of 32 values, may exceed 2^-24.5 of
// the row's sum without their few large values (q6_more). The row's other blocks are
// in that sum: SwiGLU values of large gate values, half of them almost zero, make many
// blocks wide and lose nothing (a rule block by block took further pieces for them,
// and 64 tokens 755 to 940 us). Passes of such rows of at most 16 tokens have them
// beside the records, larger ones run twice as long (hidden 6144, inter 2048, 8 of 256
// experts, 12 columns 1000 times the rest in every token, with three bf16 pieces and
// now: 7 tokens 208 and 209 us, 64 563 and 553, 256 1012 and 1030, 1000 2345 and 2187,
// 4096 8152 and 7238).
//
// Why this format: measured on MI355X the instruction runs 8.5 PFLOP/s with 6-bit
// against 4-bit operands (bf16 2.43, 8-bit 4.8), so six pieces cost 0.6 of three
// bf16 pieces' matrix time, and with 4- and 6-bit operands its sums keep f32
// precision (a probe: exact while the terms span 2^21, as the f32 accumulator). The
// GEMMs that ran three bf16 pieces against weights converted to bf16 were bound by
// those MFMAs, the conversions and the LDS reads (12 KB per 16 tokens and 128
// columns, 9 KB here). The sixth piece of the gate/up inputs takes 1 % at 256
// tokens, 4 % at 1000 and 7 % at 4096 (1533 to 1601 and 4836 to 5180 us).
//
// A quantised row is a record per 128 columns (k tile) of 16-byte units c: c =
// 4p + g the first 16 bytes of piece p of block g, c = 4P + 2p + h the last 8
// bytes of piece p of blocks 2h and 2h + 1, c = 6P + h the scale bytes (8 per
// block, P used) of blocks 2h and 2h + 1: 608 bytes for P = 6, 224 for P = 2. A DMA
// into LDS takes eight units of each of eight rows.
#pragma once
#include "dev_common.h"
#include "internal.h"

namespace wl {

typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(6))) uint32_t u32x6;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(32))) float f32x32;

constexpr uint32_t kQP = 6, kQX = 2;  // pieces of a record, further pieces
constexpr uint32_t kQUnits = 6u * kQP + 2u;
static_assert(16u * kQUnits == kQRecord && 16u * (6u * kQX + 2u) == kQMore, "record sizes");
// bytes of a row of k columns
__host__ __device__ constexpr size_t q6_row_bytes(uint32_t k) { return (size_t)kQRecord * (k / 128u); }
__host__ __device__ constexpr size_t q6_more_bytes(uint32_t k) { return (size_t)kQMore * (k / 128u); }
// Where unit c of a record lies in the record of further pieces, whose pieces are
// read as the first of a record that has no others (or ~0: a zero unit).
__host__ __device__ constexpr uint32_t q6_more_unit(uint32_t c) {
    return c < 4u * kQX                                 ? c
           : c >= 4u * kQP && c < 4u * kQP + 2u * kQX ? c - 4u * kQP + 4u * kQX
           : c >= 6u * kQP && c < 6u * kQP + 2u       ? c - 6u * kQP + 6u * kQX
                                                      : ~0u;
}

// The largest magnitude of a block, as bits.
WL_DEV uint32_t q6_max(const f32x16& even, const f32x16& odd) {
    uint32_t mx = 0u;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        mx = max(mx, __float_as_uint(even[i]) & 0x7FFFFFFFu);
        mx = max(mx, __float_as_uint(odd[i]) & 0x7FFFFFFFu);
    }
    return mx;
}
// Whether a block of largest magnitude mx is wide: at most eight of its values are
// within 2^8 of the largest, and smaller ones are there.
WL_DEV bool q6_wide(const f32x16& even, const f32x16& odd, uint32_t mx) {
    const float m = __uint_as_float(mx), lim = m * 0x1p-8f;
    uint32_t n = 0u, zero = 0u;
#pragma unroll
    for (int i = 0; i < 16; i++) n += (fabsf(even[i]) >= lim ? 1u : 0u) + (fabsf(odd[i]) >= lim ? 1u : 0u);
    if (n > 8u || m < 0x1p-100f || !(m < INFINITY)) return false;
#pragma unroll
    for (int i = 0; i < 16; i++) zero += (even[i] == 0.f ? 1u : 0u) + (odd[i] == 0.f ? 1u : 0u);
    return n + zero < 32u;
}
// What a block adds to the test of a row with wide blocks (q6_more). big: the square
// of the largest value if the block is wide. rest: the sum of squares of the smaller
// ones; in other blocks that of the values under an eighth of the largest, if at most
// eight reach that (outliers, too), or of all.
struct QRange {
    double big, rest;
};
WL_DEV QRange q6_range(const f32x16& even, const f32x16& odd) {
    const uint32_t mx = q6_max(even, odd);
    const float m = __uint_as_float(mx), inv = __builtin_amdgcn_rcpf(m);
    if (m < 0x1p-100f || !(m < INFINITY)) return QRange{0.0, 0.0};
    const bool wide = q6_wide(even, odd, mx);
    float all = 0.f, s3 = 0.f, s8 = 0.f;
    uint32_t n3 = 0u;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        const float v = fabsf(i & 1 ? odd[i / 2] : even[i / 2]), a = v * inv, q = a * a;
        const bool l3 = a >= 0x1p-3f;
        all += q;
        s3 += l3 ? 0.f : q;
        s8 += v >= m * 0x1p-8f ? 0.f : q;
        n3 += l3 ? 1u : 0u;
    }
    const double m2 = (double)m * (double)m;
    return QRange{wide ? m2 : 0.0, m2 * (wide ? s8 : n3 <= 8u ? s3 : all)};
}
// From the row's sums.
WL_DEV bool q6_more(double big, double rest) { return big > 256.0 * rest; }
// The sum over a wave.
WL_DEV double wave_sum_f64(double x) {
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}
// Block g of a k tile: 32 values (even[i], odd[i] columns 2i and 2i + 1) of largest
// magnitude mx into its parts of the record at rec, or (MORE) its further pieces
// into theirs.
template <bool MORE>
WL_DEV void q6_store(uint8_t* rec, uint32_t g, f32x16 even, f32x16 odd, uint32_t mx) {
    // biased exponent of s_1: the largest value over it is in (3.75, 7.5]; large
    // enough that all scales of a record are normal powers of two (a block of values
    // under 2^-100 keeps what that leaves of it: to 2^-129)
    constexpr uint32_t kFirst = MORE ? kQP : 0u, kEnd = MORE ? kQP + kQX : kQP, PN = kEnd - kFirst;
    constexpr uint32_t lo = 5u * (kQP - 1u);
    uint32_t e = (mx >> 23) + ((mx & 0x7FFFFFu) > 0x700000u ? 1u : 0u);
    e = e < lo + 2u ? lo : e - 2u;
    const bool bad = mx >= 0x7F800000u;  // an infinity or a NaN: the E8M0 NaN, and NaN sums
    uint64_t sc = 0;
#pragma unroll
    for (uint32_t p = 0; p < kEnd; p++) {
        const uint32_t drop = p ? 5u * p - 1u : 0u, ep = e > drop ? e - drop : 1u;
        const float s = __uint_as_float(ep << 23);
        // Both conversions take several passes and must not write over what they
        // still have to read (a fifth piece whose result the compiler had put
        // over its scale came out wrong), so their operands stay live.
        const u32x6 q = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, s);
        asm volatile("" ::"v"(q), "v"(even), "v"(odd), "v"(s));
        if (p + 1u < kEnd) {
            const f32x32 y = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, s);
            asm volatile("" ::"v"(y), "v"(q), "v"(s));
#pragma unroll
            for (int i = 0; i < 16; i++) {
                even[i] -= y[2 * i];
                odd[i] -= y[2 * i + 1];
            }
        }
        if (p < kFirst) continue;
        const uint32_t pi = p - kFirst;
        sc |= (uint64_t)(bad ? 255u : ep) << (8u * pi);
        gst((u32x4*)(rec + 16u * (4u * pi + g)), u32x4{q[0], q[1], q[2], q[3]});
        gst((uint64_t*)(rec + 16u * (4u * PN + 2u * pi + (g >> 1)) + 8u * (g & 1u)), (uint64_t)q[4] | ((uint64_t)q[5] << 32));
    }
    gst((uint64_t*)(rec + 16u * (6u * PN + (g >> 1)) + 8u * (g & 1u)), sc);
}
// The 32 values at x (16-byte aligned), split into even and odd columns.
WL_DEV void q6_load(const float* x, f32x16& even, f32x16& odd) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const f32x4 v = *(const f32x4*)(x + 4 * i);
        even[2 * i] = v.x;
        odd[2 * i] = v.y;
        even[2 * i + 1] = v.z;
        odd[2 * i + 1] = v.w;
    }
}

}  // namespace wl
