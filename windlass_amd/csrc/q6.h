// q6.h — f32 rows in five 6-bit floating-point pieces, the operands of the
// routed experts' GEMMs on gfx950's scaled matrix instruction (batched_gemm.h).
//
// v_mfma_scale_f32_16x16x128_f8f6f4 takes the MXFP4 weights as they lie in the
// native block (a lane's 16 bytes are its 32 values, its E8M0 byte the scale
// operand), so nothing is converted. The f32 activations run as P 6-bit
// floating-point pieces (E2M3) per block of 32 values, x = sum of p_i 2^s_i:
// s_1 puts the block's largest value in (3.75, 7.5], each piece takes the
// nearest E2M3 value of what the pieces before it left, and the scales fall by
// 4, then 5 powers of two a piece, which is what a piece's rounding leaves (at
// most 1/4 after the first, 1/8 of its scale after the others). Five pieces
// leave at most 2^-24 of the block's largest value, an f32 rounding of it:
// enough for the normalised input of gate/up. The SwiGLU values within a block
// differ by more; six pieces (2^-29) keep full f32 precision down to 1/32 of
// the block's largest value, and down projections whose weights single out a
// small value stay within 1e-5 of it (tests/test_gpu_e8m0_corners.py).
//
// Why: measured on MI355X the instruction runs 8.5 PFLOP/s with 6-bit against
// 4-bit operands (bf16 2.43, 8-bit 4.8), so five or six pieces cost 0.5 to 0.6
// of the three bf16 pieces' matrix time, and with 4- and 6-bit operands its sums
// keep f32 precision (a probe: exact while the terms span 2^21, as the f32
// accumulator). The GEMMs that ran three bf16 pieces against weights converted
// to bf16 were bound by those MFMAs, the conversions and the LDS reads (12 KB
// per 16 tokens and 128 columns, 7.5 and 9 KB here).
//
// A quantised row is a record per 128 columns (k tile) of 16-byte units c: c =
// 4p + g the first 16 bytes of piece p of block g, c = 4P + 2p + h the last 8
// bytes of piece p of blocks 2h and 2h + 1, c = 6P + h the scale bytes (8 per
// block, P used) of blocks 2h and 2h + 1: 512 bytes for five pieces, 608 for
// six. A DMA into LDS takes eight units of each of eight rows.
#pragma once
#include "dev_common.h"

namespace wl {

typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(6))) uint32_t u32x6;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(32))) float f32x32;

constexpr uint32_t kQPUp = 5, kQPDown = 6;  // pieces of the gate/up inputs and of the SwiGLU values
__host__ __device__ constexpr uint32_t q6_units(uint32_t P) { return 6u * P + 2u; }
__host__ __device__ constexpr uint32_t q6_record(uint32_t P) { return 16u * q6_units(P); }
// bytes of a row of k columns
__host__ __device__ constexpr size_t q6_row_bytes(uint32_t P, uint32_t k) { return (size_t)q6_record(P) * (k / 128u); }

// Block g of a k tile: 32 values (even[i], odd[i] columns 2i and 2i + 1) into
// its parts of the record at rec.
template <uint32_t P>
WL_DEV void q6_store(uint8_t* rec, uint32_t g, f32x16 even, f32x16 odd) {
    uint32_t mx = 0u;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        mx = max(mx, __float_as_uint(even[i]) & 0x7FFFFFFFu);
        mx = max(mx, __float_as_uint(odd[i]) & 0x7FFFFFFFu);
    }
    // biased exponent of s_1: the largest value over it is in (3.75, 7.5]; large
    // enough that all scales are normal powers of two (a block of values under
    // 2^-100 keeps what that leaves of it)
    constexpr uint32_t drop[6] = {0u, 4u, 9u, 14u, 19u, 24u}, lo = drop[P - 1u] + 1u;
    uint32_t e = (mx >> 23) + ((mx & 0x7FFFFFu) > 0x700000u ? 1u : 0u);
    e = e < lo + 2u ? lo : e - 2u;
    const bool bad = mx >= 0x7F800000u;  // an infinity or a NaN: the E8M0 NaN, and NaN sums
    uint64_t sc = 0;
#pragma unroll
    for (uint32_t p = 0; p < P; p++) {
        const uint32_t ep = e - drop[p];
        const float s = __uint_as_float(ep << 23);
        // Both conversions take several passes and must not write over what they
        // still have to read (a fifth piece whose result the compiler had put
        // over its scale came out wrong), so their operands stay live.
        const u32x6 q = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, s);
        asm volatile("" ::"v"(q), "v"(even), "v"(odd), "v"(s));
        if (p + 1u < P) {
            const f32x32 y = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, s);
            asm volatile("" ::"v"(y), "v"(q), "v"(s));
#pragma unroll
            for (int i = 0; i < 16; i++) {
                even[i] -= y[2 * i];
                odd[i] -= y[2 * i + 1];
            }
        }
        sc |= (uint64_t)(bad ? 255u : ep) << (8u * p);
        gst((u32x4*)(rec + 16u * (4u * p + g)), u32x4{q[0], q[1], q[2], q[3]});
        gst((uint64_t*)(rec + 16u * (4u * P + 2u * p + (g >> 1)) + 8u * (g & 1u)), (uint64_t)q[4] | ((uint64_t)q[5] << 32));
    }
    gst((uint64_t*)(rec + 16u * (6u * P + (g >> 1)) + 8u * (g & 1u)), sc);
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
