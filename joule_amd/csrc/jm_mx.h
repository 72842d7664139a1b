// Operands of the fp6 matrix-core products (gfx950,
// v_mfma_scale_f32_32x32x64_f8f6f4) of the dense expert branch and the
// plugin product (jm_mfma.hip), and the encoding of activations for them.
//
// A 6-bit float e2m3 with code n = 0..16 is n / 8 (the subnormals and the
// first binade are one linear range, 16 the next binade's first), bit 5 its
// sign.  So an unsigned Q4 nibble q, zero-extended, is the operand q / 8, and a
// balanced digit -16..15 of base 32 is an operand as well.  An activation group
// (the columns one weight scale covers) is written as integers
// a_j = rint(x_j / 2^E), |a_j| <= 507375 = 15 (1 + 32 + 32^2 + 32^3), with E the
// smallest exponent that allows it: a value is held to half a step, at most
// max|x| / 507374.  (Sixteen-valued digits under one sign, the form before, held
// it to max|x| / 65534.)  The 4 digits of a_j go to 4 planes; the products of a
// plane are scaled by 2^E 32^plane in the matrix core (E8M0 block scales), so
// that 4 accumulating instructions, starting from the group's correction
// -8 sum_j a_j 2^E (the -8 of the Q4 code), give sum_j a_j (q_j - 8) 2^E in
// float32.
//
// The corrections and products are all taken 2^F6_SHIFT times smaller, and the
// kernels' results that much larger: 8 sum|x| of a group may pass the float32
// range where its sum over the weights does not.  At the other end E stops at
// -126 (the third bf16 term of a correction, 2^(E - 2) 8 / 2, is normal
// there): groups under 2^-108 lose digits one by one, to 16 bits at 2^-111.
//
// Lane layout (checked on the device): A[i][k] at lane i % 32, B[k][n] at
// lane n % 32, k = 32 (l / 32) + j, field j at bit 6 j of 6 dwords; D
// register v of lane l = (i = 8 (v / 4) + 4 (l / 32) + v % 4, n = l % 32).
// The order of the 64 columns within an instruction is free as long as both
// sides have it: it is the one f6_spread gives.
//
// Record of one row of K columns: per 64 columns (a stage) 192 bytes = 6
// pieces x 2 lane halves x 16 bytes; piece o = 0..3 the first 4 dwords of
// operand o, piece 4 + o / 2 its last two (at 8 (o % 2)).  With Q4 groups of
// 64, operand o, half h is digit plane o of columns 32 h .. + 31.  With
// groups of 32, an instruction takes one group: operand o, half h is plane
// 2 (o % 2) + h of columns 32 (o / 2) .. + 31.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jm_device.h"

namespace jm {

typedef int int8v __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int F6_STAGE = 192;           // record bytes per 64 columns

// bytes of the records of `rows` rows of K columns (their exponents and group
// corrections are arrays of their own, one value per group)
__host__ __device__ constexpr size_t f6_rec_bytes(size_t rows, int K) { return rows * (size_t)K * 3; }

// 16 nibbles (w: values 0..7, v: values 8..15, value i in bits 4 i) as 16
// zero-extended 6-bit fields.  Fields 0.. hold values 0 1 3 4 6 7 9 10 12 13
// 15 8 2 11 5 14: every field is a nibble in place or shifted left by 2.
__device__ __forceinline__ void f6_spread(uint32_t w, uint32_t v, uint32_t& d0, uint32_t& d1, uint32_t& d2) {
    d0 = (w & 0x0F00F00Fu) | ((w << 2) & 0xC03C03C0u);
    d1 = (v & 0xF00F00F0u) | (__builtin_amdgcn_alignbit(v, w, 30) & 0x03C03C03u);
    d2 = (w & 0x00F00F00u) | ((v << 2) & 0x3C03C03Cu);
}

// the value each field of f6_spread's dwords holds
constexpr int F6_ORDER[16] = {0, 1, 3, 4, 6, 7, 9, 10, 12, 13, 15, 8, 2, 11, 5, 14};
constexpr int F6_AMAX = 15 * (1 + 32 + 1024 + 32768);       // the largest integer of 4 balanced digits
constexpr int F6_SHIFT = 2;
constexpr int F6_BIAS = 16 * (1 + 32 + 1024 + 32768);       // + a: every digit as digit + 16, 0..31

// Five digits, digit + 16 in 5 bits at bits 6 i, as operand codes: the sign in
// bit 5, the magnitude below.
__device__ __forceinline__ uint32_t f6_codes(uint32_t u) {
    const uint32_t n = ~(u >> 4) & 0x01041041u;             // 1 per negative digit
    return (((u & 0x0F3CF3CFu) ^ ((n << 4) - n)) + n) | (n << 5);
}

// Encode 16 consecutive columns (block c16 of a row: columns 16 c16 ..) held
// by one thread; the G / 16 threads of a group are aligned neighbours, and
// all must call this.  Writes the thread's dwords of the row's record, and
// for the group its E8M0 exponent (0xFF: NaN, when the group holds a
// non-finite value, so that it propagates) and its correction
// -8 sum(a) 2^(E - F6_SHIFT).  Only when `store`.
template <int G>
__device__ __forceinline__ void f6_encode16(const float (&x)[16], int c16, bool store, uint8_t* __restrict__ rec,
                                            uint8_t* __restrict__ exps, float* __restrict__ corr) {
    float mx = 0.0f;
    int bad = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const float a = fabsf(x[j]);
        bad |= !(a <= 3.4028235e38f);
        mx = fmaxf(mx, a);
    }
    mx = fmaxf(mx, dpp_f<DPP_XOR1>(mx));
    bad |= dpp_i<DPP_XOR1>(bad);
    if (G == 64) {
        mx = fmaxf(mx, dpp_f<DPP_XOR2>(mx));
        bad |= dpp_i<DPP_XOR2>(bad);
    }
    // (values below 2^-120 lose digits rather than leave the exponent's range)
    int E = (int)(__float_as_uint(mx) >> 23) - (127 + 18);
    E = E < -126 ? -126 : E;
    if (rintf(__builtin_ldexpf(mx, -E)) > (float)F6_AMAX) E++;
    uint32_t u[16];
    int sum = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const int q = bad ? 0 : (int)rintf(__builtin_ldexpf(x[j], -E));
        sum += q;
        u[j] = (uint32_t)(q + F6_BIAS);
    }
    sum += dpp_i<DPP_XOR1>(sum);
    if (G == 64) sum += dpp_i<DPP_XOR2>(sum);
    const int c = c16 & 3, b = c & 1;
    uint8_t* const st = rec + (size_t)(c16 >> 2) * F6_STAGE;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        uint32_t f[4] = {0, 0, 0, 0};                       // fields 0..4, 5..9, 10..14 and 15
#pragma unroll
        for (int i = 0; i < 16; i++) f[i / 5] |= ((u[F6_ORDER[i]] >> (5 * p)) & 31u) << (6 * (i % 5));
#pragma unroll
        for (int k = 0; k < 4; k++) f[k] = f6_codes(f[k]);
        f[3] &= 63u;                                        // (its other fields are absent, not -16)
        const uint32_t d0 = f[0] | (f[1] << 30), d1 = (f[1] >> 2) | (f[2] << 28), d2 = (f[2] >> 4) | (f[3] << 26);
        const int o = G == 64 ? p : 2 * (c >> 1) + p / 2, h = G == 64 ? c >> 1 : p & 1;
        uint32_t* const hd = (uint32_t*)(st + o * 32 + h * 16);
        if (!store) continue;
        if (b == 0) {
            *(uint2*)hd = make_uint2(d0, d1);
            hd[2] = d2;
        } else {
            hd[3] = d0;
            *(uint2*)(st + (4 + o / 2) * 32 + h * 16 + 8 * (o & 1)) = make_uint2(d1, d2);
        }
    }
    if (store && (threadIdx.x & (G / 16 - 1)) == 0) {
        const int g = c16 / (G / 16);
        exps[g] = bad ? 0xFF : (uint8_t)(E + 127);
        corr[g] = __builtin_ldexpf((float)(-8 * sum), E - F6_SHIFT);
    }
}

}  // namespace jm
