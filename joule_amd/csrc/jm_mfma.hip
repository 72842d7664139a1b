// Dense branch of the grouped Q4 expert product (gfx950 fp6 matrix cores),
// taken by the experts whose segment holds at least `dense_min` tokens
// (prefill-sized batches, skewed routing).  The same contraction as the
// wave-item kernels in jm_experts.hip (decode_kernel.c:1365-1383), as tiled
// products:
//
//   k_gateup_mfma  per (expert, 32-token tile, 128 intermediate rows):
//                  G = X . Wg^T and U = X . Wu^T over d, then
//                  act = (G / (1 + expf_fast(-G))) * U, written for the down
//                  product (and as float)
//   k_down_mfma    per (expert, 32-token tile, 256 hidden rows):
//                  y[slot] = w_slot * (act . Wd^T) over the intermediate
//
// Operands (jm_mx.h): the nibbles q as fp6, unpacked in registers from the
// packed rows; the tokens as 4 fp6 digit planes with one power-of-two scale
// per token and Q4 group, written by the dispatch launch for x and by the
// gate/up epilogue for act.  Tokens are the rows (A, i) and weight rows the
// columns (B, n) of v_mfma_scale_f32_32x32x64_f8f6f4, so a lane holds one
// weight row and 16 tokens.  Four accumulating instructions give a stage's
// (64 columns') sums already scaled per token; per element the epilogue is
// one multiply-add by the row's group scale:
//   acc += P * s_row
// The -8 of the Q4 code is what a group's sum starts from: the tokens' group
// corrections, three bf16 terms each, spread over the columns by a product
// with ones.  Added to the largest digits first, a group's partial sums need
// no more bits than float32 has (see group_mfma), so tokens of one sign lose
// nothing to the cancellation.
//
// A wave takes 32 tokens x 64 weight rows (two 32-row blocks, which share the
// token operands), a block 4 waves; two blocks share a CU and stay for several
// units (tile, row block).  Tokens go to LDS in super-stages of 256 columns (24
// KB, global_load_lds, 4 tokens x 256 bytes per load), weights straight to
// registers (16 rows x 64 bytes per load, brought into the operand layout by
// two lane-row swaps), both one super-stage ahead across units: a unit's
// tile entry, slots, corrections and first operands are requested during the
// unit before.
//
// Bound.  512 Zipf-routed Qwen3 tokens (183 tiles, 1098 gate/up units, 214 MB
// of records): gate/up takes 98 us and reads 475 MB past the L2, at 4.85 TB/s as
// fast as a large copy on this card, because an expert of several tiles reads
// its records once per tile; down takes 51 us for 214 MB.  The matrix cores are
// busy 17%, the VALU 37% (per wave and super-stage 32 fp6 MFMAs of 34 cycles, 4
// for the corrections and 625 vector instructions, the unit's epilogue included).  The
// unit's SwiGLU and encode take 3 to 5 us, and the units leave the third round
// of the 512 resident blocks a seventh full.  The form before (int8 digit pairs,
// exact int32 group sums, 4 instructions per element for two float scales): 134
// and 64 us; it moved 56 16-byte LDS reads and writes per wave and super-stage,
// 3584 LDS cycles of the 3600 that a pair of waves took.  Measured on the way:
// blocks of one unit 117 and 69 (each waited 7 to 14 us for its chain of loads),
// three such blocks per CU 108 and 64 (168 registers, spills), tokens staged 32
// bytes per lane pair 113 (64 address cycles per load instead of 16); the units'
// column order rotated by expert and row block made no difference; the -8 of
// all groups as one product of the corrections and the row scales at the unit's
// start 99 and 56 (it rounds: up to 15 times the error on tokens of one sign).
#include <algorithm>
#include <type_traits>

#include "jm_device.h"
#include "jm_items.h"
#include "jm_kernels.h"
#include "jm_mx.h"

namespace jm {

constexpr int MT = JM_DENSE_TILE;   // tokens per tile (32)
static_assert(MT == 32, "the tile's tokens are the 32 A rows of one MFMA");
constexpr int MTHREADS = 256;       // 4 waves per block
constexpr int NWAVE = MTHREADS / 64;
constexpr int WROWS = 64;           // weight rows per wave: two 32-row blocks
constexpr int GU_ROWS = 128;        // intermediate rows of a gate/up block (each wave: 32 of both matrices)
constexpr int DN_ROWS = 256;        // hidden rows of a down block (4 waves x 64)
constexpr int KMAX = 2048;          // longest contraction the kernels take
constexpr int SSC = 256;            // columns of a super-stage: 128 bytes (one cache line) per weight row
constexpr int PIECE = 64 * 16;      // LDS bytes of one record piece of a stage (16 bytes per lane)
constexpr int RING = 4 * 6 * PIECE; // LDS bytes of a super-stage's token operands

// The tokens' buffers, one super-stage each: separate arrays, so that the
// compiler sees that reading one does not wait for the loads into another.
struct Rings {
    uint8_t* r[3];      // the third for an odd count of super-stages
    uint8_t* corr;      // the unit's group corrections (CorrTok)
};

// Where a wave's product's operands come from: K columns in nss super-stages,
// two 32-row blocks of weight rows.
struct Operands {
    const uint8_t* recb;    // the tokens' records, at the first column (uniform)
    uint32_t reco[2];       // the offsets of tokens 8 w + l / 16 and 8 w + 4 + l / 16 of the tile
    const uint8_t* expb;    // their exponents, and the offset of token l % 32
    uint32_t expo;
    const uint8_t* w[2];    // each row block's first row's packed bytes, at the first column (uniform)
    const uint8_t* sc[2];   // and its scales
    uint32_t wrow, srow;    // bytes per packed row, per row of scales
    int nss, ng;            // super-stages, groups
};

// A value that is the same in every lane, as a scalar
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ unsigned long long scalar(unsigned long long v) {
    return (unsigned long long)(uint32_t)scalar((int)(v >> 32)) << 32 | (uint32_t)scalar((int)v);
}

// A lane's address from a uniform base and a 32-bit lane offset, both opaque
// to the optimiser: the base then stays in scalar registers and the load adds
// them (hoisted out of the super-stage loop, or as its induction variables,
// the lanes' 64-bit addresses take 40 vector registers and spill).
__device__ __forceinline__ gptr<const uint8_t> lane_at(const uint8_t* p, uint32_t o) {
    unsigned long long u = scalar((unsigned long long)p);
    __asm__ volatile("" : "+s"(u), "+v"(o));
    return (gptr<const uint8_t>)u + o;
}

template <typename T>
__device__ __forceinline__ T load_as(gptr<const uint8_t> p) {
    typedef uint32_t words __attribute__((ext_vector_type(sizeof(T) / 4)));
    return __builtin_bit_cast(T, *(gptr<const words>)p);
}

// A wave's weights of one super-stage: w[row block][half line][16-row half].
// Lane l of w[rb][u][b] holds row 16 b + l % 16, bytes 64 u + 16 (l / 16) ..
// + 15 of the 128-byte line: 16 rows x 64 bytes per load.  Each half line is
// requested for the next super-stage as soon as its registers are unpacked.
template <int G>
struct WStage {
    static constexpr int NSC = SSC / G;           // scales per row
    typedef typename std::conditional<NSC == 4, uint2, uint4>::type ScT;
    typedef typename std::conditional<NSC == 4, uint32_t, uint2>::type ExT;
    uint4 w[2][2][2];
    ScT sc[2];                                    // row l % 32's scales
    ExT ex;                                       // token l % 32's exponents
    __device__ __forceinline__ void load_half(const Operands& op, int S, int u) {
        const int l = threadIdx.x & 63;
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            const uint32_t o = (uint32_t)(l & 15) * op.wrow + 16 * (l >> 4);
#pragma unroll
            for (int b = 0; b < 2; b++)
                w[rb][u][b] = load_as<uint4>(
                    lane_at(op.w[rb] + (size_t)S * (SSC / 2) + (size_t)b * 16 * op.wrow, o) + 64 * u);
        }
    }
    __device__ __forceinline__ void load_scales(const Operands& op, int S) {
        const int l = threadIdx.x & 63;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
            sc[rb] = load_as<ScT>(lane_at(op.sc[rb] + (size_t)S * NSC * 2, (uint32_t)(l & 31) * op.srow));
        ex = load_as<ExT>(lane_at(op.expb + S * NSC, op.expo));
    }
};

// scale u (0..NSC-1) of a super-stage's packed fp16 scales, as float
template <int G>
__device__ __forceinline__ float sc_at(const typename WStage<G>::ScT& v, int u) {
    uint32_t w;
    if (G == 64) w = u < 2 ? ((const uint2&)v).x : ((const uint2&)v).y;
    else w = u < 2 ? ((const uint4&)v).x : u < 4 ? ((const uint4&)v).y : u < 6 ? ((const uint4&)v).z : ((const uint4&)v).w;
    return fp16_hw((uint16_t)(w >> (16 * (u & 1))));
}

// This wave's 8 tokens' records of super-stage S to the ring buffer: 768
// bytes each as three 256-byte groups, a load 4 tokens x 256 bytes (lane l:
// token l / 16).  [group][token][16 chunks of 16 bytes], chunk c of token i at
// c ^ (i % 16): a stage's reads, the same chunk of 32 tokens, fall in
// different banks.
__device__ __forceinline__ void stage_tokens(const Operands& op, int S, uint8_t* ring) {
    const int w = scalar((int)(threadIdx.x >> 6)), l = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const uint32_t i = 8 * w + 4 * q + (l >> 4);
        const gptr<const uint8_t> src = lane_at(op.recb + (size_t)S * (4 * F6_STAGE), op.reco[q] + 16 * ((l ^ i) & 15));
#pragma unroll
        for (int g = 0; g < 3; g++)
            __builtin_amdgcn_global_load_lds((gptr<void>)(src + 256 * g),
                                             (__attribute__((address_space(3))) void*)(ring + (32 * g + 8 * w + 4 * q) * 256), 16, 0, 0);
    }
}

// The unit's group corrections on their way to LDS, three bf16 terms each
// (exact: 24 bits).  Thread t holds blocks t / 32 + 8 r of 4 groups of token
// t % 32; in LDS [block][term][token][4 groups].
constexpr int CBLOCK = 3 * MT * 8;                // LDS bytes of a block of 4 groups
template <int CR>
struct CorrTok {
    float4 c[CR];
    __device__ __forceinline__ void load(const float* corr, int ng) {
#pragma unroll
        for (int r = 0; r < CR; r++) {
            const int b = (threadIdx.x >> 5) + 8 * r;
            c[r] = *(const float4*)(corr + (4 * b < ng ? 4 * b : 0));
        }
    }
    __device__ __forceinline__ void store(int ng, uint8_t* cl) const {
#pragma unroll
        for (int r = 0; r < CR; r++) {
            const int b = (threadIdx.x >> 5) + 8 * r;
            if (4 * b >= ng) continue;
            const float v[4] = {c[r].x, c[r].y, c[r].z, c[r].w};
            uint32_t t[3][2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float x = v[2 * e], y = v[2 * e + 1];
                split_bf16x2(x, y, t[0][e], t[1][e]);
                // (half the third term: its lanes meet two ones)
                t[2][e] = pack_bf16x2(
                    __fmul_rn(0.5f, __fsub_rn(__fsub_rn(x, __uint_as_float(t[0][e] << 16)), __uint_as_float(t[1][e] << 16))),
                    __fmul_rn(0.5f, __fsub_rn(__fsub_rn(y, __uint_as_float(t[0][e] & 0xFFFF0000u)),
                                              __uint_as_float(t[1][e] & 0xFFFF0000u))));
            }
#pragma unroll
            for (int k = 0; k < 3; k++)
                *(uint2*)(cl + b * CBLOCK + (k * MT + (threadIdx.x & 31)) * 8) = make_uint2(t[k][0], t[k][1]);
        }
    }
};

// A block's 4 groups as the operand of v_mfma_f32_32x32x16_bf16: lane half 0
// the first and second terms, half 1 the third twice.
__device__ __forceinline__ bf16x8 corr_operand(const uint8_t* cl, int b) {
    const int l = threadIdx.x & 63, h = l >> 5;
    const uint8_t* const p = cl + b * CBLOCK + (2 * h * MT + (l & 31)) * 8;
    const uint2 x = *(const uint2*)p, y = *(const uint2*)(p + (h ? 0 : MT * 8));
    return __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
}

// The correction of group g of the block for every column: ones at both terms
template <int GI>
__device__ __forceinline__ floatx16 corr_init(const bf16x8& c) {
    constexpr uint32_t one = GI & 1 ? 0x3F800000u : 0x3F80u, lo = GI < 2 ? one : 0u, hi = GI < 2 ? 0u : one;
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(c, __builtin_bit_cast(bf16x8, make_uint4(lo, hi, lo, hi)), floatx16{}, 0, 0, 0);
}

// Two dwords of each of the 4 sixteen-lane rows exchanged: x = rows (x0, x1,
// x2, x3), y likewise -> (x0, y0, x2, y2) and (x1, y1, x3, y3)
__device__ __forceinline__ void swap16(uint32_t& x, uint32_t& y) {
    const auto p = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = p[0];
    y = p[1];
}
// -> (x0, x1, y0, y1) and (x2, x3, y2, y3)
__device__ __forceinline__ void swap32(uint32_t& x, uint32_t& y) {
    const auto p = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = p[0];
    y = p[1];
}

__device__ __forceinline__ int8v f6_operand(const uint32_t (&d)[4]) {
    uint32_t f[6];
    f6_spread(d[0], d[1], f[0], f[1], f[2]);
    f6_spread(d[2], d[3], f[3], f[4], f[5]);
    return int8v{(int)f[0], (int)f[1], (int)f[2], (int)f[3], (int)f[4], (int)f[5], 0, 0};
}

// The weight operands of one row block from half a line (64 bytes: two
// stages) of each row.  G = 64: both stages', b[stage].  G = 32: stage S's two
// groups, b[group], each group's 32 columns in both lane halves.
template <int G, int S>
__device__ __forceinline__ void load_bops(const uint4 (&w)[2], int8v (&b)[2]) {
    const uint32_t x[4] = {w[0].x, w[0].y, w[0].z, w[0].w}, y[4] = {w[1].x, w[1].y, w[1].z, w[1].w};
    uint32_t d0[4], d1[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        uint32_t p = x[k], q = y[k];
        swap16(p, q);                             // p: chunks 0, 2 of rows 0..15, 16..31; q: chunks 1, 3
        if (G == 64) {
            swap32(p, q);                         // chunks (0, 1) and (2, 3) in the lane halves
            d0[k] = p;
            d1[k] = q;
        } else {
            uint32_t p2 = p, q2 = q;
            swap32(p, p2);                        // chunk 0 and chunk 2 in both halves
            swap32(q, q2);                        // chunk 1 and chunk 3
            d0[k] = S ? p2 : p;
            d1[k] = S ? q2 : q;
        }
    }
    b[0] = f6_operand(d0);
    b[1] = f6_operand(d1);
}

// P (+)= A . B with the token exponent in byte SA of sa and the plane's
// scale in byte SB of sb
template <int SA, int SB>
__device__ __forceinline__ floatx16 mfma_f6(const int8v& a, const int8v& b, const floatx16& c, uint32_t sa, uint32_t sb) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 2, 2, SA, (int)sa, SB, (int)sb);
}

// A piece of a stage's token operands in LDS, this lane's: piece k, half h is
// chunk 12 CS + 2 k + h of token l % 32, at `at` for chunk h.
template <int CS>
__device__ __forceinline__ uint4 token_piece(const uint8_t* ring, uint32_t at, int k) {
    const int c = 12 * CS + 2 * k;
    return *(const uint4*)(ring + (c >> 4) * (32 * 256) + (at ^ (16 * (c & 15))));
}

// One group's products: P[rb] from the stage's token operands in LDS, on top
// of the group's correction (corr: the operand of the block of 4 groups it
// lies in).  The digits' planes come largest first: the correction -8 sum(a)
// and the sums with the planes of 32^3, 32^2 and 32 are multiples of 8, which
// float32 holds up to 2^27, so they round only in groups whose values are
// nearly all of one sign and within half of the largest (|sum a| over 2^24);
// the last, sum a (q - 8), is rounded past 2^24.
template <int G, int CS, int GI>
__device__ __forceinline__ void group_mfma(floatx16 (&P)[2], const uint8_t* ring, const int8v& b0, const int8v& b1,
                                           const typename WStage<G>::ExT& ex, uint32_t sb, const bf16x8& corr) {
    // (opaque: the addresses are made here instead of being kept in registers)
    const int l = threadIdx.x & 63;
    uint32_t at = (l & 31) * 256 + 16 * ((l >> 5) ^ (l & 15));
    __asm__ volatile("" : "+v"(at));
    // operands 2 o and 2 o + 1
    const auto pair = [&](int o, int8v& x, int8v& y) __attribute__((always_inline)) {
        const uint4 p = token_piece<CS>(ring, at, 2 * o), q = token_piece<CS>(ring, at, 2 * o + 1), r = token_piece<CS>(ring, at, 4 + o);
        x = int8v{(int)p.x, (int)p.y, (int)p.z, (int)p.w, (int)r.x, (int)r.y, 0, 0};
        y = int8v{(int)q.x, (int)q.y, (int)q.z, (int)q.w, (int)r.z, (int)r.w, 0, 0};
    };
    if constexpr (G == 64) {
        int8v a0, a1, a2, a3;
        pair(1, a2, a3);
        pair(0, a0, a1);
        const floatx16 c = corr_init<CS>(corr);
        P[0] = mfma_f6<CS, 3>(a3, b0, c, ex, sb);
        P[1] = mfma_f6<CS, 3>(a3, b1, c, ex, sb);
        P[0] = mfma_f6<CS, 2>(a2, b0, P[0], ex, sb);
        P[1] = mfma_f6<CS, 2>(a2, b1, P[1], ex, sb);
        P[0] = mfma_f6<CS, 1>(a1, b0, P[0], ex, sb);
        P[1] = mfma_f6<CS, 1>(a1, b1, P[1], ex, sb);
        P[0] = mfma_f6<CS, 0>(a0, b0, P[0], ex, sb);
        P[1] = mfma_f6<CS, 0>(a0, b1, P[1], ex, sb);
    } else {
        const uint32_t e = CS < 2 ? ex.x : ex.y;
        constexpr int B0 = 2 * (CS & 1) + GI;
        int8v a0, a1;
        pair(GI, a0, a1);
        const floatx16 c = corr_init<B0>(corr);
        P[0] = mfma_f6<B0, 1>(a1, b0, c, e, sb);
        P[1] = mfma_f6<B0, 1>(a1, b1, c, e, sb);
        P[0] = mfma_f6<B0, 0>(a0, b0, P[0], e, sb);
        P[1] = mfma_f6<B0, 0>(a0, b1, P[1], e, sb);
    }
}

__device__ __forceinline__ void group_acc(floatx16& acc, const floatx16& P, float ws) {
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = __builtin_fmaf(P[v], ws, acc[v]);
}

// A result from its accumulator (exact but at the ends of the float32 range)
__device__ __forceinline__ float full(float acc) { return __fmul_rn(acc, (float)(1 << F6_SHIFT)); }

// What acc depends on comes before what follows in the source (else the
// operands of later stages are read first, into registers there are not).
__device__ __forceinline__ void pin(floatx16 (&acc)[2]) {
    __asm__ volatile("" : "+v"(acc[0]), "+v"(acc[1]) : : "memory");
}

// blocks of 4 groups of a contraction: of 256 or 768 columns for one or three
// super-stages, else of up to KMAX
constexpr int corr_blocks(int G, int nss) { return (nss ? nss * SSC : KMAX) / G / 4; }

// A wave's running state over a block's units (a unit: one token tile against
// the block's rows): the operands of the unit being computed and the next
// super-stage's weights.
template <int G, int NSS>
struct Pipe {
    using W = WStage<G>;
    static constexpr int NG = 64 / G;
    W w;
    floatx16 acc[2];
    CorrTok<(corr_blocks(G, NSS) + 7) / 8> ct;

    // the first unit's operands
    __device__ __forceinline__ void start(const Operands& op, const Rings& rg, const float* corr) {
        ct.load(corr, op.ng);
        stage_tokens(op, 0, rg.r[0]);
        w.load_half(op, 0, 0);
        w.load_half(op, 0, 1);
        w.load_scales(op, 0);
        ct.store(op.ng, rg.corr);
    }

    // Super-stage S from `ring` (its corrections at cl); the next one's
    // operands (nop's super-stage nS) are requested into nring and the weight
    // registers.  hook() runs once every wave's operands of S are there.
    template <class Hook>
    __device__ __forceinline__ void step(const uint8_t* ring, const uint8_t* cl, uint8_t* nring, Hook&& hook) {
        const uint32_t h = (threadIdx.x >> 5) & 1;
        // the planes' scales: 2^6 for the two operands' eighths, times 32^plane, 2^F6_SHIFT times smaller
        constexpr uint32_t sh = 0x01010101u * F6_SHIFT;
        const uint32_t sb = G == 64 ? 0x948F8A85u - sh : h ? 0x948Au - (sh & 0xFFFFu) : 0x8F85u - (sh & 0xFFFFu);
        // this super-stage's tokens and weights have arrived (waited for by
        // count the tokens alone would do, but the compiler then waits for
        // the next ones' loads to LDS before it takes the weights; and the
        // block barrier does not wait for loads to LDS), and every wave is
        // done with the one before, whose buffer may be filled again
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070);       // vmcnt(0), lgkmcnt(0)
        wave_meet();
        int nS;
        const Operands nop = hook(nS);
        if (nring) stage_tokens(nop, nS, nring);
        __builtin_amdgcn_sched_barrier(0);
        const typename W::ScT sc[2] = {w.sc[0], w.sc[1]};
        const typename W::ExT ex = w.ex;
        bf16x8 corr = corr_operand(cl, 0);
        auto stage = [&](auto cs_, const int8v (&b)[2][NG]) __attribute__((always_inline)) {
            constexpr int CS = decltype(cs_)::value;
            if (G == 32 && CS == 2) corr = corr_operand(cl, 1);
            floatx16 P[2];
            group_mfma<G, CS, 0>(P, ring, b[0][0], b[1][0], ex, sb, corr);
            group_acc(acc[0], P[0], sc_at<G>(sc[0], NG * CS));
            group_acc(acc[1], P[1], sc_at<G>(sc[1], NG * CS));
            if constexpr (G == 32) {
                group_mfma<G, CS, 1>(P, ring, b[0][1], b[1][1], ex, sb, corr);
                group_acc(acc[0], P[0], sc_at<G>(sc[0], NG * CS + 1));
                group_acc(acc[1], P[1], sc_at<G>(sc[1], NG * CS + 1));
            }
        };
        auto half = [&](auto u) __attribute__((always_inline)) {
            constexpr int U = decltype(u)::value;
            if constexpr (G == 64) {
                int8v t0[2], t1[2];
                load_bops<G, 0>(w.w[0][U], t0);
                load_bops<G, 0>(w.w[1][U], t1);
                __builtin_amdgcn_sched_barrier(0);
                w.load_half(nop, nS, U);
                if (U == 1) w.load_scales(nop, nS);
                __builtin_amdgcn_sched_barrier(0);
                const int8v b0[2][NG] = {{t0[0]}, {t1[0]}}, b1[2][NG] = {{t0[1]}, {t1[1]}};
                stage(std::integral_constant<int, 2 * U>{}, b0);
                pin(acc);                     // (one stage's operands at a time: registers)
                stage(std::integral_constant<int, 2 * U + 1>{}, b1);
                pin(acc);
            } else {
                int8v b[2][NG];
                load_bops<G, 0>(w.w[0][U], b[0]);
                load_bops<G, 0>(w.w[1][U], b[1]);
                stage(std::integral_constant<int, 2 * U>{}, b);
                pin(acc);                     // (one stage's operands at a time: registers)
                load_bops<G, 1>(w.w[0][U], b[0]);
                load_bops<G, 1>(w.w[1][U], b[1]);
                __builtin_amdgcn_sched_barrier(0);
                w.load_half(nop, nS, U);
                if (U == 1) w.load_scales(nop, nS);
                __builtin_amdgcn_sched_barrier(0);
                stage(std::integral_constant<int, 2 * U + 1>{}, b);
                pin(acc);
            }
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
    }

    // The unit's super-stages (NSS 0: an even count, or 1 or 3), then the next
    // unit's first operands on their way.  early() runs in the first
    // super-stage, late(nop) in the second (in the only one, after early's
    // loads): they find the next unit and fill in its operands.
    template <class Early, class Late>
    __device__ __forceinline__ void unit(const Operands& op, Operands& nop, const Rings& rg, Early&& early, Late&& late) {
        constexpr int CSS = SSC / G / 4 * CBLOCK;     // LDS bytes of a super-stage's corrections
        auto first = [&]() __attribute__((always_inline)) {
            acc[0] = floatx16{};
            acc[1] = floatx16{};
            early();
        };
        if constexpr (NSS == 1) {
            step(rg.r[0], rg.corr, nullptr, [&](int& nS) __attribute__((always_inline)) -> Operands {
                first();
                late(nop);
                nS = 0;
                return nop;
            });
            wave_meet();                      // every wave is done with the only buffer and the corrections
            stage_tokens(nop, 0, rg.r[0]);
        } else if constexpr (NSS == 3) {
            step(rg.r[0], rg.corr, rg.r[1], [&](int& nS) __attribute__((always_inline)) -> Operands { first(); nS = 1; return op; });
            step(rg.r[1], rg.corr + CSS, rg.r[2], [&](int& nS) __attribute__((always_inline)) -> Operands { late(nop); nS = 2; return op; });
            step(rg.r[2], rg.corr + 2 * CSS, rg.r[0], [&](int& nS) __attribute__((always_inline)) -> Operands { nS = 0; return nop; });
        } else {
#pragma unroll 1
            for (int S = 0; S < op.nss; S += 2) {
                step(rg.r[0], rg.corr + S * CSS, rg.r[1], [&](int& nS) __attribute__((always_inline)) -> Operands {
                    if (S == 0) first();
                    nS = S + 1;
                    return op;
                });
                const bool last = S + 2 == op.nss;
                step(rg.r[1], rg.corr + (S + 1) * CSS, rg.r[0], [&](int& nS) __attribute__((always_inline)) -> Operands {
                    if (S == 0) late(nop);
                    nS = last ? 0 : S + 2;
                    return last ? nop : op;
                });
            }
        }
    }
};

// The kernels' blocks stay for several units: unit u of the grid's gridDim.x
// blocks is tile u / nrb, row block u % nrb, then u + gridDim.x; past the
// tiles' units come the small experts' items.  A tile's entry, its slots and
// its first operands are requested during the unit before, so that only the
// block's first unit waits for that chain of loads.
__device__ __forceinline__ int4 tile_at(const ExpertArgs& a, int t) {
    const int4 ti = a.tiles[t];
    return make_int4(scalar(ti.x), scalar(ti.y), scalar(ti.z), 0);
}

// this lane's slot of a tile: token l % 32 (padding: the first)
__device__ __forceinline__ int tile_slot(const ExpertArgs& a, const int4& ti) {
    const int i = threadIdx.x & 31;
    return a.seg_slot[ti.y + (i < ti.z ? i : 0)];
}

// rows: the tokens' row of lane l % 32, K columns
template <int G>
__device__ __forceinline__ void set_tokens(Operands& op, const uint8_t* rec, const uint8_t* exps, int row, int K) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    op.recb = rec;                                // (below 4 GB: at most JM_MAX_SLOTS rows of KMAX columns)
#pragma unroll
    for (int q = 0; q < 2; q++) op.reco[q] = (uint32_t)f6_rec_bytes(__shfl(row, 8 * w + 4 * q + (l >> 4), JM_WAVE), K);
    op.expb = exps;
    op.expo = (uint32_t)row * (K / G);
    op.wrow = K / 2;
    op.srow = K / G * 2;
    op.nss = K / SSC;
    op.ng = K / G;
}

// ------------------------------------------------------------------ gate/up

template <int G>
__device__ __forceinline__ void gateup_op(Operands& op, const ExpertArgs& a, const int4& ti, int rblk, int sl) {
    const int w = scalar((int)(threadIdx.x >> 6));
    set_tokens<G>(op, a.xq, a.xe, sl / a.topk, a.d);
#pragma unroll
    for (int mat = 0; mat < 2; mat++) {           // gate rows, then the same up rows
        unsigned long long so, po;
        a.rec.get(mat, a.key0 + ti.x, so, po);
        op.w[mat] = a.blob + scalar(po) + (size_t)(rblk * GU_ROWS + 32 * w) * op.wrow;
        op.sc[mat] = a.blob + scalar(so) + (size_t)(rblk * GU_ROWS + 32 * w) * op.srow;
    }
}

constexpr int ACT_RP = GU_ROWS + 4;               // padded LDS row of one token's act values

// The unit's act values: SiLU(g) * u (dividing as the reference does,
// decode_kernel.c:1375) to LDS, then 16 consecutive rows of one token per
// thread: the float values and their record for the down product.
template <int G>
__device__ __forceinline__ void gateup_out(const ExpertArgs& a, const floatx16 (&acc)[2], const int4& ti, int rblk, int sl,
                                           float* act) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n = lane & 31, h = lane >> 5;
    const int m = a.m, r0 = rblk * GU_ROWS;
#pragma unroll
    for (int v = 0; v < 16; v++) act[(8 * (v / 4) + 4 * h + (v % 4)) * ACT_RP + 32 * w + n] = swiglu(full(acc[0][v]), full(acc[1][v]));
    __builtin_amdgcn_s_waitcnt(0xC07F);           // lgkmcnt(0)
    wave_meet();
    const int it = tid >> 3, rr = 16 * (tid & 7);
    const bool live = it < ti.z;
    const int slot = __shfl(sl, it, JM_WAVE);
    float v[16];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 f = *(const float4*)(act + it * ACT_RP + rr + 4 * q);
        v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
        if (live) *(float4*)(a.act + (size_t)slot * m + r0 + rr + 4 * q) = f;
    }
    f6_encode16<G>(v, (r0 + rr) / 16, live, a.aq + f6_rec_bytes(slot, m), a.ae + (size_t)slot * (m / G),
                   a.ac + (size_t)slot * (m / G));
}

// The experts under dense_min (n_tiles[1] entries of the small list) as
// wave items, the units after the tiles' (first = this block's first of them,
// nblk = the blocks of the grid): virtual block v takes the 4 consecutive items
// 4 (v % vpe) + w of small entry v / vpe.
template <int G, int LPR, int NDIG>
__device__ __forceinline__ void small_gateup(const ExpertArgs& a, int first, int nblk, unsigned char* sm) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int vpe = a.m / wi::GU_ROWS / NWAVE;
    const int nv = a.n_tiles[1] * vpe;
    // the act-scale slots of wi::gateup_item
    float (&gm)[2][4] = *(float (*)[2][4])sm;
    int (&gb)[2][4] = *(int (*)[2][4])(sm + sizeof(float[2][4]));
#pragma unroll 1
    for (int v = first; v < nv; v += nblk) {
        wi::gateup_item<G, NDIG, LPR, 1, false>(a, a.top, a.small[v / vpe], (v % vpe) * NWAVE + w, gm, gb);
        __syncthreads();                          // the slots serve the next item
    }
}

template <int G, int LPR, int NDIG>
__global__ void __launch_bounds__(MTHREADS, 2)
k_gateup_mfma(ExpertArgs a) {
    __shared__ __align__(16) uint8_t ring0[RING];
    __shared__ __align__(16) uint8_t ring1[RING];
    __shared__ __align__(16) uint8_t corr_l[corr_blocks(G, 0) * CBLOCK];
    __shared__ __align__(16) float act[MT * ACT_RP];
    const Rings rg{{ring0, ring1, nullptr}, corr_l};
    const int nrb = a.m / GU_ROWS, nb = gridDim.x;
    int u = blockIdx.x;
    int4 ti = tile_at(a, u / nrb);
    const int ntb = scalar(a.n_tiles[0]) * nrb;
    if (u < ntb) {
        int sl = tile_slot(a, ti);
        Operands op;
        gateup_op<G>(op, a, ti, u % nrb, sl);
        Pipe<G, 0> p;
        p.start(op, rg, a.xc + (size_t)(sl / a.topk) * op.ng);
#pragma unroll 1
        for (;;) {
            const int un = u + nb < ntb ? u + nb : u;         // past the last, the last again
            int4 tn = a.tiles[un / nrb];
            int sn = 0;
            Operands nop;
            p.unit(op, nop, rg,
                [&]() __attribute__((always_inline)) {
                    tn = make_int4(scalar(tn.x), scalar(tn.y), scalar(tn.z), 0);
                    sn = tile_slot(a, tn);
                },
                [&](Operands& o) __attribute__((always_inline)) { gateup_op<G>(o, a, tn, un % nrb, sn); });
            p.ct.load(a.xc + (size_t)(sn / a.topk) * nop.ng, nop.ng);
            gateup_out<G>(a, p.acc, ti, u % nrb, sl, act);
            if (un == u) break;
            p.ct.store(nop.ng, corr_l);           // (every wave met in gateup_out, past its last read of the old ones)
            u = un;
            ti = tn;
            sl = sn;
            op = nop;
        }
        u += nb;
        __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): nothing on its way to LDS
        __syncthreads();
    }
    small_gateup<G, LPR, NDIG>(a, u - ntb, nb, ring0);
}

// --------------------------------------------------------------------- down

template <int G>
__device__ __forceinline__ void down_op(Operands& op, const ExpertArgs& a, const int4& ti, int rblk, int sl) {
    const int w = scalar((int)(threadIdx.x >> 6));
    set_tokens<G>(op, a.aq, a.ae, sl, a.m);
    unsigned long long so, po;
    a.rec.get(2, a.key0 + ti.x, so, po);
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        op.w[rb] = a.blob + scalar(po) + (size_t)(rblk * DN_ROWS + WROWS * w + 32 * rb) * op.wrow;
        op.sc[rb] = a.blob + scalar(so) + (size_t)(rblk * DN_ROWS + WROWS * w + 32 * rb) * op.srow;
    }
}

// The unit's weighted rows of y.
__device__ __forceinline__ void down_out(const ExpertArgs& a, const floatx16 (&acc)[2], const int4& ti, int rblk, int sl,
                                         float tw) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    const int row = rblk * DN_ROWS + WROWS * w + n;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int i = 8 * (v / 4) + 4 * h + (v % 4);
        const int slot = __shfl(sl, i, JM_WAVE);
        const float t = __shfl(tw, i, JM_WAVE);
        if (i < ti.z) {
            float* const y = a.y + (size_t)slot * a.d + row;
            y[0] = __fmul_rn(t, full(acc[0][v]));
            y[32] = __fmul_rn(t, full(acc[1][v]));
        }
    }
}

// The small experts' down items (wi::down_item, no barriers) on the blocks
// past the tiles, 4 consecutive items of one entry per virtual block.
template <int G, int LPR, int NDIG>
__device__ __forceinline__ void small_down(const ExpertArgs& a, int first, int nblk) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int vpe = a.d / wi::DN_ROWS / NWAVE;
    const int nv = a.n_tiles[1] * vpe;
#pragma unroll 1
    for (int v = first; v < nv; v += nblk)
        wi::down_item<G, NDIG, LPR, 1>(a, a.small[v / vpe], (v % vpe) * NWAVE + w);
}

// NSS: super-stages of the contraction (Pipe::unit)
template <int G, int LPR, int NDIG, int NSS>
__global__ void __launch_bounds__(MTHREADS, 2)
k_down_mfma(ExpertArgs a) {
    __shared__ __align__(16) uint8_t ring0[RING];
    __shared__ __align__(16) uint8_t ring1[NSS == 1 ? 16 : RING];
    __shared__ __align__(16) uint8_t ring2[NSS == 3 ? RING : 16];
    __shared__ __align__(16) uint8_t corr_l[corr_blocks(G, NSS) * CBLOCK];
    const Rings rg{{ring0, ring1, ring2}, corr_l};
    const int nrb = a.d / DN_ROWS, nb = gridDim.x;
    int u = blockIdx.x;
    int4 ti = tile_at(a, u / nrb);
    const int ntb = scalar(a.n_tiles[0]) * nrb;
    if (u < ntb) {
        int sl = tile_slot(a, ti);
        float tw = a.tw[sl];
        Operands op;
        down_op<G>(op, a, ti, u % nrb, sl);
        Pipe<G, NSS> p;
        p.start(op, rg, a.ac + (size_t)sl * op.ng);
#pragma unroll 1
        for (;;) {
            const int un = u + nb < ntb ? u + nb : u;         // past the last, the last again
            int4 tn = a.tiles[un / nrb];
            int sn = 0;
            Operands nop;
            p.unit(op, nop, rg,
                [&]() __attribute__((always_inline)) {
                    tn = make_int4(scalar(tn.x), scalar(tn.y), scalar(tn.z), 0);
                    sn = tile_slot(a, tn);
                },
                [&](Operands& o) __attribute__((always_inline)) { down_op<G>(o, a, tn, un % nrb, sn); });
            const float twn = a.tw[sn];
            p.ct.load(a.ac + (size_t)sn * nop.ng, nop.ng);
            down_out(a, p.acc, ti, u % nrb, sl, tw);
            if (un == u) break;
            if (NSS != 1) wave_meet();            // every wave has read the unit's corrections
            p.ct.store(nop.ng, corr_l);
            u = un;
            ti = tn;
            sl = sn;
            tw = twn;
            op = nop;
        }
        u += nb;
        __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): nothing on its way to LDS
        __syncthreads();
    }
    small_down<G, LPR, NDIG>(a, u - ntb, nb);
}

// ------------------------------------------------------ plain Q4 product

// out[t][row] = X[t] . dequant(W[row]) for one Q4 matrix (the plugin
// product q4_gemm_f32, expert_ffn.c:200-215, at prefill-sized T): block
// (32-token tile, 256 rows, K split z), 4 waves x 64 rows, as a unit of the
// down kernel without routing.  The records of X come from k_prep_f6.
// With gridDim.z > 1 split z covers the columns [z kl, z kl + kl) (whole Q4
// groups and super-stages) and writes its partial sums to out + z T m, which
// k_sum_splits adds in split order.
template <int G, int NSS>
__global__ void __launch_bounds__(MTHREADS, 2)
k_q4_gemm_mfma(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales,
               const uint8_t* __restrict__ xq, const uint8_t* __restrict__ xe, const float* __restrict__ xc, int T, int m,
               int d, int kl, float* __restrict__ out) {
    __shared__ __align__(16) uint8_t ring0[RING];
    __shared__ __align__(16) uint8_t ring1[NSS == 1 ? 16 : RING];
    __shared__ __align__(16) uint8_t ring2[NSS == 3 ? RING : 16];
    __shared__ __align__(16) uint8_t corr_l[corr_blocks(G, NSS) * CBLOCK];
    const Rings rg{{ring0, ring1, ring2}, corr_l};
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = scalar(tid >> 6);
    const int ng = d / G;                         // groups per row
    const int k0 = (int)blockIdx.z * kl;          // the split's first column
    const int t0 = blockIdx.x * MT;
    const int nt = min(MT, T - t0);
    float* const o = out + (size_t)blockIdx.z * T * m;
    const int i0 = lane & 31, h = lane >> 5;
    const int t = i0 < nt ? i0 : 0;               // padding: the tile's first token
    const int row0 = blockIdx.y * DN_ROWS + WROWS * w;
    Operands op;
    set_tokens<G>(op, xq + f6_rec_bytes(t0, d) + (size_t)k0 * 3, xe + (size_t)t0 * ng + k0 / G, t, d);
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        op.w[rb] = packed + (size_t)(row0 + 32 * rb) * op.wrow + k0 / 2;
        op.sc[rb] = (const uint8_t*)scales + (size_t)(row0 + 32 * rb) * op.srow + (size_t)(k0 / G) * 2;
    }
    op.nss = kl / SSC;
    op.ng = kl / G;
    Pipe<G, NSS> p;
    p.start(op, rg, xc + (size_t)(t0 + t) * ng + k0 / G);
    Operands nop = op;
    p.unit(op, nop, rg, []() __attribute__((always_inline)) {}, [](Operands&) __attribute__((always_inline)) {});
    __builtin_amdgcn_s_waitcnt(0x0F70);           // vmcnt(0): nothing on its way to LDS
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int i = 8 * (v / 4) + 4 * h + (v % 4);
        if (i < nt) {
            float* const y = o + (size_t)(t0 + i) * m + row0 + i0;
            y[0] = full(p.acc[0][v]);
            y[32] = full(p.acc[1][v]);
        }
    }
}

// out[i] = the sum of the ns partial products part[z][i], z = 0, 1, ... in
// order (n4 float4 elements each).
__global__ void __launch_bounds__(256)
k_sum_splits(const float4* __restrict__ part, long long n4, int ns, float4* __restrict__ out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 v[8];
#pragma unroll
    for (int z = 0; z < 8; z++)
        if (z < ns) v[z] = part[(size_t)z * n4 + i];
    float4 r = v[0];
#pragma unroll
    for (int z = 1; z < 8; z++)
        if (z < ns) {
            r.x = __fadd_rn(r.x, v[z].x);
            r.y = __fadd_rn(r.y, v[z].y);
            r.z = __fadd_rn(r.z, v[z].z);
            r.w = __fadd_rn(r.w, v[z].w);
        }
    out[i] = r;
}

// The records, exponents and corrections of T rows of d floats, 16 columns per
// thread (as the dispatch launch encodes the block's tokens).
template <int G>
__global__ void __launch_bounds__(256)
k_prep_f6(const float* __restrict__ X, int T, int d, uint8_t* __restrict__ rec, uint8_t* __restrict__ exps,
          float* __restrict__ corr) {
    const long long u = (long long)blockIdx.x * 256 + threadIdx.x;
    const int nblk = d / 16, ng = d / G;
    const long long b = u / nblk;
    const int c16 = (int)(u % nblk);
    const bool ok = b < T;
    const size_t row = ok ? b : 0;
    const float4* xp = (const float4*)(X + row * d + 16 * c16);
    float v[16];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 f = xp[q];
        v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
    }
    f6_encode16<G>(v, c16, ok, rec + f6_rec_bytes(row, d), exps + row * ng, corr + row * ng);
}

// Contractions the kernels take: whole super-stages up to 1024 columns, or
// whole 1024s; row counts of whole blocks.
static bool mfma_k_ok(int K) { return K % SSC == 0 && K <= KMAX && (K <= 1024 || K % 1024 == 0); }

bool mfma_shape_ok(int d, int m) {
    return d % 512 == 0 && m % GU_ROWS == 0 && mfma_k_ok(d) && mfma_k_ok(m);
}

// Lanes per row segment of the small experts' wave items: rows of C columns
// (C / 32 chunks of 16 bytes; C <= KMAX, so one chunk per lane).
static int item_lanes(int C) { return C / 32 <= 32 ? 32 : 64; }

// Two blocks per CU (registers and LDS), or as many as there can be units:
// max_tiles tiles and one more row of blocks for the small experts' items.
static unsigned unit_blocks(int max_tiles, int row_blocks) {
    static const int ncu = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            n = 0;
        return n > 0 ? n : 256;
    }();
    return (unsigned)std::min<long long>(2 * ncu, (long long)(max_tiles + 1) * row_blocks);
}

hipError_t launch_gateup_mfma(const ExpertArgs& a, int max_tiles, hipStream_t st) {
    if (max_tiles == 0) return hipSuccess;
    if (!mfma_shape_ok(a.d, a.m) || (a.group != 64 && a.group != 32)) return hipErrorInvalidValue;
    if (!a.small || (a.m / wi::GU_ROWS) % NWAVE || (a.ndig != 4 && a.ndig != 5)) return hipErrorInvalidValue;
    const dim3 grid(unit_blocks(max_tiles, a.m / GU_ROWS));
    const bool l64 = item_lanes(a.d) == 64;
#define JM_GM(GG, L) do { if (a.ndig == 5) hipLaunchKernelGGL((k_gateup_mfma<GG, L, 5>), grid, dim3(MTHREADS), 0, st, a); \
                          else hipLaunchKernelGGL((k_gateup_mfma<GG, L, 4>), grid, dim3(MTHREADS), 0, st, a); } while (0)
    if (a.group == 64) {
        if (l64) JM_GM(64, 64);
        else JM_GM(64, 32);
    } else {
        if (l64) JM_GM(32, 64);
        else JM_GM(32, 32);
    }
#undef JM_GM
    return hipGetLastError();
}

hipError_t launch_down_mfma(const ExpertArgs& a, int max_tiles, hipStream_t st) {
    if (max_tiles == 0) return hipSuccess;
    if (!mfma_shape_ok(a.d, a.m) || (a.group != 64 && a.group != 32)) return hipErrorInvalidValue;
    if (!a.small || (a.d / wi::DN_ROWS) % NWAVE || (a.ndig != 4 && a.ndig != 5)) return hipErrorInvalidValue;
    const dim3 grid(unit_blocks(max_tiles, a.d / DN_ROWS));
    const bool l64 = item_lanes(a.m) == 64;
    const int nss = a.m / SSC;
#define JM_DN(GG, L, N) do { if (nss == 1) hipLaunchKernelGGL((k_down_mfma<GG, L, N, 1>), grid, dim3(MTHREADS), 0, st, a); \
                             else if (nss == 3) hipLaunchKernelGGL((k_down_mfma<GG, L, N, 3>), grid, dim3(MTHREADS), 0, st, a); \
                             else hipLaunchKernelGGL((k_down_mfma<GG, L, N, 0>), grid, dim3(MTHREADS), 0, st, a); } while (0)
#define JM_DM(GG, L) do { if (a.ndig == 5) JM_DN(GG, L, 5); else JM_DN(GG, L, 4); } while (0)
    if (a.group == 64) {
        if (l64) JM_DM(64, 64);
        else JM_DM(64, 32);
    } else {
        if (l64) JM_DM(32, 64);
        else JM_DM(32, 32);
    }
#undef JM_DM
#undef JM_DN
    return hipGetLastError();
}

static size_t pad256(size_t n) { return (n + 255) & ~(size_t)255; }

bool q4_gemm_mfma_ok(int m, int d, int group) {
    // whole 256-row passes; each row's scales of a super-stage in one
    // aligned 8-byte (G = 64) or 16-byte (G = 32) load
    return m % DN_ROWS == 0 && mfma_k_ok(d) && (group == 64 || group == 32) &&
           ((d / group) * 2) % (group == 64 ? 8 : 16) == 0;
}

// K splits of the plain product: when the grid of token tiles x row blocks
// would leave most of the 256 CUs idle, ns blocks share each one's
// contraction (ns a divisor of the super-stages over d, at most 8): the
// smallest ns that fills one round of 256 blocks, else the largest.
int q4_gemm_splits(int T, int m, int d) {
    const long long blocks = (long long)((T + MT - 1) / MT) * (m / DN_ROWS);
    const int nss = d / SSC;
    int ns = 1;
    for (int c = 2; c <= 8 && blocks * ns < 256; c++)
        if (nss % c == 0 && mfma_k_ok(d / c)) ns = c;
    return ns;
}

size_t q4_gemm_mfma_ws(int T, int m, int d, int group) {
    const int ns = q4_gemm_splits(T, m, d);
    return pad256(f6_rec_bytes(T, d)) + pad256((size_t)T * (d / group)) + pad256((size_t)T * (d / group) * 4) +
           (ns > 1 ? pad256((size_t)ns * T * m * 4) : 0);
}

hipError_t launch_q4_gemm_mfma(const uint8_t* packed, const uint16_t* scales, const float* X, int T, int m, int d,
                               int group, void* ws, float* out, hipStream_t st) {
    if (T == 0 || m == 0) return hipSuccess;
    if (!q4_gemm_mfma_ok(m, d, group)) return hipErrorInvalidValue;
    uint8_t* xq = (uint8_t*)ws;
    uint8_t* xe = xq + pad256(f6_rec_bytes(T, d));
    float* xc = (float*)(xe + pad256((size_t)T * (d / group)));
    float* part = (float*)((char*)xc + pad256((size_t)T * (d / group) * 4));
    const unsigned pblocks = (unsigned)(((long long)T * (d / 16) + 255) / 256);
    const int ns = q4_gemm_splits(T, m, d);
    const int kl = d / ns;
    float* dst = ns > 1 ? part : out;
    const dim3 grid((unsigned)((T + MT - 1) / MT), (unsigned)(m / DN_ROWS), (unsigned)ns);
#define JM_QG(GG, N) hipLaunchKernelGGL((k_q4_gemm_mfma<GG, N>), grid, dim3(MTHREADS), 0, st, packed, scales, xq, xe, xc, T, m, d, kl, dst)
#define JM_QGG(GG) do { hipLaunchKernelGGL(k_prep_f6<GG>, dim3(pblocks), dim3(256), 0, st, X, T, d, xq, xe, xc); \
                        if (kl / SSC == 1) JM_QG(GG, 1); else if (kl / SSC == 3) JM_QG(GG, 3); else JM_QG(GG, 0); } while (0)
    if (group == 64) JM_QGG(64);
    else JM_QGG(32);
#undef JM_QGG
#undef JM_QG
    if (ns > 1) {
        const long long n4 = (long long)T * m / 4;
        hipLaunchKernelGGL(k_sum_splits, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, (const float4*)part, n4,
                           ns, (float4*)out);
    }
    return hipGetLastError();
}

}  // namespace jm
