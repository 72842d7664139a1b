// Decoder-layer kernels around the MoE block: the bf16 projections (with the
// RMSNorm before them and the residual add after them fused in), decode
// attention over a bf16 KV cache, and the final RMSNorm.  They follow the
// reference's layer_attn_batch / decode_layers_batch
// (decode_kernel.c:1120-1234, 1518-1556) step for step, regrouped into few
// launches:
//
//   k_gemv_part   Wq/Wk/Wv . (h * norm1 weight), per 512-column slice
//                                                             (:224-230, :1126-1145)
//   k_qk_ss       whole-vector QK-norm only: each token's sums of squares
//                 of q and k                                   (:1155-1167)
//   k_attn_part   the slices summed, RMSNorm row scale, bias, per-head or
//                 whole-vector QK-norm and RoPE of the block's heads (:1146-1199; the k
//                 and v rows appended to the cache by the split that holds
//                 the token's position), then scores, softmax and P.V over
//                 one 128-position split of the cache           (:1200-1222)
//   k_attn_comb   the splits merged per head                   (flash-decoding merge)
//   k_attn_tile   instead of the two, a prompt's positions over one bf16 cache
//   k_gemv_part   Wo . att per slice; the MoE router sums the slices into
//                 the residual                                  (:1225-1232, :1546-1547)
//   k_rms_rows    the final RMSNorm                            (:1556)
//
// The projections are HBM-bound GEMVs split over 512-column slices: every
// 16-byte weight load of a lane serves all the batch's tokens, whose slice
// (16 KiB at 8 tokens) sits in LDS, and the consumer adds the slices.
// Attention streams the cache once: one block per (position split, KV head,
// token) reads 128 positions of K and V (256 bytes each per head) and serves
// every query head of that KV head.
#include "jm_device.h"
#include "jm_kernels.h"

namespace jm {

// ------------------------------------------------------------------ GEMV

// Partial products of column slices: part[s][b][row] = sum over the
// columns k of slice s of W[row][k] * x[b][k] (* norm_w[k]), rows of the
// stacked matrices w[0..2], on the matrix cores.  Block (row group, slice,
// group of 8 tokens): WV waves of 16 rows.  v_mfma_f32_16x16x32_bf16 with
// the weight rows as the A operand straight from memory (lane l: row
// row0 + l % 16, columns 32 ks + 8 (l / 16) .. + 7, one 16-byte load per
// k-step, all requested first) and the tokens as B columns: column n < 8
// holds bf16(x) of token n, column n + 8 the rest bf16(x - bf16(x)); the
// block stages them in LDS in operand order.  Columns n and n ^ 8 of the
// product (one DPP move) add up to the token's dot product at float32-level
// accuracy.  The consumer sums the slices (and applies the RMSNorm row
// scale), so that a projection spreads over hundreds of waves.
template <int SW, int WV>
__global__ void __launch_bounds__(WV * 64)
k_gemv_part(GemvArgs a) {
    constexpr int NK = SW / 32;                    // k-steps
    __shared__ __align__(16) uint4 xb[NK][64];     // B operands, [k-step][lane]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int g = lane >> 4, n = lane & 15;
    const int slice = blockIdx.y, tb0 = blockIdx.z * 8;
    const int row0 = (blockIdx.x * WV + w) * 16;
    const int k0 = slice * SW;
    const bool live = row0 < a.N;                  // wave-uniform
    // this wave's rows (a 16-row tile lies in one matrix: rows[i] % 16 == 0)
    const int row = live ? row0 + n : 0;
    const uint16_t* wr;
    if (row < a.rows[0]) wr = a.w[0] + (size_t)row * a.K;
    else if (row < a.rows[0] + a.rows[1]) wr = a.w[1] + (size_t)(row - a.rows[0]) * a.K;
    else wr = a.w[2] + (size_t)(row - a.rows[0] - a.rows[1]) * a.K;
    const uint16_t* wp = wr + k0 + 8 * g;
    // requests first: the tokens' slice (needed first; thread tid serves
    // token tb0 + tid % 8 throughout), then the weight rows
    constexpr int NI = NK * 32;                    // staging items (8 columns of one token)
    constexpr int XI = (NI + WV * 64 - 1) / (WV * 64);     // per thread, the last one partial
    static_assert((WV * 64) % 8 == 0, "token fixed per thread");
    const int tx = tid & 7;
    const bool tin = tb0 + tx < a.B;
    float4 xv[XI][2];
    uint4 nwv[XI];
#pragma unroll
    for (int it = 0; it < XI; it++) {
        const int i = (tid + it * WV * 64) % NI;   // items past NI repeat one (same token), not stored
        const int c = k0 + 32 * (i >> 5) + 8 * ((i >> 3) & 3);
        const float4* xp = (const float4*)(a.x + (size_t)(tin ? tb0 + tx : tb0) * a.K + c);
        xv[it][0] = xp[0];
        xv[it][1] = xp[1];
        if (a.norm_w) nwv[it] = *(const uint4*)(a.norm_w + c);
    }
    uint4 wa[NK];
#pragma unroll
    for (int ks = 0; ks < NK; ks++) wa[ks] = *(const uint4*)(wp + 32 * ks);
    __builtin_amdgcn_sched_barrier(0);             // keep every request ahead of the staging
    // the tokens' slice (times the norm weight), split into hi and lo
    // columns; with a.rss the first row group's blocks also sum the squares
    // of the slice (before the norm weight) per token
    __shared__ float ssw[WV][8];
    const bool want_ss = a.rss && blockIdx.x == 0;    // block-uniform
    float ss = 0.0f;
#pragma unroll
    for (int it = 0; it < XI; it++) {
        const int i = tid + it * WV * 64;
        if (NI % (WV * 64) != 0 && i >= NI) break;         // the partial last item of the thread
        const int ks = i >> 5, gg = (i >> 3) & 3;
        float v[8] = {xv[it][0].x, xv[it][0].y, xv[it][0].z, xv[it][0].w,
                      xv[it][1].x, xv[it][1].y, xv[it][1].z, xv[it][1].w};
        if (tin) {
#pragma unroll
            for (int e = 0; e < 8; e++) ss = __builtin_fmaf(v[e], v[e], ss);
            if (a.norm_w) {
                const uint32_t nn[4] = {nwv[it].x, nwv[it].y, nwv[it].z, nwv[it].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[2 * e] = __fmul_rn(v[2 * e], bf16_bits_to_f32(nn[e] & 0xFFFFu));
                    v[2 * e + 1] = __fmul_rn(v[2 * e + 1], bf16_bits_to_f32(nn[e] >> 16));
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = 0.0f;
        }
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) split_bf16x2(v[2 * e], v[2 * e + 1], hi[e], lo[e]);
        xb[ks][16 * gg + tx] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        xb[ks][16 * gg + 8 + tx] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
    if (want_ss) {
        // lanes with equal lane % 8 serve one token
        ss = __fadd_rn(ss, __shfl_xor(ss, 8, JM_WAVE));
        ss = __fadd_rn(ss, __shfl_xor(ss, 16, JM_WAVE));
        ss = __fadd_rn(ss, __shfl_xor(ss, 32, JM_WAVE));
        if (lane < 8) ssw[w][lane] = ss;
    }
    __syncthreads();
    if (want_ss && tid < 8 && tb0 + tid < a.B) {
        float t = ssw[0][tid];
#pragma unroll
        for (int u = 1; u < WV; u++) t = __fadd_rn(t, ssw[u][tid]);
        a.rss[(size_t)slice * a.B + tb0 + tid] = t;
    }
    if (!live) return;

    // two accumulators break the dependence chain of the k-steps
    floatx4 acc[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int ks = 0; ks < NK; ks++)
        acc[ks & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wa[ks]),
                                                              __builtin_bit_cast(bf16x8, xb[ks][lane]),
                                                              acc[ks & 1], 0, 0, 0);
    // lane (g, n): rows row0 + 4 g + i of column n; token n = hi + lo columns
    float tot[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float c = __fadd_rn(acc[0][i], acc[1][i]);
        tot[i] = __fadd_rn(c, dpp_f<DPP_ROR8>(c));
    }
    if (n < 8 && tb0 + n < a.B)
        *(float4*)(a.part + ((size_t)slice * a.B + tb0 + n) * a.N + row0 + 4 * g) =
            make_float4(tot[0], tot[1], tot[2], tot[3]);
}

// ------------------------------------------------------------------ GEMM
//
// The same product for many tokens at once (a prefill chunk): part[0][b][row]
// = sum over all K columns of W[row][k] * x[b][k] (* norm_w[k]), one output
// slice.  Block (128-row tile, 64-token tile), 8 waves: 2 token halves x 4
// row quarters of 32, each wave a 32 x 32 tile by v_mfma_f32_32x32x16_bf16
// with the tokens on the A side (split into bf16 hi and lo, two products
// per k-step, as the GEMV splits them) and the weight rows on the B side.
// Operands go through LDS in 64-column stages, two stages streaming into
// registers while the stage in LDS is multiplied.  Lane layout as the dense
// expert branch's: A[i][k] at lane i % 32, k = 8 (l / 32) + j; B[k][n] at
// lane n % 32, k = 8 (l / 32) + j; D register v of lane l = (i = 8 (v / 4)
// + 4 (l / 32) + v % 4, n = l % 32).  Each weight byte crosses HBM once per
// token tile instead of once per 8 tokens.
constexpr int GM_T = 64;            // tokens per block
constexpr int GM_R = 128;           // weight rows per block
constexpr int GM_KS = 64;           // columns per stage
constexpr int GM_KP = GM_KS + 8;    // padded LDS row, in bf16 (144 bytes: 16-byte aligned, bank-spread)

struct GmStage {
    float4 x0, x1;                  // 8 columns of one token
    uint4 nw;                       // their norm weights (bf16)
    uint4 w[2];                     // 2 x 8 columns of weight rows
    int s;                          // the stage (before clamping to the last one)
};

__global__ void __launch_bounds__(512, 1)
k_gemm_bf16(GemvArgs a) {
    typedef float floatx16 __attribute__((ext_vector_type(16)));
    __shared__ __align__(16) uint16_t xh[2][GM_T * GM_KP], xl[2][GM_T * GM_KP], wl[2][GM_R * GM_KP];
    __shared__ float ss_l[GM_T][8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // the first row tile also sums each token's squares (the RMSNorm of the
    // layer input, for the consumer) from the values it stages
    const bool want_ss = a.rss && blockIdx.x == 0;
    float ss = 0.0f;
    const int row0 = blockIdx.x * GM_R, tb0 = blockIdx.y * GM_T;
    // block z takes the z-th of gridDim.z equal column ranges and writes
    // slice z of part (and of rss)
    const int K = a.K, nstage = K / GM_KS / (int)gridDim.z, kz = blockIdx.z;
    const int kcol0 = kz * nstage * GM_KS;
    // the 128-row tile lies in one matrix (row counts are multiples of 128)
    const uint16_t* wm;
    int wr0;
    if (row0 < a.rows[0]) { wm = a.w[0]; wr0 = row0; }
    else if (row0 < a.rows[0] + a.rows[1]) { wm = a.w[1]; wr0 = row0 - a.rows[0]; }
    else { wm = a.w[2]; wr0 = row0 - a.rows[0] - a.rows[1]; }
    // staging: token xt, columns 8 xp .. 8 xp + 7; weight rows wrw and
    // wrw + 64, columns 8 wp .. 8 wp + 7
    const int xt = tid >> 3, xp = tid & 7;
    const int wrw = tid >> 3, wp = tid & 7;
    const bool xlive = tb0 + xt < a.B;
    const float* xrow = a.x + (size_t)(xlive ? tb0 + xt : 0) * K + kcol0 + 8 * xp;
    const uint16_t* wp0 = wm + (size_t)(wr0 + wrw) * K + kcol0 + 8 * wp;
    const uint16_t* wp1 = wp0 + (size_t)64 * K;

    // every load is unconditional (past the last stage: the last stage again)
    auto load_stage = [&](GmStage& r, int s) __attribute__((always_inline)) {
        r.s = s;
        s = s < nstage ? s : nstage - 1;
        const float4* xs = (const float4*)(xrow + s * GM_KS);
        r.x0 = xs[0];
        r.x1 = xs[1];
        if (a.norm_w) r.nw = *(const uint4*)(a.norm_w + kcol0 + s * GM_KS + 8 * xp);
        r.w[0] = *(const uint4*)(wp0 + s * GM_KS);
        r.w[1] = *(const uint4*)(wp1 + s * GM_KS);
    };
    auto store_stage = [&](const GmStage& r, int buf) __attribute__((always_inline)) {
        float v[8] = {r.x0.x, r.x0.y, r.x0.z, r.x0.w, r.x1.x, r.x1.y, r.x1.z, r.x1.w};
        if (want_ss && r.s < nstage) {
#pragma unroll
            for (int e = 0; e < 8; e++) ss = __builtin_fmaf(v[e], v[e], ss);
        }
        if (a.norm_w) {
            const uint32_t nn[4] = {r.nw.x, r.nw.y, r.nw.z, r.nw.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[2 * e] = __fmul_rn(v[2 * e], bf16_bits_to_f32(nn[e] & 0xFFFFu));
                v[2 * e + 1] = __fmul_rn(v[2 * e + 1], bf16_bits_to_f32(nn[e] >> 16));
            }
        }
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) split_bf16x2(v[2 * e], v[2 * e + 1], hi[e], lo[e]);
        const unsigned keep = xlive ? 0xFFFFFFFFu : 0u;     // tokens past B stage zeros
        *(uint4*)&xh[buf][xt * GM_KP + 8 * xp] = make_uint4(hi[0] & keep, hi[1] & keep, hi[2] & keep, hi[3] & keep);
        *(uint4*)&xl[buf][xt * GM_KP + 8 * xp] = make_uint4(lo[0] & keep, lo[1] & keep, lo[2] & keep, lo[3] & keep);
        *(uint4*)&wl[buf][wrw * GM_KP + 8 * wp] = r.w[0];
        *(uint4*)&wl[buf][(wrw + 64) * GM_KP + 8 * wp] = r.w[1];
    };

    const int th = w & 1, rq = w >> 1;            // this wave's token half and row quarter
    const int ai = th * 32 + (lane & 31), bn = rq * 32 + (lane & 31), kq = 8 * (lane >> 5);
    floatx16 acc = {};
    auto mfma_stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k2 = 0; k2 < GM_KS / 16; k2++) {
            const int k0 = k2 * 16 + kq;
            const bf16x8 a_h = *(const bf16x8*)&xh[buf][ai * GM_KP + k0];
            const bf16x8 a_l = *(const bf16x8*)&xl[buf][ai * GM_KP + k0];
            const bf16x8 b = *(const bf16x8*)&wl[buf][bn * GM_KP + k0];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_h, b, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_l, b, acc, 0, 0, 0);
        }
    };
    // stages s + 1 and s + 2 stream into registers while stage s (in LDS) is
    // multiplied; nstage is even
    GmStage r0, r1;
    load_stage(r0, 0);
    load_stage(r1, 1);
    store_stage(r0, 0);
    load_stage(r0, 2);
    __syncthreads();
    for (int s = 0; s < nstage; s += 2) {
        mfma_stage(0);
        store_stage(r1, 1);
        load_stage(r1, s + 3);
        __syncthreads();
        mfma_stage(1);
        store_stage(r0, 0);
        load_stage(r0, s + 4);
        __syncthreads();
    }
    const int n = row0 + bn;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int t = tb0 + th * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
        if (t < a.B) a.part[((size_t)kz * a.B + t) * a.N + n] = acc[v];
    }
    if (want_ss) {
        ss_l[xt][xp] = ss;
        __syncthreads();
        if (tid < GM_T && tb0 + tid < a.B) {
            float t = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) t = __fadd_rn(t, ss_l[tid][i]);
            a.rss[(size_t)kz * a.B + tb0 + tid] = t;
        }
    }
}

// The same product for the larger grids (gemm_plan): block (256-row tile,
// 64-token tile, column range), 4 waves of 64 tokens x 64 rows each, which
// read 6 operands from LDS per 8 MFMAs where k_gemm_bf16's 32 x 32 waves read
// 12, and two blocks per CU instead of one, so that one multiplies while the
// other waits for its stage.  The stage is 64 columns, so that a weight row's
// part is a whole 128-byte line (32-column stages fetched each line twice:
// 152 us against 141 for the first case below), in one LDS buffer.  At 301
// tokens, weights from HBM, us per launch in its best column ranges, against
// k_gemm_bf16 in its own: rows x columns 24576 x 4096 146 (1) vs 181 (1), 4096
// x 12288 94 (4) vs 110 (1), 4096 x 4096 37 (4) vs 41 (1).  What bounds it: a
// stage's loads, LDS writes and reads take about 1.7 us for a pair of blocks,
// of which the MFMAs are 0.85; reading the next stage's operands ahead from a
// third LDS buffer measured 158 for the first case, and two stages in registers
// no better.
constexpr int GW_R = 256;           // weight rows per block

struct GwStage {
    float4 x[2][2];                 // 8 columns of two tokens
    uint4 nw;                       // their norm weights (bf16)
    uint4 w[GW_R / 32];             // 8 columns of weight rows 32 apart
};

// Offset in bf16 of 8-column chunk c of row r of a staged operand: rows of 128
// bytes, the chunk rotated by the row so that the rows one read phase touches
// at one chunk, and the whole rows a write phase touches, spread over every
// bank.
__device__ __forceinline__ int gw_at(int r, int c) { return r * GM_KS + 8 * (c ^ ((r >> 1) & 7) ^ (4 * (r & 1))); }

template <bool NORM>
__global__ void __launch_bounds__(256, 2)
k_gemm_bf16_wide(GemvArgs a) {
    typedef float floatx16 __attribute__((ext_vector_type(16)));
    constexpr int NW = GW_R / 32;
    __shared__ __align__(16) uint16_t xh[GM_T * GM_KS], xl[GM_T * GM_KS], wl[GW_R * GM_KS];
    __shared__ float ss_l[GM_T][8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // the first row tile also sums each token's squares (the RMSNorm of the
    // layer input, for the consumer) from the values it stages
    const bool want_ss = a.rss && blockIdx.x == 0;
    float ss[2] = {};
    const int row0 = blockIdx.x * GW_R, tb0 = blockIdx.y * GM_T;
    // block z takes the z-th of gridDim.z equal column ranges and writes
    // slice z of part (and of rss)
    const int K = a.K, nstage = K / GM_KS / (int)gridDim.z, kz = blockIdx.z;
    const int kcol0 = kz * nstage * GM_KS;
    // the row tile lies in one matrix (row counts are multiples of GW_R)
    const uint16_t* wm;
    int wr0;
    if (row0 < a.rows[0]) { wm = a.w[0]; wr0 = row0; }
    else if (row0 < a.rows[0] + a.rows[1]) { wm = a.w[1]; wr0 = row0 - a.rows[0]; }
    else { wm = a.w[2]; wr0 = row0 - a.rows[0] - a.rows[1]; }
    // staging: tokens sr and sr + 32, columns 8 sc .. 8 sc + 7; the same
    // columns of weight rows sr + 32 i
    const int sr = tid >> 3, sc = tid & 7;
    const bool live[2] = {tb0 + sr < a.B, tb0 + sr + 32 < a.B};
    const float* xrow[2];
#pragma unroll
    for (int q = 0; q < 2; q++) xrow[q] = a.x + (size_t)(live[q] ? tb0 + sr + 32 * q : 0) * K + kcol0 + 8 * sc;
    const uint16_t* wrow = wm + (size_t)(wr0 + sr) * K + kcol0 + 8 * sc;
    const int sto = gw_at(sr, sc);                // (rows 32 apart rotate alike)

    // every load is unconditional (past the last stage: the last stage again)
    auto load_stage = [&](GwStage& r, int s) __attribute__((always_inline)) {
        s = s < nstage ? s : nstage - 1;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const float4* xs = (const float4*)(xrow[q] + s * GM_KS);
            r.x[q][0] = xs[0];
            r.x[q][1] = xs[1];
        }
        r.nw = NORM ? *(const uint4*)(a.norm_w + kcol0 + s * GM_KS + 8 * sc) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < NW; i++) r.w[i] = *(const uint4*)(wrow + (size_t)(32 * i) * K + s * GM_KS);
    };
    auto store_stage = [&](const GwStage& r) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NW; i++) *(uint4*)&wl[32 * i * GM_KS + sto] = r.w[i];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            float v[8] = {r.x[q][0].x, r.x[q][0].y, r.x[q][0].z, r.x[q][0].w,
                          r.x[q][1].x, r.x[q][1].y, r.x[q][1].z, r.x[q][1].w};
            if (NORM) {
#pragma unroll
                for (int e = 0; e < 8; e++) ss[q] = __builtin_fmaf(v[e], v[e], ss[q]);
                const uint32_t nn[4] = {r.nw.x, r.nw.y, r.nw.z, r.nw.w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[2 * e] = __fmul_rn(v[2 * e], bf16_bits_to_f32(nn[e] & 0xFFFFu));
                    v[2 * e + 1] = __fmul_rn(v[2 * e + 1], bf16_bits_to_f32(nn[e] >> 16));
                }
            }
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; e++) split_bf16x2(v[2 * e], v[2 * e + 1], hi[e], lo[e]);
            const unsigned keep = live[q] ? 0xFFFFFFFFu : 0u;     // tokens past B stage zeros
            *(uint4*)&xh[32 * q * GM_KS + sto] = make_uint4(hi[0] & keep, hi[1] & keep, hi[2] & keep, hi[3] & keep);
            *(uint4*)&xl[32 * q * GM_KS + sto] = make_uint4(lo[0] & keep, lo[1] & keep, lo[2] & keep, lo[3] & keep);
        }
    };

    const int wn0 = 64 * w;                       // this wave's first weight row within the block's tile
    floatx16 acc[2][2] = {};
    auto mfma_stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k2 = 0; k2 < GM_KS / 16; k2++) {
            const int off = gw_at(lane & 31, 2 * k2 + (lane >> 5));     // (rows 32 apart rotate alike)
            bf16x8 ah[2], al[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                ah[i] = *(const bf16x8*)&xh[32 * i * GM_KS + off];
                al[i] = *(const bf16x8*)&xl[32 * i * GM_KS + off];
            }
#pragma unroll
            for (int j = 0; j < 2; j++) b[j] = *(const bf16x8*)&wl[(wn0 + 32 * j) * GM_KS + off];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    // stage s + 1 streams into registers while stage s (in LDS) is multiplied
    GwStage r;
    load_stage(r, 0);
    for (int s = 0; s < nstage; s++) {
        store_stage(r);
        load_stage(r, s + 1);
        __syncthreads();
        mfma_stage();
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int t = tb0 + 32 * i + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
            if (t >= a.B) continue;
            float* out = a.part + ((size_t)kz * a.B + t) * a.N + row0 + wn0 + (lane & 31);
#pragma unroll
            for (int j = 0; j < 2; j++) out[32 * j] = acc[i][j][v];
        }
    if (NORM && want_ss) {
#pragma unroll
        for (int q = 0; q < 2; q++) ss_l[sr + 32 * q][sc] = ss[q];
        __syncthreads();
        if (tid < GM_T && tb0 + tid < a.B) {
            float t = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) t = __fadd_rn(t, ss_l[tid][i]);
            a.rss[(size_t)kz * a.B + tb0 + tid] = t;
        }
    }
}

bool gemm_shape_ok(const GemvArgs& a) {
    return a.K % (2 * GM_KS) == 0 && a.rows[0] % GM_R == 0 && a.rows[1] % GM_R == 0 && a.rows[2] % GM_R == 0;
}

static int device_cus() {
    static int ncu = 0;
    if (ncu == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu <= 0)
            ncu = 256;
    }
    return ncu;
}

// Column ranges (K slices) of k_gemm_bf16, 1, 2 or 4: one block per CU runs at
// a time, so a grid of (N / 128) x (B / 64) tiles that leaves CUs idle in
// its last round is split along K into more, shorter blocks.  Time is
// modelled as rounds x (1 / slices + 0.15), the constant a block's fixed
// part (prologue, output stores); ties keep fewer slices (fewer partial
// outputs to write and sum).
static int gemm_slices_narrow(const GemvArgs& a) {
    const int ncu = device_cus();
    const long long tiles = (long long)(a.N / GM_R) * ((a.B + GM_T - 1) / GM_T);
    const int nstage = a.K / GM_KS;
    int best = 1;
    double best_t = 1e30;
    for (int kz : {1, 2, 4}) {
        if (nstage % (2 * kz) != 0) continue;
        const long long rounds = (tiles * kz + ncu - 1) / ncu;
        const double t = (double)rounds * (1.0 / kz + 0.15);
        if (t < best_t - 1e-9) {
            best_t = t;
            best = kz;
        }
    }
    return best;
}

// Which kernel takes a, and in how many column ranges.  Both are priced in
// microseconds, for the 64-column stages of a block and the blocks a CU gets:
// k_gemm_bf16, in gemm_slices_narrow's ranges, 0.6 per stage and 3.5 per block,
// one block at a time; the wide tile 1.71 per stage of two blocks sharing a CU
// or 1.32 of one alone, 6 per such round and 1.5 once.  Each slice is written
// here and read by the consumer, together at about 2.2 TB/s.  The constants are
// fitted to both kernels' times in 1, 2 and 4 ranges on cold weights: rows x
// columns 2048 x 2048, 2048 x 4096, 4096 x 4096, 4096 x 12288, 5120 x 2048,
// 6144 x 2048, 6144 x 4096 and 24576 x 4096 at 16 token counts of 33 to 512.
// Over these 128 the rule is within 0.4% of the better kernel on average and
// never behind k_gemm_bf16 alone (slices' cost included), 2.4% ahead of it.  Some
// lines, us, narrow (ranges) vs wide (ranges) with the slices' cost: 24576 x
// 4096 at 64 tokens 54 (1) vs 56 (1), 65 76 (2) vs 71 (2), 129 118 (2) vs 115
// (4), 257 180 (1) vs 145 (1); 4096 x 12288 at 256 tokens 75 (2) vs 82 (4), 257
// 110 (1) vs 96 (4); 6144 x 4096 at 128 tokens 27 (2) vs 35 (4), 129 43 (1) vs
// 36 (4).  At 6144 x 4096 and 256 to 320 tokens it keeps the narrow kernel, 46 to
// 51, where 4 wide ranges take 43 to 47; 5120 x 2048 goes wide from 448 tokens
// (39 vs 38).
struct GemmPlan {
    bool wide;
    int kz;
};

static GemmPlan gemm_plan(const GemvArgs& a) {
    const int ncu = device_cus(), tt = (a.B + GM_T - 1) / GM_T, nstage = a.K / GM_KS;
    GemmPlan p{false, gemm_slices_narrow(a)};
    // (the wide kernel sums squares only where it applies a norm weight)
    if (a.rows[0] % GW_R != 0 || a.rows[1] % GW_R != 0 || a.rows[2] % GW_R != 0 || (a.rss && !a.norm_w)) return p;
    const double slice = (double)a.B * a.N * 4 / 2.2e6;
    const long long nb = ((long long)(a.N / GM_R) * tt * p.kz + ncu - 1) / ncu;
    double best = (double)nb * (0.6 * nstage / p.kz + 3.5) + slice * p.kz;
    for (int kz : {1, 2, 4}) {
        if (nstage % (2 * kz) != 0) continue;
        const long long n = ((long long)(a.N / GW_R) * tt * kz + ncu - 1) / ncu;
        const double t = (double)nstage / kz * (1.71 * (n / 2) + 1.32 * (n % 2)) + 6.0 * ((n + 1) / 2) + 1.5 + slice * kz;
        if (t < best) {
            best = t;
            p = {true, kz};
        }
    }
    return p;
}

int gemm_slices(const GemvArgs& a) { return gemm_plan(a).kz; }
bool gemm_wide(const GemvArgs& a) { return gemm_plan(a).wide; }

hipError_t launch_gemm_bf16(const GemvArgs& a, hipStream_t st) {
    if (a.B == 0 || a.N == 0) return hipSuccess;
    if (!gemm_shape_ok(a)) return hipErrorInvalidValue;
    const GemmPlan p = gemm_plan(a);
    const int rb = p.wide ? GW_R : GM_R;
    const dim3 grid((unsigned)(a.N / rb), (unsigned)((a.B + GM_T - 1) / GM_T), (unsigned)p.kz);
    if (!p.wide) hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(512), 0, st, a);
    else if (a.norm_w) hipLaunchKernelGGL(k_gemm_bf16_wide<true>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_gemm_bf16_wide<false>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

bool gemv_shape_ok(int K) { return K > 0 && K % 1024 == 0 && K <= 8192; }

int gemv_slice_cols(int K) { return K >= 4096 && K % 1024 == 0 ? 1024 : 512; }

// Waves per block (16 rows each) of a projection: the one of 5, 4 and 2
// whose grid fills its last round of the CUs best (one block per CU and
// round), the larger on ties.  A grid of 1.25 rounds (320 blocks on 256
// CUs) leaves the CUs with two blocks to set the time.
static int gemv_waves(int N, int slices, int zgroups) {
    const int ncu = device_cus();
    int best = 4;
    double best_eff = -1.0;
    for (int wv : {5, 4, 2}) {
        const long long nb = (long long)((N + 16 * wv - 1) / (16 * wv)) * slices * zgroups;
        const long long rounds = (nb + ncu - 1) / ncu;
        const double eff = (double)nb / (double)(rounds * ncu);
        if (eff > best_eff + 1e-9) {
            best_eff = eff;
            best = wv;
        }
    }
    return best;
}

hipError_t launch_gemv_part(const GemvArgs& a, hipStream_t st) {
    if (a.B == 0 || a.N == 0) return hipSuccess;
    if (a.rows[0] % 16 || a.rows[1] % 16 || a.rows[2] % 16) return hipErrorInvalidValue;
    const int sw = gemv_slice_cols(a.K);
    const int zg = (a.B + 7) / 8;
    const int wv = gemv_waves(a.N, a.K / sw, zg);
    const dim3 grid((unsigned)((a.N + 16 * wv - 1) / (16 * wv)), (unsigned)(a.K / sw), (unsigned)zg);
#define JM_GV(SWV, WVV) hipLaunchKernelGGL((k_gemv_part<SWV, WVV>), grid, dim3(WVV * 64), 0, st, a)
    if (sw == 1024) {
        if (wv == 5) JM_GV(1024, 5);
        else if (wv == 2) JM_GV(1024, 2);
        else JM_GV(1024, 4);
    } else {
        if (wv == 5) JM_GV(512, 5);
        else if (wv == 2) JM_GV(512, 2);
        else JM_GV(512, 4);
    }
#undef JM_GV
    return hipGetLastError();
}

// ------------------------------------------------------------- attention

// Partial sums over 16 lanes of QPK per-head dot products; head h's total
// ends in the lanes j (= lane % 16) with j / (16 / QPK) == h.
template <int QPK>
__device__ __forceinline__ float head_reduce16(float (&v)[QPK]) {
    if constexpr (QPK == 8) {
        transpose_level<8, 8>(v);
        transpose_level<4, 4>(v);
        const bool hi = (threadIdx.x & 2) != 0;
        const float keep = hi ? v[1] : v[0], send = hi ? v[0] : v[1];
        float t = __fadd_rn(keep, dpp_f<DPP_XOR2>(send));
        return __fadd_rn(t, dpp_f<DPP_XOR1>(t));
    } else {
        return transpose_reduce<16, QPK>(v);
    }
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_round(float f) { return __uint_as_float(f32_to_bf16_rne(f) << 16); }

// Four consecutive projection values of one token (rows row .. row + 3 of
// the stacked q, k, v outputs, dimensions 4 j .. 4 j + 3 of one head) with
// everything their finish reads, requested together: the first
// min(nslice, 4) column slices, the slices' sums of squares of h, the bias,
// the per-head norm weight and the RoPE factors at pos.
struct Fin4 {
    float4 sl[4];
    float rs[4];
    float4 bias;
    uint2 nw;
    float4 c, sn;
};

__device__ __forceinline__ void fin4_load(Fin4& f, const AttnArgs& a, int b, int row, const float* bias, int brow,
                                          const uint16_t* nw, bool rope, int pos, int j) {
    constexpr int HD = 128;
    const int ns = a.nslice < 4 ? a.nslice : 4;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int sl = u < ns ? u : 0;          // clamped: the select in fin4_value drops it
        f.sl[u] = *(const float4*)(a.qkv + ((size_t)sl * a.B + b) * a.nqkv + row);
        f.rs[u] = a.rss[(size_t)sl * a.B + b];
    }
    f.bias = bias ? *(const float4*)(bias + brow) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    f.nw = nw ? *(const uint2*)(nw + 4 * j) : make_uint2(0u, 0u);
    if (rope) {
        const size_t ci = (size_t)pos * HD + 4 * (j & 15);
        f.c = *(const float4*)(a.cos + ci);
        f.sn = *(const float4*)(a.sin + ci);
    }
}

// The norm weight of q head (isq) or k head `head` of the layer: per head,
// the one [128] vector; over the whole vector, the head's 128 entries.
__device__ __forceinline__ const uint16_t* qk_weight(const AttnArgs& a, bool isq, int head) {
    const uint16_t* w = isq ? a.qn : a.kn;
    if (!w) return nullptr;
    return a.qk_norm == 2 ? w + (size_t)head * 128 : w;
}

// The four values finished (decode_kernel.c:1126-1199): the column slices
// summed in slice order, times the RMSNorm row scale of h (the projections
// were taken of h * norm weight), plus the bias; then, for a q or k head,
// the QK-norm with weight nw (norm 1: the head's RMSNorm, :1174-1189;
// norm 2: the whole vector's, with its sum of squares from k_qk_ss,
// :1155-1167) and RoPE rotate-half at
// pos (:1190-1194, :259-266) over the aligned 32-lane segment that holds
// the head (lane j: dimensions 4 j .. 4 j + 3; dim i pairs with i + 64,
// i.e. lane j with j ^ 16; first half a cos - b sin, second a sin + b cos).
__device__ __forceinline__ void fin4_value(float (&v)[4], const Fin4& f, const AttnArgs& a, int b, int row,
                                           int norm, bool rope, int j) {
    constexpr int HD = 128;
    const int ns = a.nslice < 4 ? a.nslice : 4;
    float4 acc = f.sl[0];
    float ss = f.rs[0];
#pragma unroll
    for (int u = 1; u < 4; u++) {
        const bool in = u < ns;
        acc.x = in ? __fadd_rn(acc.x, f.sl[u].x) : acc.x;
        acc.y = in ? __fadd_rn(acc.y, f.sl[u].y) : acc.y;
        acc.z = in ? __fadd_rn(acc.z, f.sl[u].z) : acc.z;
        acc.w = in ? __fadd_rn(acc.w, f.sl[u].w) : acc.w;
        ss = in ? __fadd_rn(ss, f.rs[u]) : ss;
    }
    for (int sl = 4; sl < a.nslice; sl++) {     // wider inputs (d = 3072, 8192): the rest of the slices
        const float4 t = *(const float4*)(a.qkv + ((size_t)sl * a.B + b) * a.nqkv + row);
        acc.x = __fadd_rn(acc.x, t.x);
        acc.y = __fadd_rn(acc.y, t.y);
        acc.z = __fadd_rn(acc.z, t.z);
        acc.w = __fadd_rn(acc.w, t.w);
        ss = __fadd_rn(ss, a.rss[(size_t)sl * a.B + b]);
    }
    const float inv = rms_inv(ss, a.d, a.eps);
    v[0] = __fadd_rn(__fmul_rn(acc.x, inv), f.bias.x);
    v[1] = __fadd_rn(__fmul_rn(acc.y, inv), f.bias.y);
    v[2] = __fadd_rn(__fmul_rn(acc.z, inv), f.bias.z);
    v[3] = __fadd_rn(__fmul_rn(acc.w, inv), f.bias.w);
    if (norm) {
        float hinv;
        if (norm == 1) {
            float sq = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) sq = __builtin_fmaf(v[e], v[e], sq);
            // the reference sums the head's squares in dimension order; the
            // tree here changes the sum by rounding only
            hinv = rms_inv(seg_sum<32>(sq), HD, a.eps);
        } else {
            const bool isq = row < a.H * HD;
            hinv = rms_inv(a.qkss[(size_t)b * 2 + (isq ? 0 : 1)], (isq ? a.H : a.KH) * HD, a.eps);
        }
        const uint32_t nn[4] = {f.nw.x & 0xFFFFu, f.nw.x >> 16, f.nw.y & 0xFFFFu, f.nw.y >> 16};
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __fmul_rn(__fmul_rn(v[e], hinv), bf16_bits_to_f32(nn[e]));
    }
    if (rope) {
        const bool lo = j < 16;
        const float c[4] = {f.c.x, f.c.y, f.c.z, f.c.w}, sn[4] = {f.sn.x, f.sn.y, f.sn.z, f.sn.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float other = __shfl_xor(v[e], 16, JM_WAVE);
            v[e] = lo ? __builtin_fmaf(v[e], c[e], -__fmul_rn(other, sn[e]))
                      : __builtin_fmaf(other, sn[e], __fmul_rn(v[e], c[e]));
        }
    }
}

// The k and v rows of one KV head of one token, for one wave: lanes 0..31
// the k head (norm, RoPE), lanes 32..63 the v head.
struct KvFin {
    Fin4 f;
    int row;
    bool isk;
};

__device__ __forceinline__ void kv_load(KvFin& k, const AttnArgs& a, int b, int kh, int pos, int lane) {
    constexpr int HD = 128;
    k.isk = lane < 32;
    const int j = lane & 31;
    k.row = (k.isk ? a.H + kh : a.H + a.KH + kh) * HD + 4 * j;
    fin4_load(k.f, a, b, k.row, k.isk ? a.bk : a.bv, kh * HD + 4 * j, k.isk ? qk_weight(a, false, kh) : nullptr,
              k.isk, pos, j);
}

// Finished and appended to the token's caches kc, vc at pos (:1195-1199);
// with kvn, also kept there (kvn[0]: k, kvn[1]: v, bf16).
__device__ __forceinline__ void kv_store(const KvFin& k, const AttnArgs& a, int b, int kh, int pos, int lane,
                                         gptr<uint16_t> kc, gptr<uint16_t> vc, uint16_t (*kvn)[128]) {
    constexpr int HD = 128;
    const int j = lane & 31;
    float v[4];
    fin4_value(v, k.f, a, b, k.row, k.isk && a.kn ? a.qk_norm : 0, k.isk, j);
    uint16_t hb4[4];
#pragma unroll
    for (int e = 0; e < 4; e++) hb4[e] = (uint16_t)f32_to_bf16_rne(v[e]);
    if (kvn) {
#pragma unroll
        for (int e = 0; e < 4; e++) kvn[k.isk ? 0 : 1][4 * j + e] = hb4[e];
    }
    const gptr<uint16_t> dst = (k.isk ? kc : vc) + ((size_t)pos * a.KH + kh) * HD + 4 * j;
    *(uint2*)dst = make_uint2(hb4[0] | ((uint32_t)hb4[1] << 16), hb4[2] | ((uint32_t)hb4[3] << 16));
}

// The whole-vector QK-norm (decode_kernel.c:1155-1167) needs each token's
// sum of squares over all of q (H * 128 values) and all of k (KH * 128)
// before the attention blocks, which finish one KV head each, can scale
// their heads.  One block per token finishes every q and k value as
// fin4_value does (slices, row scale, bias: the same bits) and sums the
// squares; qkss[b] = (q sum, k sum).
__global__ void __launch_bounds__(256)
k_qk_ss(AttnArgs a) {
    constexpr int HD = 128;
    __shared__ float red[2][4];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int nq = a.H * HD / 4, nqk = (a.H + a.KH) * HD / 4;   // float4 groups of q, of q and k
    float sq = 0.0f, sk = 0.0f;
    for (int u = tid; u < nqk; u += 256) {
        const bool isq = u < nq;
        const int row = 4 * u;                    // q rows, then the k rows, as stacked in qkv
        Fin4 f;
        fin4_load(f, a, b, row, isq ? a.bq : a.bk, isq ? row : row - a.H * HD, nullptr, false, 0, 0);
        float v[4];
        fin4_value(v, f, a, b, row, 0, false, 0);
        float t = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) t = __builtin_fmaf(v[e], v[e], t);
        if (isq) sq = __fadd_rn(sq, t);
        else sk = __fadd_rn(sk, t);
    }
    sq = seg_sum<64>(sq);
    sk = seg_sum<64>(sk);
    if ((tid & 63) == 0) {
        red[0][tid >> 6] = sq;
        red[1][tid >> 6] = sk;
    }
    __syncthreads();
    if (tid < 2) a.qkss[(size_t)b * 2 + tid] = __fadd_rn(__fadd_rn(red[tid][0], red[tid][1]),
                                                         __fadd_rn(red[tid][2], red[tid][3]));
}

// The same for float32 caches (the reference's KVCache type): the finished
// values are appended as they are; with kvf, also kept there (kvf[0]: k,
// kvf[1]: v).
__device__ __forceinline__ void kv_store_f32(const KvFin& k, const AttnArgs& a, int b, int kh, int pos, int lane,
                                             gptr<float> kc, gptr<float> vc, float (*kvf)[128]) {
    constexpr int HD = 128;
    const int j = lane & 31;
    float v[4];
    fin4_value(v, k.f, a, b, k.row, k.isk && a.kn ? a.qk_norm : 0, k.isk, j);
    const f32x4_t v4 = f32x4_t{v[0], v[1], v[2], v[3]};
    if (kvf) *(f32x4_t*)&kvf[k.isk ? 0 : 1][4 * j] = v4;
    const gptr<float> dst = (k.isk ? kc : vc) + ((size_t)pos * a.KH + kh) * HD + 4 * j;
    *(gptr<f32x4_t>)dst = v4;
}

// For a batch whose tokens may share a cache (a prefill chunk: the
// positions of one prompt), every token's k and v rows are appended before
// the attention reads the caches: wave 0 of block (KV head, token).  With
// a.qhl the block's other waves finish the KV head's query heads, two per
// wave, for k_attn_tile: split for the matrix cores (bf16(q), bf16(q - hi))
// into qhl[token][head][2][128].
template <bool F32>
__global__ void __launch_bounds__(320)
k_kv_append(AttnArgs a) {
    constexpr int HD = 128;
    const int kh = blockIdx.x, b = blockIdx.y;
    const int pos = a.pos[b];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w > 0) {
        const int qpk = a.H / a.KH, j = threadIdx.x & 31, q = (threadIdx.x >> 5) - 2;
        const int head = kh * qpk + (q < qpk ? q : 0), row = head * HD + 4 * j;
        Fin4 f;
        fin4_load(f, a, b, row, a.bq, row, qk_weight(a, true, head), true, pos, j);
        float v[4];
        fin4_value(v, f, a, b, row, a.qn ? a.qk_norm : 0, true, j);
        uint32_t hi[2], lo[2];
        split_bf16x2(v[0], v[1], hi[0], lo[0]);
        split_bf16x2(v[2], v[3], hi[1], lo[1]);
        uint16_t* o = a.qhl + ((size_t)b * a.H + head) * 2 * HD + 4 * j;
        if (q < qpk) {
            *(uint2*)o = make_uint2(hi[0], hi[1]);
            *(uint2*)(o + HD) = make_uint2(lo[0], lo[1]);
        }
        return;
    }
    const unsigned long long* kvp = a.kv + ((size_t)b * a.L + a.layer) * 2;
    KvFin k;
    kv_load(k, a, b, kh, pos, threadIdx.x);
    if (F32) kv_store_f32(k, a, b, kh, pos, threadIdx.x, (gptr<float>)kvp[0], (gptr<float>)kvp[1], nullptr);
    else kv_store(k, a, b, kh, pos, threadIdx.x, (gptr<uint16_t>)kvp[0], (gptr<uint16_t>)kvp[1], nullptr);
}

// The 4 waves' partial outputs of a split block (wave w's at red + w *
// wstride, [QPK][128]) merged with the split's max (the flash-decoding
// merge within the block) into part_o / part_ml:
// thread tid takes head tid / 32, dimensions 4 (tid % 32) .. + 3, so that
// each thread forms the 4 waves' factors of one head once.
template <int QPK>
__device__ __forceinline__ void merge_waves(const AttnArgs& a, int b, int kh, int s, const float* red, int wstride,
                                            const float (*mls)[QPK][2]) {
    constexpr int HD = 128;
    const int tid = threadIdx.x;
    float* po = a.part_o + (((size_t)b * a.KH + kh) * a.S + s) * QPK * HD;
    {
        const int h = tid >> 5, oi = h * HD + 4 * (tid & 31);
        if (h < QPK) {
            const float M = fmaxf(fmaxf(mls[0][h][0], mls[1][h][0]), fmaxf(mls[2][h][0], mls[3][h][0]));
            float4 O = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            float L = 0.0f;
#pragma unroll
            for (int ww = 0; ww < 4; ww++) {
                const float m = mls[ww][h][0];
                const float f = m == -INFINITY ? 0.0f : expf_fast(__fsub_rn(m, M));
                const float4 r = *(const float4*)&red[(size_t)ww * wstride + oi];
                O.x = __builtin_fmaf(r.x, f, O.x);
                O.y = __builtin_fmaf(r.y, f, O.y);
                O.z = __builtin_fmaf(r.z, f, O.z);
                O.w = __builtin_fmaf(r.w, f, O.w);
                L = __builtin_fmaf(mls[ww][h][1], f, L);
            }
            *(float4*)(po + oi) = O;
            if ((tid & 31) == 0) {
                float* ml = a.part_ml + ((((size_t)b * a.KH + kh) * a.S + s) * QPK + h) * 2;
                ml[0] = M;
                ml[1] = L;
            }
        }
    }
}

// One (position split, KV head, token): QPK query heads over positions
// [128 s, 128 s + 128) of the token's T = pos + 1 cache rows (the row at pos
// finished and appended here), on the matrix cores.  Wave w takes 32 positions
// tw = 128 s + 32 w .. tw + 31 and all 128 head dimensions.
//
// Scores (:1205-1211) by v_mfma_f32_16x16x32_bf16 with the cached K rows
// as the A operand straight from memory (lane l: row tw + 16 mt + l % 16,
// dimensions 32 kk + 8 (l / 16) .. + 7, one 16-byte load) and the query
// heads as B columns: column n < 8 holds bf16(q) of head n, column n + 8 the
// rest bf16(q - bf16(q)) (split in the prologue), so the two columns' sum
// carries 16 significant bits of q against the exact bf16 keys, accumulated
// in fp32.  The sum of
// columns n and n ^ 8 (one DPP move) is the score of head n % 8 at the 4
// positions tw + 16 mt + 4 (l / 16) + i of the lane's accumulator.
//
// Softmax numerators over the wave's 32 positions with the wave's own max
// (:1212-1214), then P . V (:1215-1221) with P as the A operand: row n holds
// head n % 8's weights split the same way (bf16(p) for n < 8, the rest for
// n >= 8), already in the lanes that computed them; the contraction index
// j of lane group g is position 16 (j / 4) + 4 g + j % 4.  V goes through
// LDS (one row per position, 264 bytes, so that the 4 lane groups' reads
// fall in different banks) and is read back per column as the B operand.
// Rows m and m + 8 of the product (lanes l and l ^ 32) are added by one
// transposing step.  The 4 waves' partial outputs are merged with the
// split's max, as the split merge does across splits.
template <int QPK>
__global__ void __launch_bounds__(256)
k_attn_part(AttnArgs a) {
    constexpr int HD = 128, P = 128, PW = 32, VR = 132;
    // Each wave's V rows, then (its own region, once its last P.V read is
    // issued: a wave's LDS operations complete in order) its outputs for the
    // merge.  Until every wave has read them (the barrier after the query
    // columns), the start holds the finished query heads (bf16 hi, lo) and
    // the token's own k and v row (the split that holds it).  34 KB per
    // block: the 544 blocks of an 8-token step at 2049 positions are
    // resident at once (with a separate 16 KB output buffer, two blocks fit
    // a CU and the last 32 ran as a second round).
    __shared__ __align__(16) uint16_t vt[4][PW * VR];
    __shared__ float mls[4][QPK][2];                    // each wave's (max, sum)
    constexpr int RSTRIDE = PW * VR / 2;                // floats between the waves' output regions
    static_assert(QPK * HD <= RSTRIDE, "a wave's outputs fit its V region");
    static_assert(QPK * 2 * HD * 2 + 2 * HD * 2 <= sizeof(vt), "prologue fits the V rows' space");
    float* const red0 = (float*)&vt[0][0];
    uint16_t (*qs)[2][HD] = (uint16_t (*)[2][HD])&vt[0][0];
    uint16_t (*kvn)[HD] = (uint16_t (*)[HD])((char*)&vt[0][0] + QPK * 2 * HD * 2);
    const int kh = blockIdx.x, b = blockIdx.y, s = (int)gridDim.z - 1 - (int)blockIdx.z;
    const int pos = a.pos[b];
    const int T = pos + 1;
    const int t0 = s * P;
    if (t0 >= T) return;                 // past this token's positions (block-uniform)
    // this split holds the token's own row and appends it (block-uniform);
    // without a.append the rows were appended by k_kv_append
    const bool own = a.append && pos < t0 + P;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int g = lane >> 4, n = lane & 15;
    const int tw = t0 + PW * w;
    const unsigned long long* kvp = a.kv + ((size_t)b * a.L + a.layer) * 2;
    const gptr<const uint16_t> kc = (gptr<const uint16_t>)kvp[0];
    const gptr<const uint16_t> vc = (gptr<const uint16_t>)kvp[1];
    // requests first, in the order of use: the inputs of the block's
    // query heads and (wave 0 of the split holding the token's row) of its
    // k and v rows, then the K rows, then the V rows (unconditional: row 0
    // past the end; the token's own row, not yet in the cache, is replaced
    // below).  The projections are finished here: every split block
    // finishes its query heads itself; with a.append the split holding the
    // token's row also finishes its k and v, appends them to the cache and
    // uses them in place of the cache row.
    const int qh = tid >> 5, qj = tid & 31;          // query head qh of the block, dimensions 4 qj .. + 3
    const int qrow = (kh * QPK + (qh < QPK ? qh : 0)) * HD + 4 * qj;
    const bool kvw = own && w == 0;                  // wave-uniform
    Fin4 fq;
    fin4_load(fq, a, b, qrow, a.bq, qrow, qk_weight(a, true, kh * QPK + (qh < QPK ? qh : 0)), true, pos, qj);
    KvFin fkv;
    if (kvw) kv_load(fkv, a, b, kh, pos, lane);
    uint4 kr[2][4], vr[8];
#pragma unroll
    for (int mt = 0; mt < 2; mt++) {
        const int t = tw + 16 * mt + n;
        const gptr<const uint16_t> row = kc + ((size_t)(t < T ? t : 0) * a.KH + kh) * HD + 8 * g;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) kr[mt][kk] = load_g16(row + 32 * kk);
    }
    __builtin_amdgcn_sched_barrier(0);      // keep the K requests ahead of the arithmetic
    {
        float v[4];
        fin4_value(v, fq, a, b, qrow, a.qn ? a.qk_norm : 0, true, qj);
        // the V rows once the query's inputs are consumed: the registers
        // they take are the prologue's, so that the kernel stays at 3
        // blocks per CU (the rows arrive while the scores are formed)
#pragma unroll
        for (int jv = 0; jv < 8; jv++) {
            const int t = tw + 4 * jv + g;
            vr[jv] = load_g16(vc + ((size_t)(t < T ? t : 0) * a.KH + kh) * HD + 8 * n);
        }
        if (QPK == 8 || qh < QPK) {                 // whole 32-lane segments
#pragma unroll
            for (int e = 0; e < 4; e++) {
                // split for the matrix cores: hi = bf16(q), lo = bf16(q - hi)
                const uint32_t hi = f32_to_bf16_rne(v[e]);
                qs[qh][0][4 * qj + e] = (uint16_t)hi;
                qs[qh][1][4 * qj + e] = (uint16_t)f32_to_bf16_rne(__fsub_rn(v[e], __uint_as_float(hi << 16)));
            }
        }
        if (kvw) kv_store(fkv, a, b, kh, pos, lane, (gptr<uint16_t>)kc, (gptr<uint16_t>)vc, kvn);
    }
    __syncthreads();
    // the query columns (head n % 8, zero for heads >= QPK; the hi half of
    // the split for n < 8, the lo half above)
    const int hq = n & 7;
    const bool lo_col = n >= 8;
    uint4 qr[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
        qr[kk] = hq < QPK ? *(const uint4*)&qs[hq < QPK ? hq : 0][lo_col ? 1 : 0][8 * g + 32 * kk]
                          : make_uint4(0u, 0u, 0u, 0u);
    if (own) {
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
            if (tw + 16 * mt + n == pos) {
#pragma unroll
                for (int kk = 0; kk < 4; kk++) kr[mt][kk] = *(const uint4*)&kvn[0][8 * g + 32 * kk];
            }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (tw + 4 * j + g == pos) vr[j] = *(const uint4*)&kvn[1][8 * n];
    }
    __syncthreads();                        // vt is free from here
    bf16x8 qb[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) qb[kk] = __builtin_bit_cast(bf16x8, qr[kk]);

    // ---- scores: q . k / sqrtf_fast(hd), as q . k times the divisor's
    // reciprocal (within an ulp of the division)
    floatx4 sacc[2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++) {
        sacc[mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
            sacc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kr[mt][kk]), qb[kk],
                                                               sacc[mt], 0, 0, 0);
    }
    float sv[8];
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float c = sacc[mt][i];
            const float tot = __fadd_rn(c, dpp_f<DPP_ROR8>(c));
            const int t = tw + 16 * mt + 4 * g + i;
            const float sc = t < T ? __fmul_rn(tot, a.rsdiv) : -INFINITY;
            sv[4 * mt + i] = sc;
            mx = fmaxf(mx, sc);
        }
    // over the lane groups (positions) of the column
    mx = fmaxf(mx, swz_xor16_f(mx));
    mx = fmaxf(mx, __shfl_xor(mx, 32, JM_WAVE));
    const float mref = mx == -INFINITY ? 0.0f : mx;     // a wave wholly past T
    float l = 0.0f;
    uint32_t pp[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float p0 = expf_fast(__fsub_rn(sv[2 * i], mref));
        const float p1 = expf_fast(__fsub_rn(sv[2 * i + 1], mref));
        l = __fadd_rn(__fadd_rn(l, p0), p1);
        uint32_t hi, lo;
        split_bf16x2(p0, p1, hi, lo);
        pp[i] = lo_col ? lo : hi;
    }
    l = __fadd_rn(l, swz_xor16_f(l));
    l = __fadd_rn(l, __shfl_xor(l, 32, JM_WAVE));
    const bf16x8 pa = __builtin_bit_cast(bf16x8, make_uint4(pp[0], pp[1], pp[2], pp[3]));

    // ---- V rows through this wave's LDS rows, read back per column
    uint16_t* vw = vt[w];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        uint2* dst = (uint2*)(vw + (4 * j + g) * VR + 8 * n);
        dst[0] = make_uint2(vr[j].x, vr[j].y);
        dst[1] = make_uint2(vr[j].z, vr[j].w);
    }
    // LDS operations of one wave complete in order; this keeps the compiler
    // from moving the reads above the writes
    __asm__ volatile("" : : : "memory");
    floatx4 oacc[8];
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
        uint32_t vb[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // two 16-bit reads straight into the low and high halves
            const int j0 = 2 * i, j1 = 2 * i + 1;
            u16x2 e;
            e.x = vw[(16 * (j0 >> 2) + 4 * g + (j0 & 3)) * VR + 16 * nt + n];
            e.y = vw[(16 * (j1 >> 2) + 4 * g + (j1 & 3)) * VR + 16 * nt + n];
            vb[i] = __builtin_bit_cast(uint32_t, e);
        }
        oacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            pa, __builtin_bit_cast(bf16x8, make_uint4(vb[0], vb[1], vb[2], vb[3])),
            floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    }
    // rows m (hi) and m + 8 (lo) of a head: lanes l and l ^ 32
    float o[32];
#pragma unroll
    for (int nt = 0; nt < 8; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) o[4 * nt + i] = oacc[nt][i];
    transpose_level<32, 32>(o);
    // now o[4 nt + i] = head 4 (g % 2) + i, dimension 16 (nt + 4 (g / 2)) + n
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int hh = 4 * (g & 1) + i;
            if (hh < QPK) red0[(size_t)w * RSTRIDE + hh * HD + 16 * (nt + 4 * (g >> 1)) + n] = o[4 * nt + i];
        }
    if (g == 0 && n < QPK) {
        mls[w][n][0] = mx;
        mls[w][n][1] = l;
    }
    __syncthreads();

    merge_waves<QPK>(a, b, kh, s, red0, RSTRIDE, mls);
}

// The split block over float32 caches, in float32 arithmetic throughout
// (the reference's SDPA, :1200-1222, on its own cache type): the same
// block shape, prologue and partial outputs as k_attn_part, on the vector
// units.  Wave w takes positions tw = 128 s + 32 w .. tw + 31.
//   scores  lane l: position tw + l % 32 and dimensions 64 (l / 32) .. + 63
//           of its K row (16 float4 loads), against the finished query
//           heads in LDS; the two halves' sums added across lanes l, l ^ 32
//   P . V   lane l: dimensions 2 l, 2 l + 1 of the 32 V rows (one float2
//           load per row, a whole row per wave load), the softmax
//           numerators read back from LDS
template <int QPK>
__global__ void __launch_bounds__(256)
k_attn_part_f32(AttnArgs a) {
    constexpr int HD = 128, P = 128, PW = 32;
    __shared__ __align__(16) float qf[QPK][HD];          // the finished query heads
    __shared__ __align__(16) float kvf[2][HD];           // the token's own k and v rows
    __shared__ __align__(16) float pw[4][QPK][PW];       // each wave's softmax numerators
    __shared__ __align__(16) float red[4][QPK * HD];     // each wave's outputs
    __shared__ float mls[4][QPK][2];                     // each wave's (max, sum)
    const int kh = blockIdx.x, b = blockIdx.y, s = (int)gridDim.z - 1 - (int)blockIdx.z;
    const int pos = a.pos[b];
    const int T = pos + 1;
    const int t0 = s * P;
    if (t0 >= T) return;                 // past this token's positions (block-uniform)
    const bool own = a.append && pos < t0 + P;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int pl = lane & 31, hf = lane >> 5;
    const int tw = t0 + PW * w;
    const unsigned long long* kvp = a.kv + ((size_t)b * a.L + a.layer) * 2;
    const gptr<float> kc = (gptr<float>)kvp[0];
    const gptr<float> vc = (gptr<float>)kvp[1];
    // requests first, in the order of use (as k_attn_part): the prologue's
    // inputs, the K rows, the V rows (row 0 past the end)
    const int qh = tid >> 5, qj = tid & 31;
    const int qhc = qh < QPK ? qh : 0;
    const int qrow = (kh * QPK + qhc) * HD + 4 * qj;
    const bool kvw = own && w == 0;                  // wave-uniform
    Fin4 fq;
    fin4_load(fq, a, b, qrow, a.bq, qrow, qk_weight(a, true, kh * QPK + qhc), true, pos, qj);
    KvFin fkv;
    if (kvw) kv_load(fkv, a, b, kh, pos, lane);
    f32x4_t kr[16];
    {
        const int t = tw + pl;
        const gptr<float> row = kc + ((size_t)(t < T ? t : 0) * a.KH + kh) * HD + 64 * hf;
#pragma unroll
        for (int i = 0; i < 16; i++) kr[i] = *(gptr<const f32x4_t>)(row + 4 * i);
    }
    f32x2_t vr[PW];
#pragma unroll
    for (int j = 0; j < PW; j++) {
        const int t = tw + j;
        vr[j] = *(gptr<const f32x2_t>)(vc + ((size_t)(t < T ? t : 0) * a.KH + kh) * HD + 2 * lane);
    }
    __builtin_amdgcn_sched_barrier(0);      // keep every request ahead of the arithmetic
    {
        float v[4];
        fin4_value(v, fq, a, b, qrow, a.qn ? a.qk_norm : 0, true, qj);
        if (qh < QPK) *(float4*)&qf[qh][4 * qj] = make_float4(v[0], v[1], v[2], v[3]);
        if (kvw) kv_store_f32(fkv, a, b, kh, pos, lane, kc, vc, kvf);
    }
    __syncthreads();
    if (own) {
        // the token's own row, not read from the cache (appended above)
        if (tw + pl == pos) {
#pragma unroll
            for (int i = 0; i < 16; i++) kr[i] = *(const f32x4_t*)&kvf[0][64 * hf + 4 * i];
        }
#pragma unroll
        for (int j = 0; j < PW; j++)
            if (tw + j == pos) vr[j] = *(const f32x2_t*)&kvf[1][2 * lane];
    }

    // ---- scores q . k / sqrtf_fast(hd) (as q . k times the divisor's
    // reciprocal), softmax numerators with the wave's own max
    const bool live = tw + pl < T;
    float mx[QPK], lsum[QPK];
#pragma unroll
    for (int h = 0; h < QPK; h++) {
        const float4* q4 = (const float4*)&qf[h][64 * hf];
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float4 q = q4[i];
            acc = __builtin_fmaf(kr[i].x, q.x, acc);
            acc = __builtin_fmaf(kr[i].y, q.y, acc);
            acc = __builtin_fmaf(kr[i].z, q.z, acc);
            acc = __builtin_fmaf(kr[i].w, q.w, acc);
        }
        const float tot = __fadd_rn(acc, __shfl_xor(acc, 32, JM_WAVE));
        const float sc = live ? __fmul_rn(tot, a.rsdiv) : -INFINITY;
        mx[h] = seg_max<32>(sc);
        const float mref = mx[h] == -INFINITY ? 0.0f : mx[h];     // a wave wholly past T
        const float p = expf_fast(__fsub_rn(sc, mref));
        lsum[h] = seg_sum<32>(p);
        if (hf == 0) pw[w][h][pl] = p;
    }
    // LDS operations of one wave complete in order; this keeps the compiler
    // from moving the reads above the writes
    __asm__ volatile("" : : : "memory");

    // ---- P . V over the wave's positions, in position order
    float2 o[QPK];
#pragma unroll
    for (int h = 0; h < QPK; h++) o[h] = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int j4 = 0; j4 < PW / 4; j4++) {
#pragma unroll
        for (int h = 0; h < QPK; h++) {
            const float4 p4 = *(const float4*)&pw[w][h][4 * j4];
            const float pp[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
            for (int u = 0; u < 4; u++) {
                o[h].x = __builtin_fmaf(vr[4 * j4 + u].x, pp[u], o[h].x);
                o[h].y = __builtin_fmaf(vr[4 * j4 + u].y, pp[u], o[h].y);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < QPK; h++) *(float2*)&red[w][h * HD + 2 * lane] = o[h];
    if (lane < QPK) {
        float m = mx[0], l = lsum[0];
#pragma unroll
        for (int h = 1; h < QPK; h++)
            if (lane == h) { m = mx[h]; l = lsum[h]; }
        mls[w][lane][0] = m;
        mls[w][lane][1] = l;
    }
    __syncthreads();
    merge_waves<QPK>(a, b, kh, s, &red[0][0], QPK * HD, mls);
}

// ---------------------------------------------------- prefill attention
//
// Attention of a chunk of positions of one prompt (every token of the call
// reads the same caches, whose rows k_kv_append has written): block (KV head,
// 64 query rows = 64 / QPK tokens x QPK heads), 8 waves = 2 row groups of 32
// query rows x 4 position strides: in step i wave (rg, ks) takes the
// 32-position tile 4 i + ks of its rows' prefix with an online softmax, and
// the 4 waves of a row group merge once at the end.  k_attn_part's
// per-position form reads K and V, finishes the query heads and merges 4
// waves for every (position, split); here a K or V row is read once per 64
// query rows and the merge launch drops out.
//
// Scores by v_mfma_f32_32x32x16_bf16, K rows as A (lane l: position l % 32,
// dimensions 16 kk + 8 (l / 32) .. + 7), the query rows as B (hi and lo bf16,
// two products as k_attn_part's columns), so that lane l holds query row
// l % 32 at positions 8 (v / 4) + 4 (l / 32) + v % 4: the softmax needs one
// exchange, with lane l ^ 32.  P . V with V^T as A and the weights as B,
// taken from the registers that computed them (contraction index j of half h
// in step s is position 16 s + 8 (j / 4) + 4 h + j % 4);
// ds_read_b64_tr_b16 reads 4 positions of 16 dimensions of V transposed.
//
// A step's 128 K and V rows (64 KB) go straight to LDS (global_load_lds),
// two steps in two arrays: the rows of step i + 2 are requested when step i
// is done, so a row has a whole step to arrive.  (Two arrays, so that the
// compiler sees that a step's reads do not wait for the other's rows.)  The
// 16-byte chunk c of K row r sits at chunk c ^ (r % 16), of V row r at c ^ 4
// (r % 4): the reads of both fall in different banks.
//
// Bound: in a step the 8 waves run their products (64 MFMAs per SIMD, 2048
// cycles) and their weights (about 1700 cycles of vector work) in phase, 1.9
// us; a 512-token chunk of a 32/4-head model has at most 4 + the rows before
// it / 128 steps, and about 11 us of launch, first rows and merge.  Measured
// (append + attention launches): 512 tokens at 32/4 heads 28 us, per-position
// form 70; the chunks of a 1531-token prompt 115 us per layer, 385 before;
// 301 tokens at 32/8 heads 22 us, 54 before.  Staging each wave's own tile
// with one step's rows in flight took 2.6 us per 32 positions instead of 1.9;
// finishing the query rows here instead of in k_kv_append's launch 3 to 6 us
// more per launch.
constexpr int AT_ROWS = 64;             // query rows per block
constexpr int AT_STEP = 128;            // positions per step

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16a __attribute__((ext_vector_type(16)));

// 4 rows x 16 columns of bf16 in LDS, transposed over 16 lanes: lane i gives
// the address of 4 columns (4 (i % 4) ..) of row i / 4 and receives column
// i of rows 0..3
__device__ __forceinline__ s16x4 lds_tr16(const uint16_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(void*)p);
}

// e^-x weights as powers of two; at most -150 apart they are 0.  A NaN
// score's weight is 0 (fmaxf drops the NaN), as expf_fast(NaN) is.
__device__ __forceinline__ float exp2_w(float x) { return __builtin_amdgcn_exp2f(fmaxf(x, -150.0f)); }

template <int QPK>
__global__ void __launch_bounds__(512, 2)
k_attn_tile(AttnArgs a, float* __restrict__ att) {
    constexpr int HD = 128, TQ = AT_ROWS / QPK, RT = 32 / QPK, TILE = 32 * HD;
    // two steps' rows: 4 tiles of K, then 4 of V; after the loop the outputs
    // being merged
    __shared__ __align__(16) uint16_t kv0[2 * AT_STEP * HD];
    __shared__ __align__(16) uint16_t kv1[2 * AT_STEP * HD];
    __shared__ float mls[8][32][2];
    // per query row: which dimensions met a V value of +Inf (bit 0) or -Inf
    // (bit 1) or NaN (both), 16 dimensions per word
    __shared__ uint32_t taint[AT_ROWS][HD / 16];
    static_assert(4 * 64 * 64 * 4 == sizeof(kv0), "a step's space holds the outputs of 4 waves");
    const int kh = blockIdx.x, b0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * TQ;   // longest prefixes first
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), rg = w & 1, ks = w >> 1;
    const int n = lane & 31, h = lane >> 5;
    const unsigned long long* kvp = a.kv + ((size_t)b0 * a.L + a.layer) * 2;
    const gptr<const uint16_t> src = (gptr<const uint16_t>)kvp[rg];     // what this wave loads: K (rg 0) or V rows

    // row n of the row group is token tb; the positions of the block's 64
    // rows (lane's first and last) bound its steps and its unmasked tiles
    const int tb = b0 + rg * RT + n / QPK;
    const int prow = a.pos[min(tb, a.B - 1)];
    int pmax = a.pos[min(b0 + lane / QPK, a.B - 1)], pmin = pmax;
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        pmax = max(pmax, __shfl_xor(pmax, o, JM_WAVE));
        pmin = min(pmin, __shfl_xor(pmin, o, JM_WAVE));
    }
    pmax = __builtin_amdgcn_readfirstlane(pmax);
    pmin = __builtin_amdgcn_readfirstlane(pmin);
    const int nstep = pmax / AT_STEP + 1;

    // This wave's rows of step i: the K or V rows of tile 4 i + ks, load j
    // rows 4 j .. 4 j + 3 (lane l row 4 j + l / 16, LDS chunk l % 16).  Rows
    // past the prefixes repeat the last one (their weights are 0).
    const uint32_t rstride = (uint32_t)a.KH * HD;
    auto load_step = [&](int i, uint16_t* kv) __attribute__((always_inline)) {
        const int t = min(4 * i + ks, pmax / 32);
        const gptr<const uint16_t> base = src + ((size_t)(32 * t) * a.KH + kh) * HD;
        uint16_t* const dst = kv + (4 * rg + ks) * TILE;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int r = 4 * j + (lane >> 4);
            const int x = rg ? 4 * (lane >> 4) : (r & 15);
            __builtin_amdgcn_global_load_lds(
                (gptr<void>)(base + ((uint32_t)min(r, pmax - 32 * t) * rstride + 8 * ((lane & 15) ^ x))),
                (__attribute__((address_space(3))) void*)(dst + 4 * j * HD), 16, 0, 0);
        }
    };

    // the query rows, finished by k_kv_append
    bf16x8 qh[8], ql[8];
    {
        const uint16_t* q = a.qhl + ((size_t)min(tb, a.B - 1) * a.H + kh * QPK + n % QPK) * 2 * HD + 8 * h;
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            qh[kk] = __builtin_bit_cast(bf16x8, *(const uint4*)(q + 16 * kk));
            ql[kk] = __builtin_bit_cast(bf16x8, *(const uint4*)(q + HD + 16 * kk));
        }
    }
    load_step(0, kv0);
    (&taint[0][0])[tid] = 0;
    static_assert(sizeof(taint) == 512 * 4, "a taint word per thread");
    if (nstep > 1) load_step(1, kv1);

    // scores as powers of two: q . k / sqrtf_fast(hd) times log2(e)
    const float c2 = __fmul_rn(a.rsdiv, 1.4426950408889634f);
    const int kx = h ^ (n & 15);            // K row n: dimensions 16 kk + 8 h .. at chunk (2 kk) ^ kx
    // this lane's part of a transposed read: row 4 h + i / 4, 4 columns
    // 16 (l / 16 % 2) + 4 (i % 4) of a 32-column block, i = l % 16
    const int vrow = (lane & 15) >> 2;      // row % 4
    const int vo = (4 * h + vrow) * HD + 8 * (2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) + 4 * (lane & 1);
    floatx16a O[4] = {};
    float m = -INFINITY, l = 0.0f;

    auto step = [&](int i, uint16_t* kv) __attribute__((always_inline)) {
        // this wave's rows of step i have arrived (8 loads of step i + 1 may
        // be outstanding), then everyone's
        if (i + 1 < nstep) __builtin_amdgcn_s_waitcnt(0x0F78);      // vmcnt(8)
        else __builtin_amdgcn_s_waitcnt(0x0F70);                    // vmcnt(0)
        wave_meet();
        const int t = 4 * i + ks;
        uint16_t* const kw = kv + ks * TILE;
        uint16_t* const vw = kv + (4 + ks) * TILE;
        if (AT_STEP * i + AT_STEP - 1 > pmin) {
            // A weight of 0 does not hide a non-finite V value from the
            // matrix product.  In a step that reaches past some row's prefix
            // such values go into `taint`, for the rows whose prefix holds
            // them, and out of the step.  (Block-uniform.)
            uint32_t nf = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint4 u = *(const uint4*)(vw + 8 * (256 * rg + 64 * j + lane));
                const uint32_t x[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 4; e++)
                    nf |= (uint32_t)((x[e] & 0x7F80u) == 0x7F80u) | (uint32_t)((x[e] & 0x7F800000u) == 0x7F800000u);
            }
            if (__syncthreads_or(nf != 0)) {
#pragma unroll 1
                for (int e = lane; e < TILE; e += 64) {
                    const int r = e / HD, dim = (e % HD) ^ (32 * (r & 3));
                    const uint32_t x = vw[e];
                    if ((x & 0x7F80u) != 0x7F80u) continue;
                    const uint32_t bits = (x & 0x7Fu) ? 3u : (x >> 15) ? 2u : 1u;
#pragma unroll 1
                    for (int q = 0; q < 32; q++)
                        if (32 * t + r <= a.pos[min(b0 + rg * RT + q / QPK, a.B - 1)])
                            atomicOr(&taint[32 * rg + q][dim / 16], bits << (2 * (dim % 16)));
                }
                __syncthreads();
                if (rg == 0) {
#pragma unroll 1
                    for (int e = lane; e < TILE; e += 64)
                        if ((vw[e] & 0x7F80u) == 0x7F80u) vw[e] = 0;
                }
                __syncthreads();
            }
        }
        if (32 * t <= pmax) {
            floatx16a S = {};
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const bf16x8 k8 = __builtin_bit_cast(bf16x8, *(const uint4*)(kw + n * HD + 8 * ((2 * kk) ^ kx)));
                S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k8, ql[kk], S, 0, 0, 0);
                S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k8, qh[kk], S, 0, 0, 0);
            }
            if (32 * t + 31 > pmin) {
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (32 * t + 8 * (v / 4) + 4 * h + v % 4 > prow) S[v] = -INFINITY;
            }
            float mt = S[0];
#pragma unroll
            for (int v = 1; v < 16; v++) mt = fmaxf(mt, S[v]);
            mt = fmaxf(mt, __shfl_xor(mt, 32, JM_WAVE));
            const float mn = fmaxf(m, __fmul_rn(mt, c2));
            const float mref = mn == -INFINITY ? 0.0f : mn;         // a row with no score yet
            if (__any(mn != m)) {
                const float f = exp2_w(__fsub_rn(m, mref));
                l = __fmul_rn(l, f);
#pragma unroll
                for (int nt = 0; nt < 4; nt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) O[nt][v] = __fmul_rn(O[nt][v], f);
                m = mn;
            }
            float p[16];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                p[v] = exp2_w(__builtin_fmaf(S[v], c2, -mref));
                l = __fadd_rn(l, p[v]);
            }
#pragma unroll
            for (int s = 0; s < 2; s++) {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int e = 0; e < 4; e++) split_bf16x2(p[8 * s + 2 * e], p[8 * s + 2 * e + 1], hi[e], lo[e]);
                const bf16x8 ph = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
                const bf16x8 pl = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
#pragma unroll
                for (int nt = 0; nt < 4; nt++) {
                    const s16x4 v0 = lds_tr16(vw + vo + 16 * s * HD + 32 * (nt ^ vrow));
                    const s16x4 v1 = lds_tr16(vw + vo + (16 * s + 8) * HD + 32 * (nt ^ vrow));
                    const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
                    O[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pl, O[nt], 0, 0, 0);
                    O[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, ph, O[nt], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): this wave's reads of the step, then
        wave_meet();                        // everyone's, are done
        if (i + 2 < nstep) load_step(i + 2, kv);
    };
#pragma unroll 1
    for (int i = 0; i < nstep; i += 2) {
        step(i, kv0);
        if (i + 1 < nstep) step(i + 1, kv1);
    }

    // ---- the 4 waves of each row group merged with the rows' max
    l = __fadd_rn(l, __shfl_xor(l, 32, JM_WAVE));
    if (h == 0) {
        mls[w][n][0] = m;
        mls[w][n][1] = l;
    }
    __syncthreads();
    float M = -INFINITY, L = 0.0f;
#pragma unroll
    for (int u = 0; u < 4; u++) M = fmaxf(M, mls[2 * u + rg][n][0]);
    if (M == -INFINITY) M = 0.0f;
#pragma unroll
    for (int u = 0; u < 4; u++) L = __builtin_fmaf(mls[2 * u + rg][n][1], exp2_w(__fsub_rn(mls[2 * u + rg][n][0], M)), L);
    // every wave's outputs to LDS (row group, then 32-dimension block, then
    // wave), the rows' 32-dimension block ks summed by wave ks, over the
    // waves in order
    const float f = exp2_w(__fsub_rn(m, M));
    float4* const mb = (float4*)(rg ? &kv1[0] : &kv0[0]) + lane;        // [nt][wave][4][64 lanes]
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            mb[((nt * 4 + ks) * 4 + q) * 64] =
                make_float4(__fmul_rn(O[nt][4 * q], f), __fmul_rn(O[nt][4 * q + 1], f), __fmul_rn(O[nt][4 * q + 2], f),
                            __fmul_rn(O[nt][4 * q + 3], f));
    __syncthreads();
    const float r = __fdiv_rn(1.0f, L);
    if (tb < a.B) {
        float* out = att + ((size_t)tb * a.H + kh * QPK + n % QPK) * HD + 32 * ks + 4 * h;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float4 s = mb[((ks * 4 + 0) * 4 + q) * 64];
#pragma unroll
            for (int u = 1; u < 4; u++) {
                const float4 x = mb[((ks * 4 + u) * 4 + q) * 64];
                s = make_float4(__fadd_rn(s.x, x.x), __fadd_rn(s.y, x.y), __fadd_rn(s.z, x.z), __fadd_rn(s.w, x.w));
            }
            const uint32_t tw = taint[32 * rg + n][2 * ks + q / 2] >> (16 * (q % 2) + 8 * h);   // dimensions 8 q + 4 h ..
            float o[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t x = (tw >> (2 * e)) & 3u;
                const float add = x == 0 ? 0.0f : x == 1 ? INFINITY : x == 2 ? -INFINITY : __int_as_float(0x7FC00000);
                o[e] = __fmul_rn(__fadd_rn(o[e], add), r);
            }
            *(float4*)(out + 8 * q) = make_float4(o[0], o[1], o[2], o[3]);
        }
    }
}

// Merge of the splits of one (query head, token): out = sum_s o_s e^(m_s - M)
// / sum_s l_s e^(m_s - M), M the max over the splits.  The splits' weights
// are computed in parallel (128 at a time) and staged in LDS; each thread
// then sums its dimension over them with independent loads.  Up to
// CMB_SR splits (4096 positions), every load is issued first (thread t:
// split t's max and sum, and its dimension of every split), so the merge
// waits for one memory round trip; the sums are the same, in the same order.
constexpr int CMB_SR = 32;

__global__ void __launch_bounds__(128)
k_attn_comb(AttnArgs a, int qpk, float* __restrict__ att) {
    __shared__ float fs[128];
    __shared__ float red[2];
    const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    const int kh = h / qpk, hq = h % qpk;
    const int ns = (a.pos[b] + 128) / 128;          // splits of T = pos + 1 positions
    const size_t base = ((size_t)b * a.KH + kh) * a.S;
    const float* ml = a.part_ml + (base * qpk + hq) * 2;      // split s at ml[2 qpk s]
    if (ns <= CMB_SR) {
        const float* po = a.part_o + (base * qpk + hq) * 128 + t;
        float pv[CMB_SR];
#pragma unroll
        for (int s = 0; s < CMB_SR; s++) pv[s] = s < ns ? po[(size_t)128 * qpk * s] : 0.0f;
        const float m_t = t < ns ? ml[(size_t)2 * qpk * t] : -INFINITY;
        const float l_t = t < ns ? ml[(size_t)2 * qpk * t + 1] : 0.0f;
        const float mx = seg_max<64>(fmaxf(-INFINITY, m_t));
        if ((t & 63) == 0) red[t >> 6] = mx;
        __syncthreads();
        const float M = fmaxf(red[0], red[1]);
        float f = 0.0f, lsum = 0.0f;
        if (t < ns) {
            f = expf_fast(__fsub_rn(m_t, M));
            lsum = __builtin_fmaf(l_t, f, lsum);
        }
        fs[t] = f;
        __syncthreads();
        float O = 0.0f;
#pragma unroll
        for (int s = 0; s < CMB_SR; s++)
            if (s < ns) O = __builtin_fmaf(pv[s], fs[s], O);
        lsum = seg_sum<64>(lsum);
        if ((t & 63) == 0) red[t >> 6] = lsum;      // every thread read M before the barrier above
        __syncthreads();
        att[((size_t)b * a.H + h) * 128 + t] = __fdiv_rn(O, __fadd_rn(red[0], red[1]));
        return;
    }
    float mx = -INFINITY;
    for (int s = t; s < ns; s += 128) mx = fmaxf(mx, ml[(size_t)2 * qpk * s]);
    mx = seg_max<64>(mx);
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    const float M = fmaxf(red[0], red[1]);
    float lsum = 0.0f, O = 0.0f;
    const float* po = a.part_o + (base * qpk + hq) * 128 + t;  // split s at po[128 qpk s]
    for (int c0 = 0; c0 < ns; c0 += 128) {
        const int s = c0 + t;
        float f = 0.0f;
        if (s < ns) {
            f = expf_fast(__fsub_rn(ml[(size_t)2 * qpk * s], M));
            lsum = __builtin_fmaf(ml[(size_t)2 * qpk * s + 1], f, lsum);
        }
        __syncthreads();
        fs[t] = f;
        __syncthreads();
        const int n = ns - c0 < 128 ? ns - c0 : 128;
#pragma unroll 8
        for (int i = 0; i < n; i++) O = __builtin_fmaf(po[(size_t)128 * qpk * (c0 + i)], fs[i], O);
    }
    lsum = seg_sum<64>(lsum);
    __syncthreads();
    if ((t & 63) == 0) red[t >> 6] = lsum;
    __syncthreads();
    att[((size_t)b * a.H + h) * 128 + t] = __fdiv_rn(O, __fadd_rn(red[0], red[1]));
}

hipError_t launch_attn(const AttnArgs& a, int qpk, float* att, hipStream_t st) {
    if (a.B == 0) return hipSuccess;
    if (a.qk_norm == 2) {
        if (!a.qkss || !a.qn || !a.kn) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_qk_ss, dim3((unsigned)a.B), dim3(256), 0, st, a);
        hipError_t e0 = hipGetLastError();
        if (e0 != hipSuccess) return e0;
    }
    const bool tile = !a.append && a.shared && !a.kv_f32 && attn_tile_takes(a.B, a.KH, qpk);
    if (qpk != 1 && qpk != 2 && qpk != 4 && qpk != 8) return hipErrorInvalidValue;
    if (!a.append) {
        // (the partial outputs' buffer, unused by k_attn_tile, holds the query heads for it)
        AttnArgs ap = a;
        ap.qhl = tile ? (uint16_t*)a.part_o : nullptr;
        const dim3 ga((unsigned)a.KH, (unsigned)a.B), gb(tile ? 64 * (1 + (qpk + 1) / 2) : 64);
        if (a.kv_f32) hipLaunchKernelGGL(k_kv_append<true>, ga, gb, 0, st, ap);
        else hipLaunchKernelGGL(k_kv_append<false>, ga, gb, 0, st, ap);
        hipError_t e0 = hipGetLastError();
        if (e0 != hipSuccess) return e0;
    }
    if (tile) {
        AttnArgs ap = a;
        ap.qhl = (uint16_t*)a.part_o;
        const int tq = AT_ROWS / qpk;
        const dim3 gt((unsigned)a.KH, (unsigned)((a.B + tq - 1) / tq));
        switch (qpk) {
            case 1: hipLaunchKernelGGL(k_attn_tile<1>, gt, dim3(512), 0, st, ap, att); break;
            case 2: hipLaunchKernelGGL(k_attn_tile<2>, gt, dim3(512), 0, st, ap, att); break;
            case 4: hipLaunchKernelGGL(k_attn_tile<4>, gt, dim3(512), 0, st, ap, att); break;
            default: hipLaunchKernelGGL(k_attn_tile<8>, gt, dim3(512), 0, st, ap, att); break;
        }
        return hipGetLastError();
    }
    // Split s of (KV head kh, token b) is block (kh, b, S - 1 - s): the
    // splits are dispatched from the last one, which holds the fewest
    // positions (or none, for a token whose prefix is short).  A block that
    // lands on a CU after others has its first requests served behind
    // theirs; dispatched this way, the blocks that land late are mostly full
    // splits behind light ones rather than full splits behind full ones.
    const dim3 grid((unsigned)a.KH, (unsigned)a.B, (unsigned)a.S);
#define JM_AP(Q) if (a.kv_f32) hipLaunchKernelGGL(k_attn_part_f32<Q>, grid, dim3(256), 0, st, a); \
                 else hipLaunchKernelGGL(k_attn_part<Q>, grid, dim3(256), 0, st, a)
    switch (qpk) {
        case 1: JM_AP(1); break;
        case 2: JM_AP(2); break;
        case 4: JM_AP(4); break;
        case 8: JM_AP(8); break;
        default: return hipErrorInvalidValue;
    }
#undef JM_AP
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_attn_comb, dim3((unsigned)a.H, (unsigned)a.B), dim3(128), 0, st, a, qpk, att);
    return hipGetLastError();
}

// ------------------------------------------------------------ final norm

// out[b] = RMSNorm(x[b]) * w (decode_kernel.c:224-230), one block per token.
__global__ void __launch_bounds__(256)
k_rms_rows(const float* __restrict__ x, const uint16_t* __restrict__ w, int d, float eps,
           float* __restrict__ out) {
    __shared__ float part[4];
    const int b = blockIdx.x, tid = threadIdx.x;
    const float* xr = x + (size_t)b * d;
    float ss = 0.0f;
    for (int i = tid; i < d; i += 256) ss = __builtin_fmaf(xr[i], xr[i], ss);
    ss = seg_sum<64>(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    const float inv = rms_inv(__fadd_rn(__fadd_rn(part[0], part[1]), __fadd_rn(part[2], part[3])), d, eps);
    for (int i = tid; i < d; i += 256)
        out[(size_t)b * d + i] = __fmul_rn(__fmul_rn(xr[i], inv), bf16_bits_to_f32(w[i]));
}

hipError_t launch_rms_rows(const float* x, const uint16_t* w, int B, int d, float eps, float* out,
                           hipStream_t st) {
    if (B == 0) return hipSuccess;
    hipLaunchKernelGGL(k_rms_rows, dim3((unsigned)B), dim3(256), 0, st, x, w, d, eps, out);
    return hipGetLastError();
}

}  // namespace jm
