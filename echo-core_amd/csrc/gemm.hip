// gemm.hip — prefill GEMM over block-quantized weights on int8 MFMA (gfx950).
//
// Y[m][n] (+)= sum over K of X[m][k] * W[n][k] for M tokens (prefill chunks,
// e.g. 512), with X quantized per 32-element block by the reference quantizer
// (src/kernels/quant.cpp:18-98) and W in the tiled decode layout (quant.hip).
// Every 32-block product is one exact int32 (v_mfma_i32_32x32x32_i8: A = 32
// tokens x 32 int8, B = 32 int8 x 32 weight rows); the block scales are applied
// in fp32:
//   Q8_0: Y += d_x[m,b] * d_w[n,b] * isum_b
//   Q4_K: Y += d_x[m,s] * (d*sc_s * isum_s - dmin*m_s * xsum_s)   (per sub-block s)
// which is the reference's matvec arithmetic (matvec.cpp:62-142) on the
// quantized activations, in a different summation order.
//
// Activation layout ("XT", gemm_act.hpp), tokens in tiles of 16:
//   Q8_0: chunk (token tile T, group G of 4 blocks) = 2048 B at (T*nG+G)*2048,
//         lane l's 16 B at 16l (blocks 0,1) and 1024+16l (blocks 2,3), 8 B per
//         block = x[16T + l%16][128G + 32j + 8(l/16) .. +8];
//   Q4_K: chunk (T, super-block b) = 4096 B, lane l's 8 B per sub-block s at
//         (s/2)*1024 + 16l + 8(s%2): the sub-block's elements 4g..4g+3 and
//         16+4g..16+4g+3 (g = l/16) in the reference's Q4_K position order
//         (so they meet the weight nibbles of the same positions);
//   xd  fp32 [Mp][Kp/32] block scales; Q4_K adds dxs = xd * sum(block int8).
//
// What bounds it: the scales.  Every (token, row, block) needs its own
// d_x * d_w, 32 of them per 1024 MACs on the VALU; the matrix core alone would
// need a sixth of the time.  So: few VALU operations per element, none of them
// a half-rate conversion, and enough waves per SIMD to issue them (one wave
// issues a VALU operation every 5 clocks, two or three waves one every 2.5;
// two that depend on each other are 8 clocks apart, so a tile's operations
// are formed in three passes over its 16 elements).
//   The MFMA's C operand is the bit pattern of 1.5 * 2^23: its result read as
//   a float is f = 1.5 * 2^23 + isum exactly (|isum| <= 32 * 128 * 128 < 2^22).
//   Q8_0: Y = fma(f - 1.5 * 2^23, d_x * d_w, Y), block after block over all of
//   K: one running sum per output, the same bits whatever the tile.  (After 32
//   layers of int8 activations another order of these additions moves the
//   logits by percents, so this order is part of the result.)
//   Q4_K: u = fma(f, d_s, -1.5 * 2^23 * d_s) = round(isum * d_s), Y = fma(u,
//   d_x, Y): the product 1.5 * 2^23 * d_s is exact (d_s = d * sc has 17
//   significant bits), one rounding per block product as before and one
//   operation less.  (An infinite d gives NaN.)  Here K is cut in four
//   quarters, one per wave of a workgroup, whose sums meet in LDS and are added
//   in pairs; the cut does not depend on M, so a token's row is again the same
//   bits in every pass.
// A wave works alone: operands straight from global memory (16-byte loads half
// a chunk ahead), v_mfma_i32_32x32x32_i8 per 32-block (a quarter of the issues
// and half the time of four 16x16x32), its tokens' scales through its own
// slice of LDS, no barrier in the K loop.  Small products (launch_q8) take
// k_gemm_q8_16, tiles of 16 tokens with several chunks in flight.
//
// M x N x K, us, this kernel / the one before it (64 x 64 workgroup tiles,
// 16x16x32 MFMA, conversion + product + FMA per element, scales through a
// workgroup-wide LDS stage with a barrier per chunk; same bits for Q8_0):
//   Q8_0 1024x18432x2560 160 / 203, 1024x2560x9216 91 / 121, 512x12352x2560
//        69 / 78, 512x2560x9216 59 / 75, 200x2560x9216 44 / 57,
//        130x12352x2560 24 / 37, 40x18432x2560 20 / 23, 40x2560x9216 19 / 56
//   Q4_K 1024x18432x2560 175 / 270, 387x18432x2560 76 / 121, 387x2560x9216
//        50 / 88, 40x2560x9216 17 / 56
// Also tried at Q8_0 1024x18432x2560: both operands staged in LDS by the
// workgroup (162; 147 with 32x32x32 products and Q4_K's two operations), the
// token scales spread over the lanes by v_mfma_f32_16x16x4_f32 instead of LDS
// reads (157 with two operations), 64 x 64 tiles per wave (171), two tiles'
// products in flight at two waves per SIMD (171), a barrier per chunk to keep
// four waves on the same lines of L1 (no change), operands three halves of a
// chunk ahead instead of one (no change here nor at 130 tokens).
#include <type_traits>

#include "gemm_act.hpp"

namespace ec {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ----------------------------------------------------------- activation prep
// Q4_K with 16-byte loads: a wave takes one super-block (256 elements) of its
// token per step, lane l elements 4l .. 4l+3.  Sub-block s = 2h + j holds the
// runs 64h + 16j + (0..15) and 64h + 32 + 16j + (0..15) (the reference's
// position order), i.e. lanes 16h + 4j + (0..3) and those 8 above: the
// sub-block's amax and int8 sum take xor 1, 2, 8 over its 8 lanes, and the
// run-0 lane stores its 4 bytes with the run-1 lane's 4 (bytes 4g .. 4g+3 and
// 16+4g .. 16+4g+3 of operand lane token%16 + 16g).  The reference
// quantizer per sub-block (scale = amax/127, bytes rne(x * (1/scale)), dxs =
// scale * the sub-block's int8 sum).  grid (ceil(nch / 2), Mp / 4).
__global__ __launch_bounds__(256) void k_gemm_quantize_x4v(const float* __restrict__ x, uint8_t* __restrict__ xt,
                                                           uint32_t M, uint32_t K, uint32_t ldx, uint32_t nch,
                                                           uint32_t nbp, size_t xd_off, size_t dxs_off) {
    const uint32_t lane = threadIdx.x & 63, m = blockIdx.y * 4 + (threadIdx.x >> 6);
    const uint32_t b0 = blockIdx.x * 2, h = lane / 16, j = (lane & 7) / 4, g = lane & 3;
    const uint32_t s = 2 * h + j;
    float4 v[2];
#pragma unroll
    for (uint32_t st = 0; st < 2; ++st) {
        const uint32_t k = 256 * (b0 + st) + 4 * lane;  // K % 256 == 0
        v[st] = (m < M && k < K) ? *(const float4*)(x + (size_t)m * ldx + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (uint32_t st = 0; st < 2; ++st) {
        const uint32_t b = b0 + st;
        if (b >= nch) break;  // uniform over the wave
        float amax = fmaxf(fmaxf(fabsf(v[st].x), fabsf(v[st].y)), fmaxf(fabsf(v[st].z), fabsf(v[st].w)));
        amax = fmaxf(amax, lane_xor<1>(amax));
        amax = fmaxf(amax, lane_xor<2>(amax));
        amax = fmaxf(amax, lane_xor<8>(amax));
        const float scale = q_scale(amax);
        const float inv = __fdiv_rn(1.0f, scale);
        const int8_t q0 = q_body(v[st].x, inv), q1 = q_body(v[st].y, inv), q2 = q_body(v[st].z, inv),
                     q3 = q_body(v[st].w, inv);
        const uint32_t w4 = (uint32_t)(uint8_t)q0 | ((uint32_t)(uint8_t)q1 << 8) | ((uint32_t)(uint8_t)q2 << 16) |
                            ((uint32_t)(uint8_t)q3 << 24);
        const uint32_t hi = row_down<8>(w4);
        int sum = (int)q0 + (int)q1 + (int)q2 + (int)q3;
        sum += lane_xor_i<1>(sum);
        sum += lane_xor_i<2>(sum);
        sum += lane_xor_i<8>(sum);
        if ((lane & 8) == 0) {  // run-0 lanes
            const uint32_t l = m % 16 + 16 * g;
            *(uint2*)(xt + ((size_t)(m / 16) * nch + b) * 4096 + h * 1024 + 16 * l + 8 * j) = make_uint2(w4, hi);
            if (g == 0) {
                ((float*)(xt + xd_off))[(size_t)m * nbp + 8 * b + s] = m < M ? scale : 0.0f;
                ((float*)(xt + dxs_off))[(size_t)m * nbp + 8 * b + s] = scale * (float)sum;
            }
        }
    }
}

// Q8_0: each lane quantizes 4 consecutive elements (one 16-byte load), 8
// consecutive lanes a 32-element block; a wave covers 8 blocks (1 KB of its
// token's row) per step and kQxSteps steps, the workgroup's four waves four
// tokens.  grid (ceil(nbp / (8 kQxSteps)), Mp / 4).
constexpr uint32_t kQxSteps = 2;
__global__ __launch_bounds__(256) void k_gemm_quantize_x8(const float* __restrict__ x, uint8_t* __restrict__ xt,
                                                          uint32_t M, uint32_t K, uint32_t ldx, uint32_t nch,
                                                          uint32_t nbp, size_t xd_off) {
    const uint32_t lane = threadIdx.x & 63, m = blockIdx.y * 4 + (threadIdx.x >> 6);
    const uint32_t q0 = blockIdx.x * 64 * kQxSteps;  // first float4 of the wave
    float4 v[kQxSteps];
#pragma unroll
    for (uint32_t st = 0; st < kQxSteps; ++st) {
        const uint32_t k = 4 * (q0 + 64 * st + lane);  // K % 32 == 0: a block is all real or all padding
        v[st] = (m < M && k < K) ? *(const float4*)(x + (size_t)m * ldx + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (uint32_t st = 0; st < kQxSteps; ++st) {
        const uint32_t q = q0 + 64 * st + lane;
        if (q / 8 < nbp) xt_q8_store4(v[st], m, q, m < M, xt, nch, nbp, xd_off);  // whole 8-lane groups
    }
}

// ------------------------------------------------------------------ product
constexpr int kMagicI = 0x4B400000;        // the float 1.5 * 2^23
constexpr float kMagicF = 12582912.0f;

// The eight 6-bit (scale, min) pairs of a super-block from its 12 scale
// bytes (q[0] = bytes 0-3, ...), four per dword: sc[0] holds sub-blocks 0-3
// (byte s = scale of sub-block s), sc[1] sub-blocks 4-7, mn likewise -- the
// unpack of src/kernels/quant.cpp:222-242 on four bytes per operation.
__device__ __forceinline__ void q4k_sm4(const uint32_t (&q)[3], uint32_t (&sc)[2], uint32_t (&mn)[2]) {
    sc[0] = q[0] & 0x3F3F3F3Fu;
    mn[0] = q[1] & 0x3F3F3F3Fu;
    sc[1] = (q[2] & 0x0F0F0F0Fu) | ((q[0] >> 2) & 0x30303030u);
    mn[1] = ((q[2] >> 4) & 0x0F0F0F0Fu) | ((q[1] >> 2) & 0x30303030u);
}

// Byte n of v as a float (v_cvt_f32_ubyte<n>).
__device__ __forceinline__ float ubyte_f(uint32_t v, int n) { return (float)((v >> (8 * n)) & 0xFFu); }

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// A token's Q4_K min term
//   Y[t][n] -= sum_s (dmin*m)[n][s] * dxs[t][s]
// is a dense fp32 product with contraction over the sub-blocks: two
// v_mfma_f32_32x32x2_f32 per tile product and chunk (A = -dxs[token][2q + h],
// B = (dmin*m)[2q + h][row]; lane l holds row l % 32 and k = h = l / 32, its D
// layout the int8 MFMA's) into the same accumulators once per chunk, so the
// running sums stay at the result's magnitude (the min and scale terms, each
// larger than the result, cancel every 4 sub-blocks as in the reference's
// per-sub-block form).  The chunk is 4 blocks (Q8_0) or half a super-block.
//
// A 32-row operand is two 16-row tiles of the stored layouts: lane l takes row
// l % 32 and the 8-byte groups h and h + 2 of a block, the same ones in A and
// B, so the order of k inside a block does not matter.  D: lane l holds weight
// row l % 32 and the tokens 8 (e / 4) + 4 h + e % 4, e = 0 .. 15.  A wave
// copies its tokens' scales of the next chunk to LDS, token-minor, and reads
// them back as float4s that all lanes of a half share; only its own lanes
// read them, and a wave's LDS accesses stay in order.
//
// A workgroup is one tile: KW = 1, one wave with all of K (2 x 2 waves of
// neighbouring tiles ran 1024x2560x9216 in 104 us instead of 91 and
// 130x18432x2560 in 41 instead of 35: waves that end early leave their place
// to the next at once); KW = 4, four waves with a quarter of K each.  ONEC:
// one result tile in flight (a second one's 16 registers would cost a wave
// per SIMD, or spill).
template <int FMT, int TT, int RT, int KW, int MINW, bool ONEC>
__global__ __launch_bounds__(64 * KW, MINW) void k_gemm(const uint8_t* __restrict__ W, const uint8_t* __restrict__ xt,
                                                    float* __restrict__ y, uint32_t M, uint32_t N, uint32_t n_tt,
                                                    uint32_t n_rt, uint32_t nG, uint32_t nbp, size_t xd_off,
                                                    size_t dxs_off, uint32_t ldy, int accumulate, uint32_t gx,
                                                    uint32_t gy) {
    constexpr bool Q4 = FMT == EC_Q4_K;
    constexpr int NX = Q4 ? 8 : 4, E = TT * RT * 16;  // scale rows per token in LDS; sums per lane
    constexpr size_t kScale = KW * 2 * NX * 32 * TT * sizeof(float), kSums = KW == 1 ? 0 : KW * E * 64 * sizeof(float);
    __shared__ __align__(16) uint8_t lds[kScale > kSums ? kScale : kSums];
    // consecutive workgroups run on consecutive XCDs: an XCD takes every eighth
    // row block and all of its token blocks, so its L2 reads those weights once
    const uint32_t id = blockIdx.x, kk = id >> 3, bx = (kk / gy) * 8 + (id & 7), by = kk % gy;
    if (bx >= gx) return;
    const uint32_t lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const uint32_t T0 = 2 * TT * by, R0 = 2 * RT * bx;        // first 16-token and 16-row tile
    const uint32_t G0 = w * nG / KW, G1 = (w + 1) * nG / KW;  // this wave's chunks of 4 blocks
    float(*sc_s)[NX][32 * TT] = (float(*)[NX][32 * TT])(lds + w * (kScale / KW));  // this wave's [buffer][row][token]

    // operand lane l: row l % 32 of the 32-row tile, K groups h and h + 2 (8 elements each) of every block.
    // Wave-uniform bases and 32-bit lane offsets within the tile.
    const uint32_t l16 = 16 * ((lane & 15) + 16 * h), odd = (lane >> 4) & 1;
    const uint32_t arow = nG * 2048, brow = Q4 ? nG / 2 * kQ4TChunk : nG * kQ8TChunk;
    const uint8_t* ua = xt + (size_t)T0 * arow;
    const uint8_t* ub = W + (size_t)R0 * brow;
    uint32_t va[TT], vb[RT];
#pragma unroll
    for (int t = 0; t < TT; ++t) va[t] = (min(T0 + 2 * t + odd, n_tt - 1) - T0) * arow + l16;
#pragma unroll
    for (int r = 0; r < RT; ++r) vb[r] = (min(R0 + 2 * r + odd, n_rt - 1) - R0) * brow;
    const uint32_t tk = lane % (32 * TT), vx = (min(16 * T0 + tk, 16 * n_tt - 1) - 16 * T0) * nbp * 4;
    const uint8_t* ux = xt + xd_off + (size_t)T0 * 16 * nbp * 4;
    const uint8_t* um = xt + dxs_off + (size_t)T0 * 16 * nbp * 4;

    u32x4 a[2][TT][2], b[2][RT][2];  // Q8_0: [half of the chunk], Q4_K weights: [chunk parity]
    std::conditional_t<Q4, u32x4, uint2> hd[2][RT];  // Q4_K headers, Q8_0 the row's four block scales
    float4 rx, rm;
    auto load_a = [&](auto pc, uint32_t G) {
        constexpr int p = decltype(pc)::value;
        const uint8_t* s0 = ua + (size_t)G * 2048 + p * 1024;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s) a[p][t][s] = *(const u32x4*)(s0 + va[t] + 512 * s);
        if constexpr (!Q4) {
            const uint8_t* s1 = ub + (size_t)G * kQ8TChunk + p * 1024;
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int s = 0; s < 2; ++s) b[p][r][s] = *(const u32x4*)(s1 + (vb[r] + l16) + 512 * s);
        }
    };
    auto load_w = [&](int buf, uint32_t G) {
        const uint8_t* s1 = ub + (Q4 ? (size_t)(G >> 1) * kQ4TChunk : (size_t)G * kQ8TChunk);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            if constexpr (Q4) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    b[buf][r][s] = *(const u32x4*)(s1 + 1024 * (G & 1) + (vb[r] + l16) + 512 * s);
                hd[buf][r] = *(const u32x4*)(s1 + (vb[r] + 16 * (lane & 15)) + 2048);
            } else {
                hd[buf][r] = *(const uint2*)(s1 + (vb[r] + 8 * (lane & 15)) + 2048);
            }
        }
        rx = *(const float4*)(ux + (size_t)G * 16 + vx);
        if constexpr (Q4) rm = *(const float4*)(um + (size_t)G * 16 + vx);
    };
    auto store_x = [&](uint32_t bf) {
        sc_s[bf][0][tk] = rx.x, sc_s[bf][1][tk] = rx.y, sc_s[bf][2][tk] = rx.z, sc_s[bf][3][tk] = rx.w;
        if constexpr (Q4)
            sc_s[bf][4][tk] = -rm.x, sc_s[bf][5][tk] = -rm.y, sc_s[bf][6][tk] = -rm.z, sc_s[bf][7][tk] = -rm.w;
    };

    v16f acc[TT][RT];
    v16i magic, c[2];
#pragma unroll
    for (int e = 0; e < 16; ++e) magic[e] = kMagicI;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][r][e] = 0.0f;
    float dr[RT], dwf[RT], mdw[RT];
    uint32_t scr[RT];
    constexpr int PH = 2 * TT * RT;  // tile products of half a chunk, in order (block, token tile, row tile)
    auto half = [&](auto pc, uint32_t bf, int wb) {
        constexpr int p = decltype(pc)::value;
        v4i A[TT], B[RT];
        float4 dq[4];
        auto mfma = [&](auto ic) {
            constexpr int i = decltype(ic)::value, jj = i / (TT * RT), t = (i / RT) % TT, r = i % RT, j = 2 * p + jj;
            if constexpr (t == 0) {
                if constexpr (Q4) {
                    const u32x4 v0 = b[wb][r][0], v1 = b[wb][r][1];
                    const uint32_t q0 = j == 0 ? v0.x : j == 1 ? v0.y : j == 2 ? v0.z : v0.w;
                    const uint32_t q1 = j == 0 ? v1.x : j == 1 ? v1.y : j == 2 ? v1.z : v1.w;
                    B[r] = v4i{(int)(q0 & 0x0F0F0F0Fu), (int)((q0 >> 4) & 0x0F0F0F0Fu), (int)(q1 & 0x0F0F0F0Fu),
                               (int)((q1 >> 4) & 0x0F0F0F0Fu)};
                } else {
                    const u32x4 v0 = b[p][r][0], v1 = b[p][r][1];
                    B[r] = jj ? v4i{(int)v0.z, (int)v0.w, (int)v1.z, (int)v1.w}
                              : v4i{(int)v0.x, (int)v0.y, (int)v1.x, (int)v1.y};
                }
            }
            if constexpr (r == 0) {
                const u32x4 v0 = a[p][t][0], v1 = a[p][t][1];
                A[t] = jj ? v4i{(int)v0.z, (int)v0.w, (int)v1.z, (int)v1.w}
                          : v4i{(int)v0.x, (int)v0.y, (int)v1.x, (int)v1.y};
            }
            c[ONEC ? 0 : i & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[t], B[r], magic, 0, 0, 0);
        };
        if constexpr (!ONEC) mfma(std::integral_constant<int, 0>{});
        static_for<0, PH>([&](auto ic) {
            constexpr int i = decltype(ic)::value, jj = i / (TT * RT), t = (i / RT) % TT, r = i % RT, j = 2 * p + jj;
            if constexpr (r == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) dq[q] = *(const float4*)&sc_s[bf][j][32 * t + 8 * q + 4 * h];
            }
            if constexpr (ONEC) mfma(ic);
            else if constexpr (i + 1 < PH) mfma(std::integral_constant<int, i + 1>{});
            if constexpr (t == 0) {
                if constexpr (Q4) {
                    dwf[r] = dr[r] * ubyte_f(scr[r], j);
                } else {
                    const uint32_t hw = p ? hd[wb][r].y : hd[wb][r].x;
                    dwf[r] = h2f(jj ? hw >> 16 : hw & 0xFFFF);
                    asm("" : "+v"(dwf[r]));  // keep the product in v_fma_f32 (v_fma_mix_f32 issues at a lower rate)
                }
                mdw[r] = -kMagicF * dwf[r];
            }
            float u[16], sc[16];
            const float* d = (const float*)dq;
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = Q4 ? d[e] : d[e] * dwf[r];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float f = __int_as_float(c[ONEC ? 0 : i & 1][e]);
                u[e] = Q4 ? fmaf(f, dwf[r], mdw[r]) : f - kMagicF;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][r][e] = fmaf(u[e], sc[e], acc[t][r][e]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    auto step = [&](uint32_t G, auto wbc) {
        constexpr int wb = decltype(wbc)::value;
        const uint32_t Gn = min(G + 1, G1 - 1), bf = G & 1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        load_a(P1{}, G);
        load_w(wb ^ 1, Gn);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (Q4) {
            float bmin[RT][2];
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const uint32_t q[3] = {hd[wb][r].y, hd[wb][r].z, hd[wb][r].w};
                uint32_t sc4[2], mn4[2];
                q4k_sm4(q, sc4, mn4);
                scr[r] = (G & 1) ? sc4[1] : sc4[0];
                dr[r] = h2f(hd[wb][r].x & 0xFFFF);
                const uint32_t mn = ((G & 1) ? mn4[1] : mn4[0]) >> (8 * h);
                const float dm = h2f(hd[wb][r].x >> 16);
                bmin[r][0] = dm * (float)(mn & 0xFFu);
                bmin[r][1] = dm * (float)((mn >> 16) & 0xFFu);
            }
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const float am = sc_s[bf][4 + 2 * q + h][32 * t + (lane & 31)];
#pragma unroll
                    for (int r = 0; r < RT; ++r)
                        acc[t][r] = __builtin_amdgcn_mfma_f32_32x32x2f32(am, bmin[r][q], acc[t][r], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        half(P0{}, bf, wb);
        load_a(P0{}, Gn);
        __builtin_amdgcn_sched_barrier(0);
        half(P1{}, bf, wb);
        store_x(bf ^ 1);
    };
    if (G0 < G1) {
        load_a(P0{}, G0);
        load_w(0, G0);
        store_x(G0 & 1);
    }
    for (uint32_t G = G0; G < G1; G += 2) {
        step(G, P0{});
        if (G + 1 < G1) step(G + 1, P1{});
    }

    // a lane's sums, four consecutive tokens each: quad k of tile product (t, r) is rows 8 (k % 4) + 4 h + 0..3
    const uint32_t m0 = 16 * T0 + 4 * h, n0 = 16 * R0 + (lane & 31);
    const bool full = 16 * T0 + 32 * TT <= M && 16 * R0 + 32 * RT <= N;
    auto put = [&](uint32_t t, uint32_t r, uint32_t q0, const float* v, auto cnt) {  // quads q0 .. of one tile product
        constexpr int C = decltype(cnt)::value;
        float* yb = y + (size_t)(m0 + 32 * t + 8 * q0) * ldy + n0 + 32 * r;
        float o[4 * C];
        bool ok[4 * C];
#pragma unroll
        for (int e = 0; e < 4 * C; ++e) {
            const uint32_t mo = 8 * (e / 4) + e % 4;
            ok[e] = full || (m0 + 32 * t + 8 * q0 + mo < M && n0 + 32 * r < N);
            o[e] = accumulate && ok[e] ? yb[(size_t)mo * ldy] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 4 * C; ++e)
            if (ok[e]) yb[(size_t)(8 * (e / 4) + e % 4) * ldy] = accumulate ? o[e] + v[e] : v[e];
    };
    if constexpr (KW == 1) {
        static_for<0, TT * RT>([&](auto ic) {
            constexpr int t = decltype(ic)::value / RT, r = decltype(ic)::value % RT;
            float v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = acc[t][r][e];
            put(t, r, 0, v, std::integral_constant<int, 4>{});
        });
    } else {
        // the four waves' sums meet in LDS; wave w adds and stores its quarter
        // of every lane's quads
        float4* sum = (float4*)lds;  // [wave][quad][lane]
        __syncthreads();
        static_for<0, TT * RT * 4>([&](auto ic) {
            constexpr int k = decltype(ic)::value;
            const v16f& s = acc[k / 4 / RT][k / 4 % RT];
            constexpr int e = 4 * (k % 4);
            sum[(w * (E / 4) + k) * 64 + lane] = make_float4(s[e], s[e + 1], s[e + 2], s[e + 3]);
        });
        __syncthreads();
        constexpr int Q = E / 16;  // quads per wave: 1, 2 or 4
        float v[4 * Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const float4* s = sum + (w * Q + k) * 64 + lane;
            const float4 s0 = s[0], s1 = s[E / 4 * 64], s2 = s[E / 2 * 64], s3 = s[3 * E / 4 * 64];
            v[4 * k] = (s0.x + s1.x) + (s2.x + s3.x), v[4 * k + 1] = (s0.y + s1.y) + (s2.y + s3.y);
            v[4 * k + 2] = (s0.z + s1.z) + (s2.z + s3.z), v[4 * k + 3] = (s0.w + s1.w) + (s2.w + s3.w);
        }
        const uint32_t k0 = w * Q, tr = k0 / 4;
        put(tr / RT, tr % RT, k0 % 4, v, std::integral_constant<int, Q>{});
    }
}

// Small Q8_0 products: one wave per workgroup takes 16 tokens x 16 RT rows
// (v_mfma_i32_16x16x32_i8, the stored layouts' own operands: lane l's 8 bytes
// of a block are row l % 16, group l / 16; D: lane l holds weight row l % 16
// and tokens 4 (l / 16) .. +3).  With less than a wave per SIMD nothing hides
// a load but the wave's own later loads, so D chunks stay in flight (registers
// for D = 6 at RT = 1: 232).  The same sums in the same order as k_gemm.
// 40x2560x9216: 19 us, 56 with 32 x 32 tiles; 3 / 4 / 6 chunks ahead 25 / 21 / 19.
template <int RT, int D>
__global__ __launch_bounds__(64, 2) void k_gemm_q8_16(const uint8_t* __restrict__ W, const uint8_t* __restrict__ xt,
                                                       float* __restrict__ y, uint32_t M, uint32_t N, uint32_t n_rt,
                                                       uint32_t nG, uint32_t nbp, size_t xd_off, uint32_t ldy,
                                                       int accumulate, uint32_t gx, uint32_t gy) {
    const uint32_t id = blockIdx.x, kk = id >> 3, bx = (kk / gy) * 8 + (id & 7), T = kk % gy;
    const uint32_t lane = threadIdx.x, g = lane >> 4, R0 = bx * RT;
    if (bx >= gx) return;
    const uint32_t arow = nG * 2048, brow = nG * kQ8TChunk;
    const uint8_t* ua = xt + (size_t)T * arow;
    const uint8_t* ub = W + (size_t)R0 * brow;
    const uint8_t* ux = xt + xd_off + (size_t)T * 16 * nbp * 4;
    uint32_t vb[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) vb[r] = (min(R0 + r, n_rt - 1) - R0) * brow;
    const uint32_t l16 = 16 * lane, vx = 4 * g * nbp * 4;
    u32x4 a[D][2], b[D][RT][2];
    uint2 dw[D][RT];
    float4 dx[D][4];
    auto load = [&](auto dc, uint32_t G) {
        constexpr int d = decltype(dc)::value;
        const uint8_t* s0 = ua + (size_t)G * 2048;
        a[d][0] = *(const u32x4*)(s0 + l16);
        a[d][1] = *(const u32x4*)(s0 + l16 + 1024);
        const uint8_t* s1 = ub + (size_t)G * kQ8TChunk;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            b[d][r][0] = *(const u32x4*)(s1 + (vb[r] + l16));
            b[d][r][1] = *(const u32x4*)(s1 + (vb[r] + l16) + 1024);
            dw[d][r] = *(const uint2*)(s1 + (vb[r] + 8 * (lane & 15)) + 2048);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) dx[d][e] = *(const float4*)(ux + (size_t)G * 16 + (vx + e * nbp * 4));
    };
    v4f acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = v4f{0.f, 0.f, 0.f, 0.f};
    const v4i magic = {kMagicI, kMagicI, kMagicI, kMagicI};
    auto use = [&](auto dc) {
        constexpr int d = decltype(dc)::value;
        v4i c[4][RT];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const u32x4 A = a[d][j >> 1], B = b[d][r][j >> 1];
                const long al = (j & 1) ? ((uint64_t)A.w << 32 | A.z) : ((uint64_t)A.y << 32 | A.x);
                const long bl = (j & 1) ? ((uint64_t)B.w << 32 | B.z) : ((uint64_t)B.y << 32 | B.x);
                c[j][r] = __builtin_amdgcn_mfma_i32_16x16x32_i8(al, bl, magic, 0, 0, 0);
            }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const uint32_t hw = j < 2 ? dw[d][r].x : dw[d][r].y;
                float dwf = h2f((j & 1) ? hw >> 16 : hw & 0xFFFF);
                asm("" : "+v"(dwf));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float dv = j == 0 ? dx[d][e].x : j == 1 ? dx[d][e].y : j == 2 ? dx[d][e].z : dx[d][e].w;
                    acc[r][e] = fmaf(__int_as_float(c[j][r][e]) - kMagicF, dv * dwf, acc[r][e]);
                }
            }
    };
    static_for<0, D>([&](auto dc) { load(dc, min((uint32_t)decltype(dc)::value, nG - 1)); });
    for (uint32_t G = 0; G < nG; G += D) {
        static_for<0, D>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            if (d == 0 || G + d < nG) {
                use(dc);
                load(dc, min(G + d + D, nG - 1));
            }
        });
    }
    const uint32_t m0 = 16 * T + 4 * g, n0 = 16 * R0 + (lane & 15);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = accumulate && m0 + e < M && n0 + 16 * r < N ? y[(size_t)(m0 + e) * ldy + n0 + 16 * r] : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m0 + e < M && n0 + 16 * r < N)
                y[(size_t)(m0 + e) * ldy + n0 + 16 * r] = accumulate ? o[e] + acc[r][e] : acc[r][e];
    }
}

template <int FMT, int TT, int RT, int KW, int MINW, bool ONEC>
static void launch_tile(const XtLayout& L, const uint8_t* W, const uint8_t* xt, float* y, uint32_t M, uint32_t N,
                        uint32_t ldy, int accumulate, hipStream_t st) {
    const uint32_t n_tt = L.Mp / 16, n_rt = round_up(N, 16) / 16;
    const uint32_t gx = (n_rt + 2 * RT - 1) / (2 * RT), gy = (n_tt + 2 * TT - 1) / (2 * TT);
    hipLaunchKernelGGL((k_gemm<FMT, TT, RT, KW, MINW, ONEC>), dim3(round_up(gx, 8) * gy), dim3(64 * KW), 0, st, W, xt, y,
                       M, N, n_tt, n_rt, L.Kp / 128, L.Kp / 32, L.xd_off, L.dxs_off, ldy, accumulate, gx, gy);
}

template <int RT, int D>
static void launch_q8_16(const XtLayout& L, const uint8_t* W, const uint8_t* xt, float* y, uint32_t M, uint32_t N,
                         uint32_t ldy, int accumulate, hipStream_t st) {
    const uint32_t n_rt = round_up(N, 16) / 16, gx = (n_rt + RT - 1) / RT, gy = L.Mp / 16;
    hipLaunchKernelGGL((k_gemm_q8_16<RT, D>), dim3(round_up(gx, 8) * gy), dim3(64), 0, st, W, xt, y, M, N, n_rt,
                       L.Kp / 128, L.Kp / 32, L.xd_off, ldy, accumulate, gx, gy);
}

// The tile, by the number of 32 x 32 tiles for 1024 SIMDs.  32 x 64 per wave
// reads less per product and needs two waves per SIMD (18432 tiles:
// 1024x18432 160 us, 198 with 32 x 32; 6144: 1024x6144 55 / 62; 4032:
// 200x18432 40 / 48; 3072: 512x6144 36 / 32).  32 x 32 until a SIMD has less
// than about 1.2 waves (1280: 512x2560x9216 59, 84 with 16 x 32; 1152:
// 40x18432 21 / 20; 800: 300x2560x9216 55 / 51), then 16 x 32 down to half a
// wave (720 waves: 130x2560x4096 17, 18 with 16 x 16; 240: 40x2560x9216 30 / 19).
static void launch_q8(const XtLayout& L, const uint8_t* W, const uint8_t* xt, float* y, uint32_t M, uint32_t N,
                      uint32_t ldy, int accumulate, hipStream_t st) {
    const uint64_t tiles = (uint64_t)((M + 31) / 32) * ((N + 31) / 32);
    if (tiles >= 4000)
        launch_tile<EC_Q8_0, 1, 2, 1, 3, true>(L, W, xt, y, M, N, ldy, accumulate, st);
    else if (tiles >= 1216)
        launch_tile<EC_Q8_0, 1, 1, 1, 3, true>(L, W, xt, y, M, N, ldy, accumulate, st);
    else if ((uint64_t)(L.Mp / 16) * ((N + 31) / 32) >= 512)
        launch_q8_16<2, 4>(L, W, xt, y, M, N, ldy, accumulate, st);
    else
        launch_q8_16<1, 6>(L, W, xt, y, M, N, ldy, accumulate, st);
}

// 64 x 64 reads the fewest operand bytes per product and runs two workgroups
// per CU; it needs a few workgroups per slot and tokens that fill its 64 (2016
// workgroups: 387x18432 76 us, 78 with 32 x 64; 320: 512x2560x4096 31 / 28).
// 32 x 64 (two per CU) beats 32 x 32 (three per CU) from 768 workgroups
// (512x12352 68 / 73; 640: 512x2560x4096 28 / 26; 80: 40x2560x9216 25 / 17).
static void launch_q4(const XtLayout& L, const uint8_t* W, const uint8_t* xt, float* y, uint32_t M, uint32_t N,
                      uint32_t ldy, int accumulate, hipStream_t st) {
    const uint64_t t32 = (M + 31) / 32, t64 = (M + 63) / 64, r64 = (N + 63) / 64;
    if (t64 * r64 >= 1280 && 16 * t64 <= 9 * t32)
        launch_tile<EC_Q4_K, 2, 2, 4, 2, true>(L, W, xt, y, M, N, ldy, accumulate, st);
    else if (t32 * r64 >= 768)
        launch_tile<EC_Q4_K, 1, 2, 4, 2, false>(L, W, xt, y, M, N, ldy, accumulate, st);
    else
        launch_tile<EC_Q4_K, 1, 1, 4, 3, false>(L, W, xt, y, M, N, ldy, accumulate, st);
}

}  // namespace ec

using namespace ec;

extern "C" size_t ec_gemm_act_bytes(int fmt, uint32_t M, uint32_t K) {
    if (fmt != EC_Q8_0 && fmt != EC_Q4_K) return 0;
    return xt_layout(fmt, M, K).total;
}

extern "C" int ec_gemm_quantize_act(int fmt, const float* x, void* act, uint32_t M, uint32_t K, void* stream) {
    if (M == 0) return EC_OK;
    if (!x || !act || (fmt != EC_Q8_0 && fmt != EC_Q4_K) || K == 0 || K % 32 || (fmt == EC_Q4_K && K % 256))
        return ec_set_error(EC_ERR_ARG, "ec_gemm_quantize_act: bad argument (Q8_0: K % 32 == 0, Q4_K: K % 256 == 0)");
    if ((uintptr_t)x % 16)  // the quantizers read x with 16-byte loads
        return ec_set_error(EC_ERR_ARG, "ec_gemm_quantize_act: x must be 16-byte aligned");
    const XtLayout L = xt_layout(fmt, M, K);
    const uint32_t nbp = L.Kp / 32;
    if (fmt == EC_Q8_0)
        hipLaunchKernelGGL(k_gemm_quantize_x8, dim3((nbp + 8 * kQxSteps - 1) / (8 * kQxSteps), L.Mp / 4), dim3(256), 0,
                           (hipStream_t)stream, x, (uint8_t*)act, M, K, K, L.nch, nbp, L.xd_off);
    else
        hipLaunchKernelGGL(k_gemm_quantize_x4v, dim3((L.nch + 1) / 2, L.Mp / 4), dim3(256), 0, (hipStream_t)stream,
                           x, (uint8_t*)act, M, K, K, L.nch, nbp, L.xd_off, L.dxs_off);
    EC_CHECK_LAUNCH();
    return EC_OK;
}

extern "C" int ec_gemm(int fmt, const void* tiled, const void* act, float* y, uint32_t M, uint32_t N, uint32_t K,
                       uint32_t ldy, int accumulate, void* stream) {
    if (M == 0 || N == 0) return EC_OK;
    if (!tiled || !act || !y || ldy < N || (fmt != EC_Q8_0 && fmt != EC_Q4_K) || K == 0 ||
        (fmt == EC_Q4_K && K % 256) || K % 32)
        return ec_set_error(EC_ERR_ARG, "ec_gemm: bad argument");
    const XtLayout L = xt_layout(fmt, M, K);
    (fmt == EC_Q8_0 ? launch_q8 : launch_q4)(L, (const uint8_t*)tiled, (const uint8_t*)act, y, M, N, ldy, accumulate,
                                             (hipStream_t)stream);
    EC_CHECK_LAUNCH();
    return EC_OK;
}
