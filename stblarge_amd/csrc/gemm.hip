// Multi-token expert GEMM on CDNA4 scaled MFMA: Y[m][n] = sum_k Aq[m][k] * Wdeq[n][k].
//
// Reference: fp8_gemm / fp4_gemm of ref/kernel.py:85-102 with M = 64 rows of activations:
//   A = act_quant(X, block, "ue8m0") (e4m3 codes, power-of-two scales per `block` along K),
//   FP8 W: e4m3 with fp32 scales per 128x128 block; FP4 W: e2m1 with E8M0 scales per 32 along K;
//   fp32 accumulation, bf16 output.
// Kernels:
//   k_act_quant_e4m3  X bf16 -> e4m3 codes + E8M0 scale bytes, one 16-lane group per block of 128
//                     (or 4 lanes per block of 32); the e4m3 rounding uses v_cvt_pk_fp8_f32, which
//                     equals the round-to-nearest-even encoder bit for bit on every bf16 input;
//                     k_act_quant_e4m3_ops the same codes in MFMA operand order;
//   k_gemm, ...       v_mfma_scale_f32_16x16x128_f8f6f4 with A = e4m3 activations and B = the e4m3 or
//                     e2m1 weights. The activation scales (powers of two) and the FP4 weight scales
//                     (E8M0) are the MFMA's own per-32 scale operands, so the hardware applies them
//                     exactly; the FP8 weights' fp32 block scale multiplies each 128-K step's product
//                     in fp32. gemm_plan (gemm_plan.hpp) chooses between them: k_gemm_one (the configurations' shapes)
//                     and k_gemm_waves, one launch over all of K by waves that each take a part of it;
//                     k_gemm and k_gemm_reduce, split K; k_gemm_tile, many rows through LDS, on operands
//                     laid out by k_gemm_prep;
//   k_gemm_pack       the weight codes rearranged once into MFMA operand order (WOPS below), which
//                     every kernel reads to the same results bit for bit.
// Operand layout of the 16x16x128 f8f6f4 MFMA (probed on gfx950): lane l = r + 16 g holds row r of A
// (column r of B); e4m3 operands hold K bytes [16g, 16g+16) and [64+16g, 64+16g+16) of the 128-K
// step, e2m1 operands K elements [32g, 32g+32) (low nibble first); the lane's E8M0 scale covers K
// block [32g, 32g+32); D lane l holds rows 4g..4g+3 of column r.
#include "abi_util.hpp"
#include "common.hpp"
#include "gemm_plan.hpp"

namespace stbl {

// ---- operand order --------------------------------------------------------------------------------

// WOPS: weights in MFMA operand order. Per group G of 16 columns and 128-K step s, the 64 lanes'
// 16-byte operand pieces lie in lane order: FP4 one kilobyte, lane r + 16 g holding bytes [16g,
// 16g + 16) of column 16 G + r's 64-byte step; FP8 two kilobytes, the first holding bytes [16g, 16g
// + 16) and the second [64 + 16g, 64 + 16g + 16) of the column's 128-byte step. Blocks run over the
// steps of a group, then over the groups, so a column group's weights stay one contiguous run and
// the packed array has the size of the codes. Byte offset of the block (G, s):
__device__ __forceinline__ size_t ops_block(int G, int s, int KS, bool fp4) {
    return ((size_t)G * KS + s) * (fp4 ? 1024 : 2048);
}

// ---- activation quantization --------------------------------------------------------------------

// x bf16 [rows][k] -> codes e4m3 [rows][k], scales E8M0 bytes [rows][k / block]. Each thread takes 8
// consecutive values; block / 8 threads share a block (8 or 16 lanes of one wave).
__global__ __launch_bounds__(256) void k_act_quant_e4m3(const uint16_t *__restrict__ x, int n8, int block,
                                                        uint8_t *__restrict__ codes, uint8_t *__restrict__ scales) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool ok = i < n8;
    const u32x4 v = *(const u32x4 *)(x + (size_t)(ok ? i : 0) * 8);
    float f[8];
#pragma unroll
    for (int j = 0; j < 4; j++) f[2 * j] = bf16_lo(v[j]), f[2 * j + 1] = bf16_hi(v[j]);
    float a = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) a = fmaxf(a, fabsf(f[j]));
    const int lanes = block >> 3;  // 4 or 16, a power of two
    for (int o = 1; o < lanes; o <<= 1) a = fmaxf(a, __shfl_xor(a, o, kWave));
    const float s = pow2_ceil(fmaxf(a, 1e-4f) * (1.0f / 448.0f));
    // 1/s, exact; 0 for s = +Inf (a block holding an infinity), where x * 0 is x / s: a signed zero for
    // a finite x, NaN for an infinite one
    const float inv = __builtin_isinf(s) ? 0.f : __uint_as_float((uint32_t)(254 - ((__float_as_uint(s) >> 23) & 0xffu)) << 23);
    uint32_t w[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        // x / s is exact (s is a power of two); the clamp is ref/kernel.py:41's
        float q[4];
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = fminf(fmaxf(f[4 * j + e] * inv, -448.f), 448.f);
        int p = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
        p = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], p, true);
        w[j] = (uint32_t)p;
    }
    if (!ok) return;
    *(u32x2 *)(codes + (size_t)i * 8) = u32x2{w[0], w[1]};
    if ((threadIdx.x & (lanes - 1)) == 0) scales[(size_t)i * 8 / block] = (uint8_t)((__float_as_uint(s) >> 23) & 0xffu);
}

// The quantization of one operand lane: src points at its row's 16 values of the step's first half, 16 g
// on; q gets the codes of both halves, sb their scale bytes.
__device__ __forceinline__ void quant_ops(const uint16_t *src, int block, u32x4 (&out)[2], uint32_t (&sb)[2]) {
    float f[2][16];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const u32x4 v = *(const u32x4 *)(src + 64 * h + 8 * q);
#pragma unroll
            for (int j = 0; j < 4; j++) f[h][8 * q + 2 * j] = bf16_lo(v[j]), f[h][8 * q + 2 * j + 1] = bf16_hi(v[j]);
        }
    }
    float a[2] = {0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < 16; j++) a[h] = fmaxf(a[h], fabsf(f[h][j]));
#pragma unroll
    for (int h = 0; h < 2; h++) a[h] = fmaxf(a[h], __shfl_xor(a[h], 16, kWave));  // the lane pair g, g ^ 1
    if (block == 128) {
        const float t = fmaxf(a[0], a[1]);
        a[0] = a[1] = fmaxf(t, __shfl_xor(t, 32, kWave));
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const float sc = pow2_ceil(fmaxf(a[h], 1e-4f) * (1.0f / 448.0f));
        // 1/sc, exact, or 0 for sc = +Inf, as in k_act_quant_e4m3
        const float inv =
            __builtin_isinf(sc) ? 0.f : __uint_as_float((uint32_t)(254 - ((__float_as_uint(sc) >> 23) & 0xffu)) << 23);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // x / sc is exact (sc is a power of two); the clamp is ref/kernel.py:41's
            float q[4];
#pragma unroll
            for (int e = 0; e < 4; e++) q[e] = fminf(fmaxf(f[h][4 * j + e] * inv, -448.f), 448.f);
            int p = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
            p = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], p, true);
            out[h][j] = (uint32_t)p;
        }
        sb[h] = (__float_as_uint(sc) >> 23) & 0xffu;
    }
}

// The same quantization written in MFMA operand order (stbl_amd_gemm's one-launch plans, whose
// operand loads then each read one contiguous kilobyte): per group of 16 rows and 128-K step, 2 KB,
// in which the 16 bytes lane l = r + 16 g of an operand load takes (row r, bytes [16 g, 16 g + 16) of
// the step's first 64, then of its second 64) sit at l * 16 of the first, then of the second
// kilobyte. One wave per group and step: lane l reads row r's 16 values at [16 g, 16 g + 16) of each
// half of the step and stores their codes as that piece, so each store instruction writes a
// contiguous kilobyte (measured against 8-byte stores scattered into the same layout by
// k_act_quant_e4m3's lanes: full FP4 GEMM at 2048x7168 10.14 -> 9.75 us, FP8 12.83 -> 12.43). A block's amax
// comes from the lanes of the same row: all four for a 128-block (xor 16, 32), the pair g, g ^ 1 of
// one half for a 32-block (block 2 h + g / 2 of the step). Rows past m (up to the group's 16) store
// zero codes and no scales. The codes and scales of rows < m are k_act_quant_e4m3's, byte for byte.
__global__ __launch_bounds__(64) void k_act_quant_e4m3_ops(const uint16_t *__restrict__ x, int m, int k, int block,
                                                          uint8_t *__restrict__ codes, uint8_t *__restrict__ scales) {
    const int ks = k >> 7;
    const int w = blockIdx.x, mg = w / ks, s = w % ks;  // grid: ceil(m / 16) * ks waves
    const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
    const int row = mg * 16 + r;
    const bool ok = row < m;
    u32x4 q[2];
    uint32_t sb[2];
    quant_ops(x + (size_t)(ok ? row : 0) * k + (size_t)s * 128 + 16 * g, block, q, sb);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        *(u32x4 *)(codes + ops_block(mg, s, ks, false) + 1024 * h + lane * 16) = ok ? q[h] : u32x4{0, 0, 0, 0};
        if (ok && block == 128 && h == 0 && g == 0) scales[(size_t)row * ks + s] = (uint8_t)sb[0];
        if (ok && block == 32 && (g & 1) == 0) scales[(size_t)row * (k >> 5) + 4 * s + 2 * h + (g >> 1)] = (uint8_t)sb[h];
    }
}

// ---- GEMM ---------------------------------------------------------------------------------------

// codes [n][k / 2] (FP4) or [n][k] (FP8), n % 16 == 0, k % 128 == 0 -> the same codes in operand
// order. Thread t moves the 16-byte piece t of the packed array.
__global__ __launch_bounds__(256) void k_gemm_pack(const uint8_t *__restrict__ codes, uint8_t *__restrict__ packed,
                                                   int n, int k, int fp4, size_t pieces) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= pieces) return;
    const int KS = k >> 7, lane = (int)(t & 63), r = lane & 15, g = lane >> 4;
    size_t src;
    if (fp4) {
        const size_t blk = t >> 6;  // G * KS + s
        const size_t G = blk / KS, st = blk % KS;
        src = (16 * G + r) * (size_t)(k >> 1) + st * 64 + 16 * g;
    } else {
        const size_t blk = t >> 7, half = (t >> 6) & 1;  // (G * KS + s) * 2 + half
        const size_t G = blk / KS, st = blk % KS;
        src = (16 * G + r) * (size_t)k + st * 128 + 64 * half + 16 * g;
    }
    *(u32x4 *)(packed + 16 * t) = *(const u32x4 *)(codes + src);
}

// One workgroup owns a 64 x 64 output tile (MT m-tiles x NT n-tiles of 16 x 16) and a slice of up to NW 128-K
// steps; wave w takes step w of the slice for all MT * NT tiles, loading its activations and weights
// straight from global memory (no operand is shared between waves, so nothing is staged through LDS),
// from addresses clamped into the buffers; a step past the slice gets zero operands instead of a
// branch. The waves' tiles are summed through LDS in wave order, the workgroup writes its slice's partial
// tile, and k_gemm_reduce adds the slices in order. (Summing the slices in the last workgroup to finish
// needs an agent-scope release/acquire per workgroup, which writes back and invalidates the XCD's L2 each
// time: measured at about 4x the whole GEMM, so the kernel boundary is the synchronization point.) A
// rows are K bytes apart. Partial tiles and the LDS sum hold f32x4 q = t * 64 + lane with t = m-tile * NT +
// n-tile.
template <bool FP4W, bool WOPS>
__global__ __launch_bounds__(512) void k_gemm(const uint8_t *__restrict__ wc, const void *__restrict__ ws,
                                              const uint8_t *__restrict__ aq, const uint8_t *__restrict__ as_,
                                              f32x4 *__restrict__ part, int M, int N, int K, int act_shift, int ntiles,
                                              int slices, int steps_wg) {
    constexpr int MT = 4, NT = 4, NW = 8, kTileVecs = MT * NT * 64, kThreads = NW * 64;
    __shared__ f32x4 red[NW * kTileVecs];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    const int tile = blockIdx.x % ntiles, slice = blockIdx.x / ntiles;
    const int n0 = tile * 16 * NT, KS = K >> 7;
    const int step = slice * steps_wg + wave;
    const bool live = step < min(KS, (slice + 1) * steps_wg);  // wave-uniform

    // 1. loads: lane (r, g) holds rows 16 mt + r of A and columns n0 + 16 nt + r of W
    u32x4 av[MT][2];
    uint32_t asc[MT];
    u32x4 bv[NT][FP4W ? 1 : 2];
    uint32_t bsc[NT];
    const size_t kb = (size_t)(live ? step : 0) * 128;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int m = min(16 * mt + r, M - 1);
        const uint8_t *row = aq + (size_t)m * K + kb;
        av[mt][0] = *(const u32x4 *)(row + 16 * g);
        av[mt][1] = *(const u32x4 *)(row + 64 + 16 * g);
        asc[mt] = as_[(size_t)m * (K >> act_shift) + ((kb + 32 * g) >> act_shift)];
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int n = min(n0 + 16 * nt + r, N - 1);
        if constexpr (WOPS) {  // operand order: one contiguous kilobyte (two for FP8) per load
            const uint8_t *blk = wc + ops_block(min((n0 >> 4) + nt, (N >> 4) - 1), (int)(kb >> 7), KS, FP4W) + 16 * lane;
            bv[nt][0] = *(const u32x4 *)blk;
            if constexpr (!FP4W) bv[nt][1] = *(const u32x4 *)(blk + 1024);
            if constexpr (FP4W) bsc[nt] = ((const uint8_t *)ws)[(size_t)n * (K >> 5) + (kb >> 5) + g];
        } else if constexpr (FP4W) {
            bv[nt][0] = *(const u32x4 *)(wc + (size_t)n * (K >> 1) + (kb >> 1) + 16 * g);
            bsc[nt] = ((const uint8_t *)ws)[(size_t)n * (K >> 5) + (kb >> 5) + g];
        } else {
            const uint8_t *row = wc + (size_t)n * K + kb;
            bv[nt][0] = *(const u32x4 *)(row + 16 * g);
            bv[nt][1] = *(const u32x4 *)(row + 64 + 16 * g);
        }
    }
    float wsc = 0.f;
    if constexpr (!FP4W) wsc = ((const float *)ws)[(size_t)(n0 >> 7) * KS + (kb >> 7)];
    // 2. MFMAs
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const u32x4 z4 = {0, 0, 0, 0};
    i32x8 b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const u32x4 b0 = live ? bv[nt][0] : z4;
        if constexpr (FP4W) {
            b[nt] = i32x8{(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], 0, 0, 0, 0};
        } else {
            const u32x4 b1 = live ? bv[nt][1] : z4;
            b[nt] = i32x8{(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const u32x4 a0 = live ? av[mt][0] : z4, a1 = live ? av[mt][1] : z4;
        const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            if constexpr (FP4W) {
                acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[nt], acc[mt][nt], 0, 4, 0, (int)asc[mt],
                                                                               0, (int)bsc[nt]);
            } else {
                const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[nt], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0,
                                                                                  0, (int)asc[mt], 0, 127);
                const float sw = live ? wsc : 0.f;
#pragma unroll
                for (int e = 0; e < 4; e++) acc[mt][nt][e] = fmaf(sw, d[e], acc[mt][nt][e]);
            }
        }
    }
    // 3. the workgroup's sum, in wave order; thread tid takes q = tid + kThreads j
#pragma unroll
    for (int t = 0; t < MT * NT; t++) red[(wave * MT * NT + t) * 64 + lane] = acc[t / NT][t % NT];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTileVecs / kThreads; j++) {
        const int q = tid + kThreads * j;
        f32x4 v = red[q];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w * kTileVecs + q];
        part[((size_t)tile * slices + slice) * kTileVecs + q] = v;
    }
}

// Y = the slices' partial tiles added in slice order; thread i takes f32x4 i of every tile (the
// layout k_gemm stored them in), so partial reads are contiguous per slice.
__global__ __launch_bounds__(256) void k_gemm_reduce(const f32x4 *__restrict__ part, int slices, int ntiles,
                                                     void *__restrict__ y, int y_f32, int M, int N) {
    constexpr int NT = 4, kTileVecs = 4 * NT * 64;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ntiles * kTileVecs) return;
    const int tile = i / kTileVecs, q = i % kTileVecs;
    const f32x4 *tp = part + (size_t)tile * slices * kTileVecs + q;
    // slices are loaded up to 8 at a time, all loads issued before the first add (a plain loop waits
    // for each load in turn), and added in slice order
    constexpr int kBatch = 8;
    f32x4 s = tp[0];
    for (int sl0 = 1; sl0 < slices; sl0 += kBatch) {
        f32x4 v[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; i++)
            if (sl0 + i < slices) v[i] = tp[(size_t)(sl0 + i) * kTileVecs];
#pragma unroll
        for (int i = 0; i < kBatch; i++)
            if (sl0 + i < slices) s += v[i];
    }
    const int t = q >> 6, ql = q & 63, mt = t / NT, nt = t % NT;
    const int n = tile * 16 * NT + 16 * nt + (ql & 15);
    if (n >= N) return;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int m = 16 * mt + 4 * (ql >> 4) + e;
        if (m >= M) continue;
        if (y_f32) ((float *)y)[(size_t)m * N + n] = s[e];
        else ((uint16_t *)y)[(size_t)m * N + n] = f32_to_bf16_bits(s[e]);
    }
}

// One-launch GEMM for K % 512 == 0: a workgroup owns a 16 MT x 16 NT output tile over all of K; wave w
// takes the 4 SW consecutive 128-K steps [4 SW w, 4 SW w + 4 SW) (waves past K do nothing), and the
// waves' tiles are summed through LDS in wave order, so the result does not depend on timing.
// Three things keep the loads, which bound this kernel, few and cheap (each measured):
//  - every load of a wave is issued before its first MFMA (a scheduling fence keeps the compiler
//    from interleaving waits with the loads);
//  - the operand loads alternate 64-byte halves: an MFMA operand load reads 16 rows x 64 bytes, all
//    in the same half of their 128-byte lines, which the vector L1 serves at half rate. Lanes of odd
//    rows (odd columns for W) read the other half first, and a per-lane select puts the halves back
//    in operand order. For FP4 W, whose step is 64 bytes, steps s and s + 1 of a column are the two
//    halves of one line, so steps come in pairs;
//  - scales are loaded four steps per instruction (one dword of A scale bytes per row with
//    act_block 128, 16 bytes per row or column for the per-32 scales), not one byte per step: a
//    one-byte wave load costs the L1 as much as a 1 KB one. The MFMA reads the low byte of its scale
//    operand, so each lane shifts its byte down.
template <bool FP4W, int MT, int NT, int NW, int QW, bool AARR, bool WOPS>
__global__ __launch_bounds__(NW * 64) void k_gemm_one(const uint8_t *__restrict__ wc, const void *__restrict__ ws,
                                                      const uint8_t *__restrict__ aq, const uint8_t *__restrict__ as_,
                                                      void *__restrict__ y, int y_f32, int M, int N, int K, int act32,
                                                      int ntiles) {
    constexpr int SW = 4 * QW;  // steps per wave
    constexpr int kTileVecs = MT * NT * 64;
    constexpr int kThreads = NW * 64;
    __shared__ f32x4 red[NW * kTileVecs];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool odd = r & 1;
    const int h0 = odd ? 64 : 0, h1 = 64 - h0;
    const int tile = blockIdx.x % ntiles, m0 = (blockIdx.x / ntiles) * 16 * MT;
    const int n0 = tile * 16 * NT, KS = K >> 7;
    const int s0 = wave * SW;
    const int nst = max(0, min(SW, KS - s0));  // wave-uniform; a multiple of 4

    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (nst > 0) {
        // 1. loads: lane (r, g) holds rows 16 mt + r of A and columns n0 + 16 nt + r of W; step
        // s < nst is step s0 + s of K (nst is a multiple of 4: KS % 4 == 0; steps past nst read
        // step s0 again and are not used). Issued in order of their latency:
        // the scales, then W (from HBM: a column tile's weights are first read by one of its row
        // groups), then A (the activations, resident in L2): 2048x7168 FP4 8.55 -> 8.15 us, FP8
        // 11.04 -> 10.60, 7168x2048 6.86 -> 6.33 against A, W, then the scales.
        u32x4 av[SW][MT][2];
        u32x4 bv[SW][NT][FP4W ? 1 : 2];
        u32x4 asw[QW][MT];  // A scale bytes: dword 0 (act_block 128) or 16 bytes (act_block 32)
        u32x4 bsw[QW][NT];  // FP4 W scale bytes, 16 per column per 4 steps
        float wsc[SW];      // FP8 W: the 128 x 128 block scale of each step
#pragma unroll
        for (int q = 0; q < QW; q++) {
            // groups of 4 steps past nst (the last wave of a K with KS % SW == 4) reload the last
            // group's words, in range, and are not used
            const int sq = s0 + 4 * min(q, (nst >> 2) - 1);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const size_t m = min(m0 + 16 * mt + r, M - 1);
                if (act32) asw[q][mt] = *(const u32x4 *)(as_ + m * (K >> 5) + 4 * sq);
                else asw[q][mt][0] = *(const uint32_t *)(as_ + m * KS + sq);
            }
            if constexpr (FP4W) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    bsw[q][nt] = *(const u32x4 *)((const uint8_t *)ws + (size_t)min(n0 + 16 * nt + r, N - 1) * (K >> 5) + 4 * sq);
            }
        }
#pragma unroll
        for (int s = 0; s < SW; s++) {
            const size_t kb = (size_t)(s < nst ? s0 + s : s0) * 128;
            if constexpr (WOPS) {  // operand order: steps s and s + 1 of a group are adjacent blocks
                if (!FP4W || s % 2 == 0) {
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) {
                        const uint8_t *blk = wc + ops_block(min((n0 >> 4) + nt, (N >> 4) - 1), (int)(kb >> 7), KS, FP4W) + 16 * lane;
                        bv[s][nt][0] = *(const u32x4 *)blk;
                        if constexpr (FP4W) bv[s + 1][nt][0] = *(const u32x4 *)(blk + 1024);
                        else bv[s][nt][1] = *(const u32x4 *)(blk + 1024);
                    }
                }
                if constexpr (!FP4W) wsc[s] = ((const float *)ws)[(size_t)(n0 >> 7) * KS + (kb >> 7)];
            } else if constexpr (FP4W) {
                if (s % 2 == 0) {
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) {
                        const uint8_t *row = wc + (size_t)min(n0 + 16 * nt + r, N - 1) * (K >> 1) + (kb >> 1);
                        bv[s][nt][0] = *(const u32x4 *)(row + h0 + 16 * g);
                        bv[s + 1][nt][0] = *(const u32x4 *)(row + h1 + 16 * g);
                    }
                }
            } else {
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const uint8_t *row = wc + (size_t)min(n0 + 16 * nt + r, N - 1) * K + kb;
                    bv[s][nt][0] = *(const u32x4 *)(row + h0 + 16 * g);
                    bv[s][nt][1] = *(const u32x4 *)(row + h1 + 16 * g);
                }
                wsc[s] = ((const float *)ws)[(size_t)(n0 >> 7) * KS + (kb >> 7)];
            }
        }
#pragma unroll
        for (int s = 0; s < SW; s++) {
            const size_t kb = (size_t)(s < nst ? s0 + s : s0) * 128;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if constexpr (AARR) {  // operand order (k_act_quant_e4m3_ops): two contiguous kilobytes
                    const uint8_t *blk = aq + ops_block(operand_group(m0, mt, M), (int)(kb >> 7), KS, false) + lane * 16;
                    av[s][mt][0] = *(const u32x4 *)blk;
                    av[s][mt][1] = *(const u32x4 *)(blk + 1024);
                } else {
                    const uint8_t *row = aq + (size_t)min(m0 + 16 * mt + r, M - 1) * K + kb;
                    av[s][mt][0] = *(const u32x4 *)(row + h0 + 16 * g);
                    av[s][mt][1] = *(const u32x4 *)(row + h1 + 16 * g);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // 2. halves back in operand order, then the MFMAs, NT independent accumulators per step
        // (steps past nst, in the last wave of a K with KS % SW == 4, take zero weights: a branch
        // there made the compiler wait for each step's loads before its MFMAs)
        const int gsh = 8 * g;
        const u32x4 z4 = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < SW; s++) {
            const bool live = SW == 4 || s < nst;  // SW == 4: nst is 0 or 4
            i32x8 b[NT];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                if constexpr (FP4W) {
                    const u32x4 x0 = bv[s & ~1][nt][0], x1 = bv[s | 1][nt][0];
                    const u32x4 b0 = live ? (WOPS ? bv[s][nt][0] : (odd == (s & 1)) ? x0 : x1) : z4;
                    b[nt] = i32x8{(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], 0, 0, 0, 0};
                } else {
                    const u32x4 x0 = bv[s][nt][0], x1 = bv[s][nt][1];
                    const bool sw = odd && !WOPS;  // operand-order weights need no half swap
                    const u32x4 b0 = live ? (sw ? x1 : x0) : z4, b1 = live ? (sw ? x0 : x1) : z4;
                    b[nt] = i32x8{(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
                }
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const u32x4 x0 = av[s][mt][0], x1 = av[s][mt][1];
                const u32x4 a0 = odd && !AARR ? x1 : x0, a1 = odd && !AARR ? x0 : x1;
                const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
                const uint32_t aw = asw[s / 4][mt][act32 ? s % 4 : 0];
                const int ascale = (int)(act32 ? aw >> gsh : aw >> (8 * (s % 4)));
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    if constexpr (FP4W) {
                        const int bscale = (int)(bsw[s / 4][nt][s % 4] >> gsh);
                        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[nt], acc[mt][nt], 0, 4, 0,
                                                                                       ascale, 0, bscale);
                    } else {
                        const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                            a, b[nt], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, ascale, 0, 127);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[mt][nt][e] = fmaf(wsc[s], d[e], acc[mt][nt][e]);
                    }
                }
            }
        }
    }
    // 3. the workgroup's sum in wave order (idle waves add zeros); thread tid takes q = tid + kThreads j
#pragma unroll
    for (int t = 0; t < MT * NT; t++) red[(wave * MT * NT + t) * 64 + lane] = acc[t / NT][t % NT];
    __syncthreads();
    constexpr int kPer = (kTileVecs + kThreads - 1) / kThreads;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int q = tid + kThreads * j;
        if (q >= kTileVecs) break;
        f32x4 v = red[q];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w * kTileVecs + q];
        // element e of v is row 16 mt + 4 g' + e, column n0 + 16 nt + r' of the lane q % 64
        const int t = q >> 6, ql = q & 63, mt = t / NT, nt = t % NT;
        const int n = n0 + 16 * nt + (ql & 15);
        if (n >= N) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + 16 * mt + 4 * (ql >> 4) + e;
            if (m >= M) continue;
            if (y_f32) ((float *)y)[(size_t)m * N + n] = v[e];
            else ((uint16_t *)y)[(size_t)m * N + n] = f32_to_bf16_bits(v[e]);
        }
    }
}

// GEMM of many rows: a workgroup of WR x WC waves owns a BM x BN output tile over all of K, each wave a
// BM / WR x BN / WC part. A 128-K step's A rows, W columns and scale dwords go to LDS once for the
// workgroup, by loads that write LDS directly (they hold no registers), S - 1 steps ahead of their use,
// and a wave reads the next step's operands from LDS while its products of this one run. A and packed W
// lie in LDS in operand order, row-major W with its 16-byte pieces permuted by the column, so that operand
// reads hit every bank once.
// The sum runs as a call of 64 rows at the same n and k sums (gemm_plan): steps in groups of `group`;
// within a group CHAIN keeps one running sum (FP4: in the MFMA's accumulator, FP8: an FMA per element and
// step), otherwise each step's product is rounded and added; then the groups' sums are added in order.
// Measured (FP4 / FP8, with k_gemm_prep, us) against 64 rows a launch: 1024 x 7168 x 2048 84.6 / 107.2 -> 31.1 /
// 33.9, 300 x 2048 x 7168 38.5 / 48.0 -> 22.6 / 26.8. What bounds it: of 23.6 us at 1024 x 7168 x 2048 FP4, 17.5
// are the products alone (7.5 at the matrix cores' rate; a 64 x 128 tile's 16 steps are short against its
// start and end), 9.5 the loads and LDS reads alone.
// 64 lanes x 16 (4) bytes at base + off -> LDS at lds + 16 (4) x lane. The LDS address goes through M0,
// which is left as it was. Counted by vmcnt (wait_lds_vmem): the compiler's builtin for this load makes it
// wait for every such load before any LDS read that could alias, which is each step's.
__device__ __forceinline__ void lds_dma16(uint32_t lds, const uint8_t *base, uint32_t off) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(lds), "v"(off), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void lds_dma4(uint32_t lds, const uint8_t *base, uint32_t off) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(lds), "v"(off), "s"(base)
                 : "memory");
}
template <int N>
__device__ __forceinline__ void wait_lds_vmem() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

template <bool FP4W, int BM, int BN, int WR, int WC, int S, bool CHAIN, bool WOPS>
__global__ __launch_bounds__(WR *WC * 64, 2) void k_gemm_tile(const uint8_t *__restrict__ wc, const void *__restrict__ ws,
                                                      const uint8_t *__restrict__ aq, const uint8_t *__restrict__ as4,
                                                      const uint8_t *__restrict__ ws4, void *__restrict__ y, int y_f32,
                                                      int M, int N, int K, int group, int mtiles, int ntiles) {
    constexpr int W = WR * WC, WM = BM / WR, WN = BN / WC, MT = WM / 16, NT = WN / 16;
    constexpr int kStepB = FP4W ? 64 : 128;                     // bytes of a W column per step
    constexpr int kA = BM * 128, kB = BN * kStepB;              // LDS bytes per step
    constexpr int kSA = BM * 4, kSB = FP4W ? BN * 4 : 0, kStage = kA + kB + kSA + kSB;
    constexpr int kPieces = (kA + kB) / 1024, PV = (kPieces + W - 1) / W;  // kilobyte loads, and per wave
    constexpr int SV = (BM + (FP4W ? BN : 0)) / 64;             // scale loads per workgroup (64 dwords each)
    constexpr int SW = (SV + W - 1) / W;                        // ... per wave (the last waves repeat one)
    constexpr int kLoads = PV + SW;  // the last waves repeat a load where they do not divide
    static_assert(BM % 64 == 0 && BN % 64 == 0 && (S - 1) * kLoads < 64, "tile");
    extern __shared__ __align__(1024) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WC, wn = wave % WC;
    const int KS = K >> 7;
    // workgroup b runs on XCD b % 8: each XCD gets a contiguous run of tiles, row tiles innermost, so
    // its L2 holds its columns' weights while every row tile passes over them
    const int total = mtiles * ntiles, xcd = blockIdx.x & 7, per = total >> 3, rem = total & 7;
    const int t0 = xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int m0 = (t0 % mtiles) * BM, n0 = (t0 / mtiles) * BN;

    // this lane's 32-bit offsets from the tile's uniform bases; rows past the edge reload the last
    const int mg = (M + 15) >> 4;
    const uint8_t *pa = aq + ops_block(m0 >> 4, 0, KS, false);
    const uint8_t *pb = wc + (WOPS ? ops_block(n0 >> 4, 0, KS, FP4W) : (size_t)n0 * (FP4W ? K >> 1 : K));
    uint32_t off[PV], os[SW];
#pragma unroll
    for (int i = 0; i < PV; i++) {
        const int q = min(i * W + wave, kPieces - 1), u = (q - kA / 1024) * 64 + lane;
        if (q < kA / 1024) {
            off[i] = (uint32_t)ops_block(min(q >> 1, mg - 1 - (m0 >> 4)), 0, KS, false) + (uint32_t)((q & 1) * 1024 + lane * 16);
        } else if constexpr (WOPS) {
            const int blk = FP4W ? u >> 6 : u >> 7;
            off[i] = (uint32_t)ops_block(min(blk, (N >> 4) - 1 - (n0 >> 4)), 0, KS, FP4W) + (uint32_t)(FP4W ? u & 63 : u & 127) * 16;
        } else if constexpr (FP4W) {
            const int col = u >> 2;
            off[i] = (uint32_t)min(col, N - 1 - n0) * (uint32_t)(K >> 1) + (uint32_t)(((u & 3) ^ ((col >> 1) & 3)) * 16);
        } else {
            const int col = u >> 3;
            off[i] = (uint32_t)min(col, N - 1 - n0) * (uint32_t)K + (uint32_t)(((u & 7) ^ (col & 7)) * 16);
        }
    }
    constexpr uint32_t kAdvB = WOPS ? (FP4W ? 1024 : 2048) : kStepB;
#pragma unroll
    for (int i = 0; i < SW; i++) {
        const int q = min(wave * SW + i, SV - 1);  // 64 rows of A, then of W
        const bool a = q < BM / 64;
        const int row = a ? m0 + q * 64 + lane : n0 + (q - BM / 64) * 64 + lane;
        os[i] = 4u * (uint32_t)min(row, (a ? M : N) - 1);
    }
    const int spa = 4 * M, spw = 4 * N;  // bytes per step of the scales
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    auto issue = [&](int s, int st) {
        const uint32_t base = lds0 + st * kStage;
#pragma unroll
        for (int i = 0; i < PV; i++) {
            const int q = min(i * W + wave, kPieces - 1);
            lds_dma16(base + q * 1024, q < kA / 1024 ? pa + (size_t)s * 2048 : pb + (size_t)s * kAdvB, off[i]);
        }
#pragma unroll
        for (int i = 0; i < SW; i++) {
            const int q = min(wave * SW + i, SV - 1);
            lds_dma4(base + kA + kB + q * 256, q < BM / 64 ? as4 + (size_t)s * spa : ws4 + (size_t)s * spw, os[i]);
        }
    };
    const int a0 = wm * MT * 2048 + lane * 16, a1 = a0 + 1024;
    int b0, b1 = 0;
    if constexpr (WOPS) {
        b0 = kA + wn * NT * (FP4W ? 1024 : 2048) + lane * 16, b1 = b0 + 1024;
    } else if constexpr (FP4W) {
        b0 = kA + (wn * WN + r) * 64 + ((g ^ ((r >> 1) & 3)) << 4);
    } else {
        const int lb = kA + (wn * WN + r) * 128;
        b0 = lb + ((g ^ (r & 7)) << 4), b1 = lb + (((g + 4) ^ (r & 7)) << 4);
    }
    const int sa0 = kA + kB + (wm * WM + r) * 4 + g, sb0 = kA + kB + kSA + (wn * WN + r) * 4 + g;
    const float *wsc = (const float *)ws + (size_t)(n0 >> 7) * KS;

    f32x4 acc[MT][NT], tot[MT][NT];
#pragma unroll
    for (int i = 0; i < MT * NT; i++) acc[i / NT][i % NT] = tot[i / NT][i % NT] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Frag {  // a wave's operands of one step
        i32x8 a[MT], b[NT];
        int sa[MT], sb[NT];
    };
    auto read = [&](Frag &F, int st) {
        const uint8_t *T = smem + st * kStage;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const u32x4 x0 = *(const u32x4 *)(T + b0 + nt * (FP4W ? 1024 : 2048));
            u32x4 x1 = {0, 0, 0, 0};
            if constexpr (!FP4W) x1 = *(const u32x4 *)(T + b1 + nt * 2048);
            F.b[nt] = i32x8{(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
            F.sb[nt] = FP4W ? T[sb0 + nt * 64] : 127;
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const u32x4 x0 = *(const u32x4 *)(T + a0 + mt * 2048), x1 = *(const u32x4 *)(T + a1 + mt * 2048);
            F.a[mt] = i32x8{(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
            F.sa[mt] = T[sa0 + mt * 64];
        }
    };
    float sw = FP4W ? 0.f : wsc[0];
    int left = group, st = 0;
    // Step s, its operands in F; reads step s + 1's into G. This wave's loads of step s + 1 are in LDS once at
    // most those of the S - 2 later steps are outstanding; after the barrier everybody's are, and everybody
    // has step s in registers, so the loads of step s + S (past the last step: of it again, unread) may
    // fill its stage.
    auto step = [&](Frag &F, Frag &G, int s) {
        wait_lds_vmem<(S - 2) * kLoads>();
        __builtin_amdgcn_s_barrier();
        const int nx = st + 1 == S ? 0 : st + 1;
        read(G, nx);
        issue(min(s + S, KS - 1), st);
        st = nx;
        const float sw_next = FP4W ? 0.f : wsc[min(s + 1, KS - 1)];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                constexpr int bf = FP4W ? 4 : 0;
                const f32x4 c = CHAIN && FP4W ? acc[mt][nt] : f32x4{0.f, 0.f, 0.f, 0.f};
                const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(F.a[mt], F.b[nt], c, 0, bf, 0, F.sa[mt], 0, F.sb[nt]);
                if constexpr (CHAIN && FP4W) {
                    acc[mt][nt] = d;
                } else if constexpr (CHAIN) {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] = fmaf(sw, d[e], acc[mt][nt][e]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] += FP4W ? d[e] : fmaf(sw, d[e], 0.f);
                }
            }
        if (--left == 0 || s == KS - 1) {
            left = group;
#pragma unroll
            for (int i = 0; i < MT * NT; i++) {
                tot[i / NT][i % NT] += acc[i / NT][i % NT];
                acc[i / NT][i % NT] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        sw = sw_next;
    };
#pragma unroll
    for (int s = 0; s < S; s++) issue(min(s, KS - 1), s);
    Frag F, G;
    wait_lds_vmem<(S - 1) * kLoads>();
    __builtin_amdgcn_s_barrier();
    read(F, 0);
    for (int s = 0; s < KS; s += 2) {
        step(F, G, s);
        if (s + 1 < KS) step(G, F, s + 1);
    }
    // no load may still be writing LDS when the workgroup reuses it, or ends
    wait_lds_vmem<0>();
    __builtin_amdgcn_s_barrier();
    // 16 rows at a time through the wave's own LDS, so that stores write whole row segments
    const int mw = m0 + wm * WM, nw = n0 + wn * WN;
    const bool wide = (N & 7) == 0 && ((uintptr_t)y & 15) == 0;
    float *buf = (float *)smem + wave * (16 * (WN + 4));
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        if (!wide) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int n = nw + 16 * nt + r;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int m = mw + 16 * mt + 4 * g + e;
                    if (m >= M || n >= N) continue;
                    if (y_f32) ((float *)y)[(size_t)m * N + n] = tot[mt][nt][e];
                    else ((uint16_t *)y)[(size_t)m * N + n] = f32_to_bf16_bits(tot[mt][nt][e]);
                }
            }
            continue;
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int e = 0; e < 4; e++) buf[(4 * g + e) * (WN + 4) + 16 * nt + r] = tot[mt][nt][e];
        __builtin_amdgcn_wave_barrier();
        constexpr int kLanes = WN / 8;  // lanes per row segment, 8 values each
#pragma unroll
        for (int i = 0; i < 16 * kLanes / 64; i++) {
            const int row = (i * 64 + lane) / kLanes, col = (lane % kLanes) * 8;
            const int m = mw + 16 * mt + row, n = nw + col;
            const f32x4 v0 = *(const f32x4 *)(buf + row * (WN + 4) + col), v1 = *(const f32x4 *)(buf + row * (WN + 4) + col + 4);
            if (m >= M || n >= N) continue;
            if (y_f32) {
                *(f32x4 *)((float *)y + (size_t)m * N + n) = v0;
                *(f32x4 *)((float *)y + (size_t)m * N + n + 4) = v1;
            } else {
                u32x4 o;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float x = j < 2 ? v0[2 * j] : v1[2 * j - 4], z = j < 2 ? v0[2 * j + 1] : v1[2 * j - 3];
                    o[j] = (uint32_t)f32_to_bf16_bits(x) | (uint32_t)f32_to_bf16_bits(z) << 16;
                }
                *(u32x4 *)((uint16_t *)y + (size_t)m * N + n) = o;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// What k_gemm_tile reads besides the weight codes, one wave per piece: waves [0, na) take 16 rows x
// 128 K of the activations (QUANT: of bf16 x, quantized as k_act_quant_e4m3 does; else of codes and scale
// bytes already quantized) into operand order (k_act_quant_e4m3_ops) and their scales into as4 [step][m]
// dwords, byte g of which is K block 32 g's of the step; the others take the FP4 weights' scale bytes
// ws [n][K / 32], 64 columns x 16 steps each, into ws4 [step][n] the same way. A tile's operands are then
// contiguous kilobytes and its scales of a step contiguous dwords: reads of 16 rows x 64 or 8 rows x 128
// bytes run at half the L2 rate of contiguous ones (measured 23-33 against 44-53 bytes per clock and CU).
template <bool QUANT>
__global__ __launch_bounds__(256) void k_gemm_prep(const void *__restrict__ x, const uint8_t *__restrict__ as_, int m,
                                                   int k, int block, const uint8_t *__restrict__ ws, int n,
                                                   uint8_t *__restrict__ aq, uint32_t *__restrict__ as4,
                                                   uint32_t *__restrict__ ws4, int na, int nw) {
    const int ks = k >> 7, lane = threadIdx.x & 63;
    const int w = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w >= na) {
        const int u = w - na, cols = (n + 63) >> 6;
        if (u >= nw) return;
        const int c = (u % cols) * 64 + lane, s0 = (u / cols) * 16;
        if (c >= n) return;
        const uint8_t *p = ws + (size_t)c * (k >> 5) + 4 * s0;
        const bool al = ((uintptr_t)p & 3) == 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (s0 + i >= ks) break;
            const uint8_t *q = p + 4 * i;
            ws4[(size_t)(s0 + i) * n + c] = al ? *(const uint32_t *)q : q[0] | q[1] << 8 | q[2] << 16 | (uint32_t)q[3] << 24;
        }
        return;
    }
    const int mg = w / ks, s = w % ks, r = lane & 15, g = lane >> 4, row = mg * 16 + r;
    const bool ok = row < m;
    uint8_t *dst = aq + ops_block(mg, s, ks, false) + lane * 16;
    if constexpr (!QUANT) {
        const uint8_t *src = (const uint8_t *)x + (size_t)(ok ? row : 0) * k + (size_t)s * 128 + 16 * g;
#pragma unroll
        for (int h = 0; h < 2; h++) *(u32x4 *)(dst + 1024 * h) = *(const u32x4 *)(src + 64 * h);
        if (ok && block == 128 && g == 0) as4[(size_t)s * m + row] = as_[(size_t)row * ks + s] * 0x01010101u;
        if (ok && block == 32) ((uint8_t *)as4)[((size_t)s * m + row) * 4 + g] = as_[(size_t)row * (k >> 5) + 4 * s + g];
        return;
    } else {
        u32x4 q[2];
        uint32_t sb[2];
        quant_ops((const uint16_t *)x + (size_t)(ok ? row : 0) * k + (size_t)s * 128 + 16 * g, block, q, sb);
#pragma unroll
        for (int h = 0; h < 2; h++) *(u32x4 *)(dst + 1024 * h) = q[h];
        // lane pair (g, g ^ 1) of half h holds the scale of the step's block 2 h + g / 2
        if (ok && block == 128 && g == 0) as4[(size_t)s * m + row] = sb[0] * 0x01010101u;
        if (ok && block == 32 && (g & 1) == 0) {
            uint8_t *d = (uint8_t *)(as4 + (size_t)s * m + row) + (g >> 1);
            d[0] = (uint8_t)sb[0], d[2] = (uint8_t)sb[1];
        }
    }
}

// GEMM of any number of rows in one launch, for calls whose tiles do not fill the GPU twice: a workgroup
// owns a 16 MT x 16 NT output tile over all of K; wave w takes the groups w, w + NW, ... of `group` steps
// each, loads its operands straight from global memory one step ahead of their products, and the groups'
// sums are added in order through LDS, NW groups at a time. The waves of a tile need no barrier but the
// sum's and no partial tiles in memory. The order of the sum is gemm_plan's, as in k_gemm_tile; chained
// groups (a multiple of 4 steps, 4- and 16-byte aligned scales) load their scales four steps at once.
// q form, FP4, against 64 rows a launch, us: 100 x 2048 x 7168 15.9 -> 11.3, 200 x 512 x 7168 38.6 -> 14.8,
// 700 x 512 x 4096 100.9 -> 19.3 (2 x 4 tiles); against split K and its second launch: 64 x 4096 x 2176
// 10.4 -> 5.9, 16 x 256 x 512 7.3 -> 3.2, 8 x 7168 x 2048 11.5 -> 6.5.
template <bool FP4W, int MT, int NT, bool CHAIN, bool AARR, bool WOPS>
__global__ __launch_bounds__(512) void k_gemm_waves(const uint8_t *__restrict__ wc, const void *__restrict__ ws,
                                                        const uint8_t *__restrict__ aq, const uint8_t *__restrict__ as_,
                                                        void *__restrict__ y, int y_f32, int M, int N, int K, int act32,
                                                        int group, int mtiles, int ntiles) {
    constexpr int NW = 8, kTileVecs = MT * NT * 64, kThreads = NW * 64, kPer = (kTileVecs + kThreads - 1) / kThreads;
    __shared__ f32x4 red[NW * kTileVecs];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = K >> 7;
    const bool odd = r & 1;
    const int h0 = odd ? 64 : 0, h1 = 64 - h0;
    const int total = mtiles * ntiles, xcd = blockIdx.x & 7, per = total >> 3, rem = total & 7;
    const int t0 = xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int m0 = (t0 % mtiles) * 16 * MT, n0 = (t0 / mtiles) * 16 * NT;
    const uint8_t *pa = aq + (AARR ? ((size_t)(m0 >> 4) * KS * 2) * 1024 : (size_t)m0 * K);
    const uint8_t *pb = wc + (WOPS ? ops_block(n0 >> 4, 0, KS, FP4W) : (size_t)n0 * (FP4W ? K >> 1 : K));
    uint32_t oa[MT], ob[NT], osa[MT], osb[NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int row = min(m0 + 16 * mt + r, M - 1) - m0;
        if (AARR) oa[mt] = (uint32_t)ops_block(operand_group(m0, mt, M) - (m0 >> 4), 0, KS, false) + lane * 16;
        else oa[mt] = (uint32_t)row * (uint32_t)K + 16 * g;
        osa[mt] = (uint32_t)row * (uint32_t)(act32 ? K >> 5 : KS);
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int col = min(n0 + 16 * nt + r, N - 1) - n0;
        if (WOPS) ob[nt] = (uint32_t)ops_block(min((n0 >> 4) + nt, (N >> 4) - 1) - (n0 >> 4), 0, KS, FP4W) + lane * 16;
        else ob[nt] = (uint32_t)col * (uint32_t)(FP4W ? K >> 1 : K) + 16 * g;
        osb[nt] = (uint32_t)col * (uint32_t)(K >> 5);
    }
    const uint8_t *psa = as_ + (size_t)m0 * (act32 ? K >> 5 : KS);
    const uint8_t *psb = (const uint8_t *)ws + (FP4W ? (size_t)n0 * (K >> 5) : 0);
    const float *wsc = (const float *)ws + (size_t)(n0 >> 7) * KS;

    struct Step {
        u32x4 a[MT][2], b[NT][FP4W ? 1 : 2];
        uint32_t sa[MT], sb[NT];
        float sw;
    };
    auto load = [&](Step &S, int s) {
        const size_t ka = AARR ? (size_t)s * 2048 : (size_t)s * 128;
        const size_t kb = WOPS ? (size_t)s * (FP4W ? 1024 : 2048) : (size_t)s * (FP4W ? 64 : 128);
        if constexpr (!CHAIN) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) S.sa[mt] = psa[osa[mt] + (act32 ? 4 * s + g : s)];
            if constexpr (FP4W) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++) S.sb[nt] = psb[osb[nt] + 4 * s + g];
            }
        }
        if constexpr (!FP4W) S.sw = wsc[s];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const uint8_t *p = pb + ob[nt] + kb;
            if constexpr (FP4W) {
                S.b[nt][0] = *(const u32x4 *)p;
            } else if constexpr (WOPS) {
                S.b[nt][0] = *(const u32x4 *)p;
                S.b[nt][1] = *(const u32x4 *)(p + 1024);
            } else {
                S.b[nt][0] = *(const u32x4 *)(p + h0);
                S.b[nt][1] = *(const u32x4 *)(p + h1);
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint8_t *p = pa + oa[mt] + ka;
            S.a[mt][0] = *(const u32x4 *)(p + (AARR ? 0 : h0));
            S.a[mt][1] = *(const u32x4 *)(p + (AARR ? 1024 : h1));
        }
    };
    f32x4 acc[MT][NT], tot[kPer];
    auto compute = [&](const Step &S, const uint32_t (&sa)[MT], const uint32_t (&sb)[NT]) {
        i32x8 b[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const u32x4 y0 = S.b[nt][0];
            if constexpr (FP4W) {
                b[nt] = i32x8{(int)y0[0], (int)y0[1], (int)y0[2], (int)y0[3], 0, 0, 0, 0};
            } else {
                const u32x4 y1 = S.b[nt][1];
                const bool swp = odd && !WOPS;
                const u32x4 x0 = swp ? y1 : y0, x1 = swp ? y0 : y1;
                b[nt] = i32x8{(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const bool swp = odd && !AARR;
            const u32x4 x0 = swp ? S.a[mt][1] : S.a[mt][0], x1 = swp ? S.a[mt][0] : S.a[mt][1];
            const i32x8 a = {(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                constexpr int bf = FP4W ? 4 : 0;
                const f32x4 c = CHAIN && FP4W ? acc[mt][nt] : f32x4{0.f, 0.f, 0.f, 0.f};
                const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[nt], c, 0, bf, 0, (int)sa[mt], 0,
                                                                                 FP4W ? (int)sb[nt] : 127);
                if constexpr (CHAIN && FP4W) {
                    acc[mt][nt] = d;
                } else if constexpr (CHAIN) {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] = fmaf(S.sw, d[e], acc[mt][nt][e]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] += FP4W ? d[e] : fmaf(S.sw, d[e], 0.f);
                }
            }
        }
    };
#pragma unroll
    for (int j = 0; j < kPer; j++) tot[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int groups = (KS + group - 1) / group;
    for (int base = 0; base < groups; base += NW) {
        const int gi = base + wave;
        if (gi < groups) {
            const int s0 = gi * group, n = min(group, KS - s0);
#pragma unroll
            for (int i = 0; i < MT * NT; i++) acc[i / NT][i % NT] = f32x4{0.f, 0.f, 0.f, 0.f};
            Step S[2];
            if constexpr (CHAIN) {  // n is a multiple of 4, and scale words of 4 steps are aligned
                const int gsh = 8 * g;
                load(S[0], s0);
                for (int u = 0; u < n; u += 4) {
                    u32x4 asw[MT], bsw[NT];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        if (act32) asw[mt] = *(const u32x4 *)(psa + osa[mt] + 4 * (s0 + u));
                        else asw[mt][0] = *(const uint32_t *)(psa + osa[mt] + s0 + u);
                    }
                    if constexpr (FP4W) {
#pragma unroll
                        for (int nt = 0; nt < NT; nt++) bsw[nt] = *(const u32x4 *)(psb + osb[nt] + 4 * (s0 + u));
                    }
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        load(S[(q + 1) & 1], min(s0 + u + q + 1, s0 + n - 1));
                        __builtin_amdgcn_sched_barrier(0);
                        uint32_t sa[MT], sb[NT];
#pragma unroll
                        for (int mt = 0; mt < MT; mt++) sa[mt] = act32 ? asw[mt][q] >> gsh : asw[mt][0] >> (8 * q);
#pragma unroll
                        for (int nt = 0; nt < NT; nt++) sb[nt] = FP4W ? bsw[nt][q] >> gsh : 0;
                        compute(S[q & 1], sa, sb);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            } else {
                load(S[0], s0);
                for (int u = 0; u < n; u += 2) {
                    load(S[1], min(s0 + u + 1, s0 + n - 1));
                    __builtin_amdgcn_sched_barrier(0);
                    compute(S[0], S[0].sa, S[0].sb);
                    __builtin_amdgcn_sched_barrier(0);
                    if (u + 1 < n) {
                        load(S[0], min(s0 + u + 2, s0 + n - 1));
                        __builtin_amdgcn_sched_barrier(0);
                        compute(S[1], S[1].sa, S[1].sb);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        if (base > 0) __syncthreads();
        if (gi < groups) {
#pragma unroll
            for (int t = 0; t < MT * NT; t++) red[(wave * MT * NT + t) * 64 + lane] = acc[t / NT][t % NT];
        }
        __syncthreads();
        const int live = min(NW, groups - base);
#pragma unroll
        for (int j = 0; j < kPer; j++)
            if (kTileVecs % kThreads == 0 || tid + kThreads * j < kTileVecs)
                for (int w = 0; w < live; w++) tot[j] += red[w * kTileVecs + tid + kThreads * j];
    }
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int q = tid + kThreads * j, t = q >> 6, ql = q & 63, mt = t / NT, nt = t % NT;
        const int n = n0 + 16 * nt + (ql & 15);
        if (n >= N || q >= kTileVecs) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + 16 * mt + 4 * (ql >> 4) + e;
            if (m >= M) continue;
            if (y_f32) ((float *)y)[(size_t)m * N + n] = tot[j][e];
            else ((uint16_t *)y)[(size_t)m * N + n] = f32_to_bf16_bits(tot[j][e]);
        }
    }
}

// One GEMM call on quantized activations; arr: aq is in operand order (not for kSplit).
struct GemmArgs {
    int fmt;
    bool wops, arr;  // weights / activations in operand order
    void *y;
    const uint8_t *codes;
    const void *scales;
    const uint8_t *aq, *as_;
    int m, n, k, act_block, y_f32;
    hipStream_t st;
};

template <bool FP4W, bool WOPS>
static hipError_t launch_split(const GemmPlan &p, const GemmArgs &c, void *work) {
    const int tiles = ceil_div(c.n, 64);
    f32x4 *part = (f32x4 *)work;
    hipLaunchKernelGGL((k_gemm<FP4W, WOPS>), dim3(tiles * p.slices), dim3(512), 0, c.st, c.codes, c.scales, c.aq,
                       c.as_, part, c.m, c.n, c.k, c.act_block == 32 ? 5 : 7, tiles, p.slices, p.group);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_gemm_reduce, dim3(tiles * (4 * 4 * 64) / 256), dim3(256), 0, c.st, part, p.slices, tiles, c.y,
                       c.y_f32, c.m, c.n);
    return hipGetLastError();
}

template <bool FP4W, int MT, int NT, int NW, int QW, bool ARR, bool WOPS>
static hipError_t launch_one(const GemmArgs &c) {
    const int tiles = ceil_div(c.n, 16 * NT);
    hipLaunchKernelGGL((k_gemm_one<FP4W, MT, NT, NW, QW, ARR, WOPS>), dim3(tiles * ceil_div(c.m, 16 * MT)), dim3(NW * 64), 0,
                       c.st, c.codes, c.scales, c.aq, c.as_, c.y, c.y_f32, c.m, c.n, c.k, c.act_block == 32, tiles);
    return hipGetLastError();
}

template <bool FP4W, int MT, int NT, bool ARR, bool WOPS>
static hipError_t launch_waves(const GemmPlan &p, const GemmArgs &c) {
    const int mt = ceil_div(c.m, 16 * MT), nt = ceil_div(c.n, 16 * NT);
#define STBL_WAVES(CHAIN)                                                                                             \
    hipLaunchKernelGGL((k_gemm_waves<FP4W, MT, NT, CHAIN, ARR, WOPS>), dim3((unsigned)mt * nt), dim3(512), 0, c.st,    \
                       c.codes, c.scales, c.aq, c.as_, c.y, c.y_f32, c.m, c.n, c.k, c.act_block == 32, p.group, mt, nt)
    if (p.chain) STBL_WAVES(true);
    else STBL_WAVES(false);
#undef STBL_WAVES
    return hipGetLastError();
}

template <bool FP4W, bool ARR, bool WOPS>
static hipError_t launch_direct(const GemmPlan &p, const GemmArgs &c) {
    if (p.kernel == kOne64) return launch_one<FP4W, tile_rows(kOne64) / 16, 4, 4, 1, ARR, WOPS>(c);
    if (p.kernel == kOne32) return launch_one<FP4W, tile_rows(kOne32) / 16, 2, FP4W ? 8 : 16, FP4W ? 2 : 1, ARR, WOPS>(c);
    if (p.kernel == kWaves24) return launch_waves<FP4W, tile_rows(kWaves24) / 16, 4, ARR, WOPS>(p, c);
    return launch_waves<FP4W, tile_rows(kWaves22) / 16, 2, ARR, WOPS>(p, c);
}

template <bool FP4W, int BN, int WC, int S, bool WOPS>
static hipError_t launch_tile(const GemmPlan &p, const GemmArgs &c, const uint8_t *as4, const uint8_t *ws4) {
    constexpr int BM = tile_rows(kTile64), lds = S * (BM * 128 + BN * (FP4W ? 64 : 128) + BM * 4 + (FP4W ? BN * 4 : 0));
    const int mt = ceil_div(c.m, BM), nt = ceil_div(c.n, BN);
#define STBL_TILE(CHAIN)                                                                                              \
    hipLaunchKernelGGL((k_gemm_tile<FP4W, BM, BN, 2, WC, S, CHAIN, WOPS>), dim3((unsigned)mt * nt), dim3(2 * WC * 64),   \
                       lds, c.st, c.codes, c.scales, c.aq, as4, ws4, c.y, c.y_f32, c.m, c.n, c.k, p.group, mt, nt)
    if (p.chain) STBL_TILE(true);
    else STBL_TILE(false);
#undef STBL_TILE
    return hipGetLastError();
}

template <bool FP4W, bool WOPS>
static hipError_t launch_fmt(const GemmPlan &p, const GemmArgs &c, void *work, const uint8_t *as4, const uint8_t *ws4) {
    if (p.kernel == kTile64) return launch_tile<FP4W, 64, 2, 4, WOPS>(p, c, as4, ws4);
    if (p.kernel == kTile128) return launch_tile<FP4W, 128, 4, 3, WOPS>(p, c, as4, ws4);
    if (p.kernel == kSplit) return launch_split<FP4W, WOPS>(p, c, work);
    return c.arr ? launch_direct<FP4W, true, WOPS>(p, c) : launch_direct<FP4W, false, WOPS>(p, c);
}

static hipError_t launch_gemm(const GemmPlan &p, const GemmArgs &c, void *work, const uint8_t *as4 = nullptr,
                              const uint8_t *ws4 = nullptr) {
    if (c.fmt == 0) return c.wops ? launch_fmt<true, true>(p, c, work, as4, ws4) : launch_fmt<true, false>(p, c, work, as4, ws4);
    return c.wops ? launch_fmt<false, true>(p, c, work, as4, ws4) : launch_fmt<false, false>(p, c, work, as4, ws4);
}

static int check_gemm(const char *name, int fmt, const void *y, const void *codes, const void *scales, int m, int max_m,
                      int n, int k, int act_block, const void *work, bool wops) {
    if (fmt != 0 && fmt != 1) return abi_fail(hipErrorInvalidValue, "%s: unknown format %d", name, fmt);
    if (!y || !codes || !scales || !work) return abi_fail(hipErrorInvalidValue, "%s: null pointer", name);
    if (m < 1 || m > max_m || n < 1 || n > kGemmMaxN || k < 128 || k % 128 || (act_block != 32 && act_block != 128))
        return abi_fail(hipErrorInvalidValue,
                        "%s: need 1 <= m <= %d, n <= %d, k %% 128 == 0, act_block 32 or 128 (m=%d n=%d k=%d)", name,
                        max_m, kGemmMaxN, m, n, k);
    if (!aligned16(codes) || !aligned16(work)) return abi_fail(hipErrorInvalidValue, "%s: codes and work must be 16-byte aligned", name);
    if (wops && n % 16) return abi_fail(hipErrorInvalidValue, "%s: packed weights need n %% 16 == 0 (n=%d)", name, n);
    return 0;
}

// Activations prepared into `work` as the plan's kernel reads them, then the GEMM. x: bf16, or (quantized) e4m3
// codes with their scale bytes as_.
static hipError_t gemm_prepared(GemmPlan p, GemmArgs c, const void *x, bool quantized, uint8_t *aq, uint8_t *as, uint8_t *ws4,
                                void *work) {
    const int ks = c.k / 128, na = ceil_div(c.m, 16) * ks;
    if (is_tile(p)) {
        const int nw = c.fmt == 0 ? ceil_div(c.n, 64) * ceil_div(ks, 16) : 0;
        const dim3 grid(ceil_div(na + nw, 4));
        if (quantized)
            hipLaunchKernelGGL(k_gemm_prep<false>, grid, dim3(256), 0, c.st, x, c.as_, c.m, c.k, c.act_block,
                               (const uint8_t *)c.scales, c.n, aq, (uint32_t *)as, (uint32_t *)ws4, na, nw);
        else
            hipLaunchKernelGGL(k_gemm_prep<true>, grid, dim3(256), 0, c.st, x, (const uint8_t *)nullptr, c.m, c.k,
                               c.act_block, (const uint8_t *)c.scales, c.n, aq, (uint32_t *)as, (uint32_t *)ws4, na, nw);
        c.arr = true;
    } else if (quantized) {
        return launch_gemm(p, c, work);  // read in place
    } else if (p.kernel == kSplit) {
        const int n8 = c.m * c.k / 8;
        hipLaunchKernelGGL(k_act_quant_e4m3, dim3(ceil_div(n8, 256)), dim3(256), 0, c.st, (const uint16_t *)x, n8, c.act_block,
                           aq, as);
    } else {
        // operand order: one contiguous kilobyte per load instead of 16 rows x 64 bytes
        hipLaunchKernelGGL(k_act_quant_e4m3_ops, dim3(na), dim3(64), 0, c.st, (const uint16_t *)x, c.m, c.k, c.act_block, aq, as);
        c.arr = true;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    c.aq = aq, c.as_ = as;
    return launch_gemm(p, c, work, as, ws4);
}

static int gemm_any(const char *name, int max_m, bool wops, int fmt, void *y, const void *codes, const void *scales,
                    const void *x, const void *as, bool quantized, int m, int n, int k, int act_block, int y_f32, void *work,
                    hipStream_t st) {
    if (int e = check_gemm(name, fmt, y, codes, scales, m, max_m, n, k, act_block, work, wops)) return e;
    if (quantized && (!x || !as || !aligned16(x))) return abi_fail(hipErrorInvalidValue, "%s: aq (16-byte aligned) and as needed", name);
    if (!quantized && (!x || !aligned16(x))) return abi_fail(hipErrorInvalidValue, "%s: x must be 16-byte aligned", name);
    const bool aligned = (!quantized || aligned16(as)) && (fmt != 0 || aligned16(scales));
    const GemmPlan p = gemm_plan(fmt, m, n, k, aligned);
    uint8_t *aq = (uint8_t *)work + (m <= kGemmMaxM ? part_reserve(n, k) : 0), *as_ = aq + aq_bytes(m, k);
    uint8_t *ws4 = as_ + a256((uint64_t)m * (k / 32));
    const GemmArgs c = {fmt, wops, false, y, (const uint8_t *)codes, scales, (const uint8_t *)x, (const uint8_t *)as,
                        m, n, k, act_block, y_f32, st};
    return abi_status(gemm_prepared(p, c, x, quantized, aq, as_, ws4, work), name);
}

}  // namespace stbl

using namespace stbl;

extern "C" {

uint64_t stbl_amd_gemm_work_bytes(int m, int n, int k) { return gemm_work_bytes(m, n, k); }

int stbl_amd_gemm_q(int fmt, void *y, const void *codes, const void *scales, const void *aq, const void *as, int m,
                    int n, int k, int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm_q", kGemmMaxM, false, fmt, y, codes, scales, aq, as, true, m, n, k, act_block, y_f32, work, st);
}

int stbl_amd_gemm(int fmt, void *y, const void *codes, const void *scales, const void *x, int m, int n, int k,
                  int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm", kGemmMaxM, false, fmt, y, codes, scales, x, nullptr, false, m, n, k, act_block, y_f32, work, st);
}

int stbl_amd_gemm_pack(int fmt, void *packed, const void *codes, int n, int k, hipStream_t st) {
    if (fmt != 0 && fmt != 1) return abi_fail(hipErrorInvalidValue, "gemm_pack: unknown format %d", fmt);
    if (!packed || !codes || n < 16 || n % 16 || n > kGemmMaxN || k < 128 || k % 128)
        return abi_fail(hipErrorInvalidValue, "gemm_pack: need n %% 16 == 0 and k %% 128 == 0 (n=%d k=%d)", n, k);
    if (!aligned16(packed) || !aligned16(codes) || packed == codes)
        return abi_fail(hipErrorInvalidValue, "gemm_pack: codes and packed must be distinct 16-byte aligned buffers");
    const size_t pieces = (size_t)n * k / (fmt == 0 ? 32 : 16);
    hipLaunchKernelGGL(k_gemm_pack, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st, (const uint8_t *)codes,
                       (uint8_t *)packed, n, k, fmt == 0 ? 1 : 0, pieces);
    return abi_status(hipGetLastError(), "gemm_pack launch");
}

int stbl_amd_gemm_q_packed(int fmt, void *y, const void *packed, const void *scales, const void *aq, const void *as,
                           int m, int n, int k, int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm_q_packed", kGemmMaxM, true, fmt, y, packed, scales, aq, as, true, m, n, k, act_block, y_f32, work, st);
}

int stbl_amd_gemm_packed(int fmt, void *y, const void *packed, const void *scales, const void *x, int m, int n, int k,
                         int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm_packed", kGemmMaxM, true, fmt, y, packed, scales, x, nullptr, false, m, n, k, act_block, y_f32, work,
                    st);
}

int stbl_amd_gemm_rows(int fmt, int packed, void *y, const void *codes, const void *scales, const void *x, int m, int n,
                       int k, int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm_rows", kGemmMaxRows, packed != 0, fmt, y, codes, scales, x, nullptr, false, m, n, k, act_block, y_f32,
                    work, st);
}

int stbl_amd_gemm_q_rows(int fmt, int packed, void *y, const void *codes, const void *scales, const void *aq, const void *as,
                         int m, int n, int k, int act_block, int y_f32, void *work, hipStream_t st) {
    return gemm_any("gemm_q_rows", kGemmMaxRows, packed != 0, fmt, y, codes, scales, aq, as, true, m, n, k, act_block, y_f32,
                    work, st);
}

// act_quant(x, block, "ue8m0") of ref/kernel.py:35-45 with the codes and E8M0 scale bytes it feeds
// the GEMM: x bf16 [rows][k] -> codes [rows][k], scales [rows][k / block]. k % block == 0.
int stbl_amd_act_quant_e4m3(const void *x, int rows, int k, int block, void *codes, void *scales, hipStream_t st) {
    if (!x || !codes || !scales || rows < 1 || (block != 32 && block != 128) || k % block)
        return abi_fail(hipErrorInvalidValue, "act_quant_e4m3: need block 32 or 128 and k %% block == 0");
    if (!aligned16(x) || ((uintptr_t)codes & 7)) return abi_fail(hipErrorInvalidValue, "act_quant_e4m3: x 16-byte, codes 8-byte aligned");
    const int n8 = rows * k / 8;
    hipLaunchKernelGGL(k_act_quant_e4m3, dim3((n8 + 255) / 256), dim3(256), 0, st, (const uint16_t *)x, n8, block,
                       (uint8_t *)codes, (uint8_t *)scales);
    return abi_status(hipGetLastError(), "act_quant_e4m3 launch");
}

}  // extern "C"
