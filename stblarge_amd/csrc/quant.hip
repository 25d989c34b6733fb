// Quantizers, dequantizers and the elementwise epilogues of the expert-GEMV path.
//
//   act_quant          ref/kernel.py:35-45 (v2, bf16 in, codes + scales out) and the reference
//                      engine's in-place fp32 form stbl/kernels.cu:54-63 (stbl_act_quant_fp8).
//   weight quantizers  FP4: fp4_act_quant's E8M0 path, ref/kernel.py:55-72, on weight rows.
//                      FP8: one fp32 scale per 128x128 block, s = max(amax, 1e-4) / 448.
//   dequantizers       one fp32 product per element, ref/kernel.py:89-90 and :98-101.
//   epilogues          round_bf16 / swiglu / axpy, stbl/kernels.cu:86-89, :444-464.
// All are bound by their bytes; the quantizers read each value once, in 16-byte loads.
#include "common.hpp"
#include "abi_util.hpp"
#include "expert_layout.hpp"

namespace stbl {

// ---- activation quantization ---------------------------------------------------------------------

// 1/s for a power of two s below 2^127, exact; 0 for s = +Inf (a block holding an infinity), where v *
// 0 is v / s: a signed zero for a finite v, NaN for an infinite one.
__device__ __forceinline__ float pow2_inverse(float s) {
    return __builtin_isinf(s) ? 0.f : __uint_as_float((254u - ((__float_as_uint(s) >> 23) & 0xffu)) << 23);
}

// Four values, clamped to +-448 (a NaN to -448), as e4m3 codes; the rounding is the hardware's round to
// nearest even, which equals f32_to_e4m3.
__device__ __forceinline__ uint32_t e4m3x4_sat(float a, float b, float c, float d) {
    auto clamp = [](float v) { return fminf(fmaxf(v, -448.f), 448.f); };
    int p = __builtin_amdgcn_cvt_pk_fp8_f32(clamp(a), clamp(b), 0, false);
    p = __builtin_amdgcn_cvt_pk_fp8_f32(clamp(c), clamp(d), p, true);
    return (uint32_t)p;
}

// The reference engine's form: per 32 values in place, s = pow2_ceil(max(amax, 1e-4) * (1/448)),
// x = bf16(e4m3(clamp(x / s, +-448)) * s). One 32-lane half-wave per block of 32.
// The block's amax comes from its 32 lanes (half a wave) by four DPP moves and one lane shuffle
// (instead of five shuffles, each an LDS round trip); x / s is x times the exact inverse of the power of two s; the e4m3 rounding is the
// hardware v_cvt_pk_fp8_f32 (round to nearest even, equal to the software encoder f32_to_e4m3 on
// fp32 inputs), and e4m3 * s is exact.
__device__ __forceinline__ float dpp_max(float a, int ctrl_sel) {
    int m;
    switch (ctrl_sel) {  // compile-time after inlining
        case 0: m = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0xB1, 0xF, 0xF, false); break;   // lane ^ 1
        case 1: m = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x4E, 0xF, 0xF, false); break;   // lane ^ 2
        case 2: m = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x141, 0xF, 0xF, false); break;  // 7 - lane in 8
        default: m = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x140, 0xF, 0xF, false); break; // 15 - lane in 16
    }
    return fmaxf(a, __builtin_bit_cast(float, m));
}

__global__ void k_act_quant_fp8_inplace(float *x, int n_blocks) {
    const int b = (blockIdx.x * blockDim.x + threadIdx.x) >> 5;
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) & 31;
    const bool ok = b < n_blocks;
    const float v = ok ? x[(size_t)b * 32 + i] : 0.f;
    float a = fabsf(v);
    a = dpp_max(a, 0);
    a = dpp_max(a, 1);
    a = dpp_max(a, 2);
    a = dpp_max(a, 3);
    a = fmaxf(a, __shfl_xor(a, 16, kWave));  // lanes l and l ^ 16
    const float s = pow2_ceil(fmaxf(a, 1e-4f) * (1.0f / 448.0f));
    const float inv = pow2_inverse(s);
    if (ok) {
        const float q = fminf(fmaxf(v * inv, -448.f), 448.f);
        const uint32_t c = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(q, q, 0, false) & 0xffu;
        x[(size_t)b * 32 + i] = bf16_round(e4m3_to_f32(c) * s);
    }
}

// The maximum over the aligned group of `lanes` (1, 2, 4, ... 64, uniform) that a lane belongs to.
__device__ __forceinline__ float group_max(float a, int lanes) {
    if (lanes > 1) a = dpp_max(a, 0);
    if (lanes > 2) a = dpp_max(a, 1);
    if (lanes > 4) a = dpp_max(a, 2);
    if (lanes > 8) a = dpp_max(a, 3);
    if (lanes > 16) a = fmaxf(a, __shfl_xor(a, 16, kWave));
    if (lanes > 32) a = fmaxf(a, __shfl_xor(a, 32, kWave));
    return a;
}

// ref/kernel.py:35-45 on bf16 rows. codes [rows][n] e4m3, scales [rows][n/block] fp32, and the
// dequantized bf16 values bf16(e4m3 * s), each optional. Bound by its bytes (2 read, 1 to 3 written per
// value): each lane holds 8 consecutive values, read once as 16 bytes, and the block's `lanes` = block /
// 8 lanes share its maximum, so a wave's loads and stores are contiguous runs. 512 x 7168, block 128:
// 62.3 us with one thread walking each block twice, value by value; 4.0 us (2.8 TB/s) so.
template <bool POW2>
__global__ __launch_bounds__(256) void k_act_quant8(const uint16_t *x, int n8, int lanes, uint8_t *codes,
                                                    float *scales, uint16_t *deq) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool ok = i < n8;  // n8 is a multiple of lanes: a block's lanes are all in or all out
    const u32x4 v = *(const u32x4 *)(x + (size_t)(ok ? i : 0) * 8);
    float f[8];
#pragma unroll
    for (int j = 0; j < 4; j++) f[2 * j] = bf16_lo(v[j]), f[2 * j + 1] = bf16_hi(v[j]);
    float a = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) a = fmaxf(a, fabsf(f[j]));
    const float t = fmaxf(group_max(a, lanes), 1e-4f) * (float)(1.0 / 448.0);
    const float s = POW2 ? pow2_ceil(t) : t;
    // x times the exact inverse of a power of two is x / s
    const float inv = POW2 ? pow2_inverse(s) : 0.f;
    float q[8];
#pragma unroll
    for (int j = 0; j < 8; j++) q[j] = POW2 ? f[j] * inv : __fdiv_rn(f[j], s);
    const u32x2 c = {e4m3x4_sat(q[0], q[1], q[2], q[3]), e4m3x4_sat(q[4], q[5], q[6], q[7])};
    if (!ok) return;
    if (scales && (threadIdx.x & (lanes - 1)) == 0) scales[i / lanes] = s;
    if (codes) *(u32x2 *)(codes + (size_t)i * 8) = c;
    if (deq) {
        u32x4 d;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const f32x2 e = e4m3x2(c[j >> 1], j & 1);
            d[j] = (uint32_t)f32_to_bf16_bits(e.x * s) | (uint32_t)f32_to_bf16_bits(e.y * s) << 16;
        }
        *(u32x4 *)(deq + (size_t)i * 8) = d;
    }
}

// The same for any block length and alignment: one thread per block of `block` values.
__global__ void k_act_quant(const uint16_t *x, int n_blocks, int block, int pow2, uint8_t *codes, float *scales,
                            uint16_t *deq) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n_blocks) return;
    const uint16_t *xb = x + (size_t)b * block;
    float amax = 0.f;
    for (int i = 0; i < block; i++) amax = fmaxf(amax, fabsf(bf16_bits_to_f32(xb[i])));
    const float t = fmaxf(amax, 1e-4f) * (float)(1.0 / 448.0);
    const float s = pow2 ? pow2_ceil(t) : t;
    if (scales) scales[b] = s;
    for (int i = 0; i < block; i++) {
        const float q = fminf(fmaxf(__fdiv_rn(bf16_bits_to_f32(xb[i]), s), -448.f), 448.f);
        const uint32_t c = f32_to_e4m3(q);
        if (codes) codes[(size_t)b * block + i] = (uint8_t)c;
        if (deq) deq[(size_t)b * block + i] = f32_to_bf16_bits(e4m3_to_f32(c) * s);
    }
}

// ---- weight quantizers ---------------------------------------------------------------------------

// The matrices of one launch: a matrix on its own, or the three of an expert, whose launch then fills
// the GPU to the end once instead of three times (quantizing a 7168 x 2048 expert into its slot: three FP8
// launches and six copies of their outputs 69.1 us, one launch 37.7).
struct QuantJob {
    const float *w;
    uint8_t *codes;
    void *scales;
    int rows, k;
    uint32_t first;  // the matrix's first workgroup; past every workgroup for an unused entry
};
struct QuantJobs {
    QuantJob j[3];
};

// This workgroup's matrix, and its index among the matrix's workgroups in `b`.
__device__ __forceinline__ const QuantJob &quant_job(const QuantJobs &jobs, uint32_t &b) {
    const int m = (blockIdx.x >= jobs.j[1].first) + (blockIdx.x >= jobs.j[2].first);
    b = blockIdx.x - jobs.j[m].first;
    return jobs.j[m];
}

// FP4 e2m1 with E8M0 scales per 32 along K. Four lanes per group of 32, 8 values (two 16-byte loads)
// each, two groups per lane: a wave reads 2 KB and writes 256 bytes of codes (element 2i in the low
// nibble) in contiguous runs, and a group's maximum comes over two DPP moves. s is a power of two, so w
// times its exact inverse is w / s. Bound by its bytes: 7168 x 2048 23.3 us with one thread per group
// (128 bytes apart, so each load of a wave touched 64 lines), 20.5 with 16 consecutive values a lane,
// 16.6 with 4, 15.8 with 8 rounded in software, 14.2 (4.7 TB/s) so.
__global__ __launch_bounds__(256) void k_quant_fp4(QuantJobs jobs) {
    uint32_t wg;
    const QuantJob &J = quant_job(jobs, wg);
    const size_t n8 = (size_t)J.rows * (J.k >> 3);  // a multiple of 4: a group's lanes are all in or all out
    const size_t i0 = (size_t)wg * 512 + threadIdx.x;
    f32x4 v[2][2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const f32x4 *src = (const f32x4 *)J.w + 2 * (i0 + 256 * q < n8 ? i0 + 256 * q : 0);
        v[q][0] = __builtin_nontemporal_load(src);
        v[q][1] = __builtin_nontemporal_load(src + 1);
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const size_t i = i0 + 256 * q;
        float amax = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(v[q][j >> 2][j & 3]));
        amax = fmaxf(group_max(amax, 4), 6.0f * 0x1p-126f);
        const float s = pow2_ceil(amax * (float)(1.0 / 6.0));
        const float inv = pow2_inverse(s);
        // v_cvt_scalef32_pk_fp4_f32 at scale 1 rounds to nearest, ties to the even code, as ref/kernel.py:48-52
        // does (8 instead of about 140 VALU operations a lane)
        auto at = [&](int j) { return fminf(fmaxf(v[q][j >> 2][j & 3] * inv, -6.f), 6.f); };
        uint32_t out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0, at(0), at(1), 1.0f, 0);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, at(2), at(3), 1.0f, 1);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, at(4), at(5), 1.0f, 2);
        out = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(out, at(6), at(7), 1.0f, 3);
        if (i >= n8) return;
        *(uint32_t *)(J.codes + i * 4) = out;
        if ((threadIdx.x & 3) == 0) ((uint8_t *)J.scales)[i >> 2] = (uint8_t)((__float_as_uint(s) >> 23) & 0xffu);
    }
}

// FP8 e4m3 with one fp32 scale per 128x128 block (partial blocks at the edges): s = amax / 448 and
// e4m3(clamp(w / s)), both true fp32 divisions. One workgroup of 512 threads per block, each holding 8
// rows x 4 columns of it in registers: the block is read once, in 16-byte loads that are all in flight
// together (rows and columns past the edge reload the last ones, which changes no maximum). k % 4 == 0,
// w 16-byte and codes 4-byte aligned. 7168 x 2048: 73.9 us with two scalar passes over the block by 256
// threads, 16.1 us (4.6 TB/s) so.
__global__ __launch_bounds__(512) void k_quant_fp8_b128_x4(QuantJobs jobs) {
    __shared__ float red[8];
    uint32_t wg;
    const QuantJob &J = quant_job(jobs, wg);
    const int rows = J.rows, k = J.k, kb = (k + 127) >> 7, bi = (int)(wg / kb), bj = (int)(wg % kb);
    const int r0 = bi * 128 + (threadIdx.x >> 5), c0 = bj * 128 + (threadIdx.x & 31) * 4, c = min(c0, k - 4);
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; i++)
        v[i] = __builtin_nontemporal_load((const f32x4 *)(J.w + (size_t)min(r0 + 16 * i, rows - 1) * k + c));
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) amax = fmaxf(amax, fabsf(v[i][j]));
    amax = group_max(amax, kWave);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) amax = fmaxf(amax, red[i]);
    const float s = __fdiv_rn(fmaxf(amax, 1e-4f), 448.0f);
    if (threadIdx.x == 0) ((float *)J.scales)[wg] = s;
    if (c0 >= k) return;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (r0 + 16 * i >= rows) return;
        *(uint32_t *)(J.codes + (size_t)(r0 + 16 * i) * k + c0) =
            e4m3x4_sat(__fdiv_rn(v[i].x, s), __fdiv_rn(v[i].y, s), __fdiv_rn(v[i].z, s), __fdiv_rn(v[i].w, s));
    }
}

// The same for any k and alignment: one workgroup of 256 threads per block, value by value.
__global__ __launch_bounds__(256) void k_quant_fp8_b128(const float *w, int rows, int k, uint8_t *codes,
                                                        float *scales) {
    __shared__ float red[4];
    const int bi = blockIdx.y, bj = blockIdx.x, kb = gridDim.x;
    const int r0 = bi * 128, c0 = bj * 128;
    const int nr = min(128, rows - r0), nc = min(128, k - c0);
    float amax = 0.f;
    for (int i = threadIdx.x; i < nr * nc; i += 256) amax = fmaxf(amax, fabsf(w[(size_t)(r0 + i / nc) * k + c0 + i % nc]));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = __fdiv_rn(fmaxf(amax, 1e-4f), 448.0f);
    if (threadIdx.x == 0) scales[(size_t)bi * kb + bj] = s;
    for (int i = threadIdx.x; i < nr * nc; i += 256) {
        const size_t at = (size_t)(r0 + i / nc) * k + c0 + i % nc;
        codes[at] = (uint8_t)f32_to_e4m3(fminf(fmaxf(__fdiv_rn(w[at], s), -448.f), 448.f));
    }
}

// FP8 e4m3 with one E8M0 scale per 32x32 block (the reference engine's FP8 layout, stbl/kernels.cu:
// 98-103): s = pow2_ceil(max(amax, 1e-4) * fp32(1/448)) as act_quant's power-of-two rule
// (ref/kernel.py:38-40), q = e4m3_rne(clamp(w / s, +-448)) (w / s is exact, and w times the inverse of
// s is). scales [(rows+31)/32][k/32] bytes. One wave per block, holding it in registers: lane l has 4
// columns of rows l / 8, l / 8 + 8, ... (rows past the edge reload the last one), so every load reads
// eight whole 128-byte lines, and the block is read once. w 16-byte, codes 4-byte aligned. 5120 x 2304:
// 35.6 us with two scalar passes by 256 threads, 12.2 us (4.8 TB/s) so.
__global__ __launch_bounds__(256) void k_quant_fp8_e8m0_x4(QuantJobs jobs) {
    uint32_t wg;
    const QuantJob &J = quant_job(jobs, wg);
    const int rows = J.rows, k = J.k, kb = k >> 5, kw = (kb + 3) >> 2;  // kw: workgroups (four blocks) per block row
    const int bi = (int)(wg / kw), bj = (int)(wg % kw) * 4 + (threadIdx.x >> 6);
    if (bj >= kb) return;  // the whole wave
    const int lane = threadIdx.x & 63, r0 = bi * 32 + (lane >> 3), c0 = bj * 32 + (lane & 7) * 4;
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        v[i] = __builtin_nontemporal_load((const f32x4 *)(J.w + (size_t)min(r0 + 8 * i, rows - 1) * k + c0));
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) amax = fmaxf(amax, fabsf(v[i][j]));
    const float s = pow2_ceil(fmaxf(group_max(amax, kWave), 1e-4f) * (1.0f / 448.0f));
    const float inv = pow2_inverse(s);
    if (lane == 0) ((uint8_t *)J.scales)[(size_t)bi * kb + bj] = (uint8_t)((__float_as_uint(s) >> 23) & 0xffu);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (r0 + 8 * i >= rows) return;
        *(uint32_t *)(J.codes + (size_t)(r0 + 8 * i) * k + c0) =
            e4m3x4_sat(v[i].x * inv, v[i].y * inv, v[i].z * inv, v[i].w * inv);
    }
}

// The same for any alignment: one 256-thread workgroup per block, value by value.
__global__ __launch_bounds__(256) void k_quant_fp8_e8m0(const float *w, int rows, int k, uint8_t *codes,
                                                        uint8_t *scales) {
    __shared__ float red[4];
    const int bi = blockIdx.y, bj = blockIdx.x, kb = gridDim.x;
    const int r0 = bi * 32, c0 = bj * 32, nr = min(32, rows - r0);
    float amax = 0.f;
    for (int i = threadIdx.x; i < nr * 32; i += 256) amax = fmaxf(amax, fabsf(w[(size_t)(r0 + i / 32) * k + c0 + i % 32]));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = pow2_ceil(fmaxf(amax, 1e-4f) * (1.0f / 448.0f));
    if (threadIdx.x == 0) scales[(size_t)bi * kb + bj] = (uint8_t)((__float_as_uint(s) >> 23) & 0xffu);
    for (int i = threadIdx.x; i < nr * 32; i += 256) {
        const size_t at = (size_t)(r0 + i / 32) * k + c0 + i % 32;
        codes[at] = (uint8_t)f32_to_e4m3(fminf(fmaxf(__fdiv_rn(w[at], s), -448.f), 448.f));
    }
}

// ---- dequantizers (the bit-exactness check of the decoders the GEMVs use) ------------------------

// FP4 OCP: out[r][c] = e2m1(code) * 2^(s-127), one fp32 product. One thread per 32-group.
__global__ void k_dequant_fp4(const uint8_t *codes, const uint8_t *scales, int n_groups, float *out) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_groups) return;
    const u32x4 w = *(const u32x4 *)(codes + (size_t)g * 16);
    const float s = e8m0_to_f32(scales[g]);
    float *o = out + (size_t)g * 32;
#pragma unroll
    for (int d = 0; d < 4; d++) {
        const f32x2 a = e2m1x2<0>(w[d]), b = e2m1x2<1>(w[d]), c = e2m1x2<2>(w[d]), e = e2m1x2<3>(w[d]);
        *(f32x4 *)(o + 8 * d) = f32x4{a.x * s, a.y * s, b.x * s, b.y * s};
        *(f32x4 *)(o + 8 * d + 4) = f32x4{c.x * s, c.y * s, e.x * s, e.y * s};
    }
}

// GGUF MXFP4 rows of 17-byte blocks (byte 0: E8M0 scale; bytes 1..16: element i in the low nibble
// and element 16+i in the high nibble of byte 1+i). One thread per block, byte reads.
__global__ void k_dequant_gguf17(const uint8_t *w, int n_blocks, float *out) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_blocks) return;
    const uint8_t *blk = w + (size_t)g * 17;
    const float s = e8m0_to_f32(blk[0]);
    float *o = out + (size_t)g * 32;
    for (int i = 0; i < 16; i++) {
        const uint32_t byte = blk[1 + i];
        const f32x2 v = e2m1x2<0>(byte);
        o[i] = v.x * s;
        o[16 + i] = v.y * s;
    }
}

// FP8 e4m3 with fp32 128x128 block scales (scale_e8m0 == 0), or with E8M0 bytes per 32x32 block, the
// reference engine's layout [(rows+31)/32][k/32] (scale_e8m0 == 1). One thread per 16 values.
__global__ void k_dequant_fp8(const uint8_t *codes, const void *scales, int rows, int k, int scale_e8m0, float *out) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 16;
    if (i >= (size_t)rows * k) return;
    const int r = (int)(i / k), c = (int)(i % k);
    const u32x4 w = *(const u32x4 *)(codes + i);
    float s;
    if (scale_e8m0) s = e8m0_to_f32(((const uint8_t *)scales)[(size_t)(r >> 5) * (k >> 5) + (c >> 5)]);
    else s = ((const float *)scales)[(size_t)(r >> 7) * ((k + 127) >> 7) + (c >> 7)];
    float *o = out + i;
#pragma unroll
    for (int d = 0; d < 4; d++) {
        const f32x2 a = e4m3x2(w[d], false), b = e4m3x2(w[d], true);
        *(f32x4 *)(o + 4 * d) = f32x4{a.x * s, a.y * s, b.x * s, b.y * s};
    }
}

// ---- epilogues (stbl/kernels.cu:86-89, 444-464) --------------------------------------------------

__global__ void k_round_bf16(float *x, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = bf16_round(x[i]);
}

constexpr int kSegMax = 16;
struct SegWeights {
    float w[kSegMax];
};

// out = bf16(silu(min(g, lim)) * clamp(u, +-lim) * w), no clamps when lim <= 0; segment blockIdx.y
// of `count` consecutive n-long segments uses weight w[blockIdx.y]. silu(g) = g / (1 + exp(-g)).
__global__ void k_swiglu(float *out, const float *g, const float *u, SegWeights ws, float limit, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t at = (size_t)blockIdx.y * n + i;
    float gv = g[at], uv = u[at];
    if (limit > 0) {
        uv = fminf(fmaxf(uv, -limit), limit);
        gv = fminf(gv, limit);
    }
    out[at] = bf16_round(__fdiv_rn(gv, 1.f + expf(-gv)) * uv * ws.w[blockIdx.y]);
}

// y += a * x as one fused multiply-add (nvcc contracts the reference's `y[i] += a * x[i]`).
__global__ void k_axpy(float *y, const float *x, float a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = fmaf(a, x[i], y[i]);
}

static inline unsigned grid_for(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Quantizes n <= 3 matrices to one format (ExpertFmt) in one launch; each as its kernel above needs it.
static hipError_t launch_quant(int fmt, const QuantJob *jobs, int n, hipStream_t st) {
    QuantJobs all = {};
    uint32_t wgs = 0;
    for (int i = 0; i < 3; i++) {
        if (i >= n) {
            all.j[i].first = UINT32_MAX;
            continue;
        }
        all.j[i] = jobs[i];
        all.j[i].first = wgs;
        const size_t rows = jobs[i].rows, k = jobs[i].k;
        if (fmt == EXPERT_FP4) wgs += grid_for(rows * (k / 16), 256);
        else if (fmt == EXPERT_FP8) wgs += (uint32_t)(((rows + 127) / 128) * ((k + 127) / 128));
        else wgs += (uint32_t)(((rows + 31) / 32) * ((k / 32 + 3) / 4));
    }
    if (fmt == EXPERT_FP4) hipLaunchKernelGGL(k_quant_fp4, dim3(wgs), dim3(256), 0, st, all);
    else if (fmt == EXPERT_FP8) hipLaunchKernelGGL(k_quant_fp8_b128_x4, dim3(wgs), dim3(512), 0, st, all);
    else hipLaunchKernelGGL(k_quant_fp8_e8m0_x4, dim3(wgs), dim3(256), 0, st, all);
    return hipGetLastError();
}

}  // namespace stbl

using namespace stbl;

extern "C" {

// stbl/kernels.h:9. n % 32 == 0.
void stbl_act_quant_fp8(float *x, int n, hipStream_t st) {
    if (!x || n <= 0 || n % 32) {
        abi_fail(hipErrorInvalidValue, "stbl_act_quant_fp8: need n %% 32 == 0 (n=%d)", n);
        return;
    }
    hipLaunchKernelGGL(k_act_quant_fp8_inplace, dim3(grid_for((size_t)n, 256)), dim3(256), 0, st, x, n / 32);
    abi_status(hipGetLastError(), "stbl_act_quant_fp8 launch");
}

// stbl/kernels.h:11.
void stbl_round_bf16(float *x, int n, hipStream_t st) {
    if (!x || n <= 0) {
        abi_fail(hipErrorInvalidValue, "stbl_round_bf16: bad arguments (n=%d)", n);
        return;
    }
    hipLaunchKernelGGL(k_round_bf16, dim3(grid_for((size_t)n, 256)), dim3(256), 0, st, x, n);
    abi_status(hipGetLastError(), "stbl_round_bf16 launch");
}

// stbl/kernels.h:37-38. `weights` is a host array of `count` <= 16 floats.
void stbl_swiglu_batch(float *out, const float *g, const float *u, const float *weights, int count, float limit, int n,
                       hipStream_t st) {
    if (!out || !g || !u || !weights || count <= 0 || count > kSegMax || n <= 0) {
        abi_fail(hipErrorInvalidValue, "stbl_swiglu_batch: bad arguments (count=%d n=%d)", count, n);
        return;
    }
    SegWeights ws = {};
    for (int j = 0; j < count; j++) ws.w[j] = weights[j];
    hipLaunchKernelGGL(k_swiglu, dim3(grid_for((size_t)n, 256), count), dim3(256), 0, st, out, g, u, ws, limit, n);
    abi_status(hipGetLastError(), "stbl_swiglu_batch launch");
}

// stbl/kernels.h:35.
void stbl_swiglu(float *out, const float *g, const float *u, float weight, float limit, int n, hipStream_t st) {
    stbl_swiglu_batch(out, g, u, &weight, 1, limit, n, st);
}

// stbl/kernels.h:39.
void stbl_axpy(float *y, const float *x, float a, int n, hipStream_t st) {
    if (!y || !x || n <= 0) {
        abi_fail(hipErrorInvalidValue, "stbl_axpy: bad arguments (n=%d)", n);
        return;
    }
    hipLaunchKernelGGL(k_axpy, dim3(grid_for((size_t)n, 256)), dim3(256), 0, st, y, x, a, n);
    abi_status(hipGetLastError(), "stbl_axpy launch");
}

int stbl_amd_act_quant(const void *x, int rows, int n, int block, int pow2, void *codes, float *scales, void *deq,
                       hipStream_t st) {
    if (!x || rows <= 0 || n <= 0 || block <= 0 || n % block) return abi_fail(hipErrorInvalidValue, "act_quant: need n %% block == 0");
    // 8 values a lane where a block is 1, 2, 4, ... 64 lanes and the pointers take its wide accesses; the
    // index of 8 values is an int
    const int lanes = block / 8;
    const size_t n8 = (size_t)rows * n / 8;
    if (block % 8 == 0 && lanes <= kWave && (lanes & (lanes - 1)) == 0 && n8 <= 0x7fffff00u && aligned16(x) &&
        ((uintptr_t)codes & 7) == 0 && aligned16(deq)) {
        const dim3 grid(grid_for(n8, 256));
        if (pow2)
            hipLaunchKernelGGL(k_act_quant8<true>, grid, dim3(256), 0, st, (const uint16_t *)x, (int)n8, lanes,
                               (uint8_t *)codes, scales, (uint16_t *)deq);
        else
            hipLaunchKernelGGL(k_act_quant8<false>, grid, dim3(256), 0, st, (const uint16_t *)x, (int)n8, lanes,
                               (uint8_t *)codes, scales, (uint16_t *)deq);
        return abi_status(hipGetLastError(), "act_quant launch");
    }
    const int nb = rows * (n / block);
    hipLaunchKernelGGL(k_act_quant, dim3(grid_for((size_t)nb, 128)), dim3(128), 0, st, (const uint16_t *)x, nb, block,
                       pow2, (uint8_t *)codes, scales, (uint16_t *)deq);
    return abi_status(hipGetLastError(), "act_quant launch");
}

int stbl_amd_quant_fp4(void *codes, void *scales, const float *w, int rows, int k, hipStream_t st) {
    if (!codes || !scales || !w || rows <= 0 || k <= 0 || k % 32) return abi_fail(hipErrorInvalidValue, "quant_fp4: need k %% 32 == 0");
    if (!aligned16(codes) || !aligned16(w)) return abi_fail(hipErrorInvalidValue, "quant_fp4: codes and w must be 16-byte aligned");
    const QuantJob job = {w, (uint8_t *)codes, scales, rows, k, 0};
    return abi_status(launch_quant(EXPERT_FP4, &job, 1, st), "quant_fp4 launch");
}

int stbl_amd_quant_fp8_b128(void *codes, float *scales, const float *w, int rows, int k, hipStream_t st) {
    if (!codes || !scales || !w || rows <= 0 || k <= 0) return abi_fail(hipErrorInvalidValue, "quant_fp8_b128: bad arguments");
    if (k % 4 == 0 && aligned16(w) && ((uintptr_t)codes & 3) == 0) {
        const QuantJob job = {w, (uint8_t *)codes, scales, rows, k, 0};
        return abi_status(launch_quant(EXPERT_FP8, &job, 1, st), "quant_fp8_b128 launch");
    }
    hipLaunchKernelGGL(k_quant_fp8_b128, dim3((k + 127) / 128, (rows + 127) / 128), dim3(256), 0, st, w, rows, k,
                       (uint8_t *)codes, scales);
    return abi_status(hipGetLastError(), "quant_fp8_b128 launch");
}

// FP8 e4m3 with E8M0 scales per 32x32 block: codes [rows][k], scales [(rows+31)/32][k/32]. k % 32 == 0.
int stbl_amd_quant_fp8_e8m0(void *codes, void *scales, const float *w, int rows, int k, hipStream_t st) {
    if (!codes || !scales || !w || rows <= 0 || k <= 0 || k % 32)
        return abi_fail(hipErrorInvalidValue, "quant_fp8_e8m0: need k %% 32 == 0");
    if (aligned16(w) && ((uintptr_t)codes & 3) == 0) {
        const QuantJob job = {w, (uint8_t *)codes, scales, rows, k, 0};
        return abi_status(launch_quant(EXPERT_FP8_E8M0, &job, 1, st), "quant_fp8_e8m0 launch");
    }
    hipLaunchKernelGGL(k_quant_fp8_e8m0, dim3(k / 32, (rows + 31) / 32), dim3(256), 0, st, w, rows, k, (uint8_t *)codes,
                       (uint8_t *)scales);
    return abi_status(hipGetLastError(), "quant_fp8_e8m0 launch");
}

int stbl_amd_quant_expert(int fmt, void *slot, const float *w_gate, const float *w_up, const float *w_down, int dim,
                          int inter, hipStream_t st) {
    const int step = fmt == EXPERT_FP8 ? 4 : 32;
    if (fmt != EXPERT_FP4 && fmt != EXPERT_FP8 && fmt != EXPERT_FP8_E8M0)
        return abi_fail(hipErrorInvalidValue, "quant_expert: unknown format %d", fmt);
    if (!slot || !w_gate || !w_up || !w_down || dim <= 0 || inter <= 0 || dim % step || inter % step)
        return abi_fail(hipErrorInvalidValue, "quant_expert: need dim and inter %% %d == 0 (dim=%d inter=%d)", step, dim, inter);
    if (!aligned16(slot) || !aligned16(w_gate) || !aligned16(w_up) || !aligned16(w_down))
        return abi_fail(hipErrorInvalidValue, "quant_expert: slot and weights must be 16-byte aligned");
    const ExpertLayout L = expert_layout(fmt, dim, inter);
    uint8_t *base = (uint8_t *)slot;
    const QuantJob jobs[3] = {{w_gate, base + L.off[0], base + L.off[1], inter, dim, 0},
                              {w_up, base + L.off[2], base + L.off[3], inter, dim, 0},
                              {w_down, base + L.off[4], base + L.off[5], dim, inter, 0}};
    return abi_status(launch_quant(fmt, jobs, 3, st), "quant_expert launch");
}

int stbl_amd_dequant_fp4(float *out, const void *codes, const void *scales, int rows, int k, hipStream_t st) {
    if (!out || !codes || !scales || rows <= 0 || k <= 0 || k % 32) return abi_fail(hipErrorInvalidValue, "dequant_fp4: need k %% 32 == 0");
    if (!aligned16(codes) || !aligned16(out)) return abi_fail(hipErrorInvalidValue, "dequant_fp4: codes and out must be 16-byte aligned");
    const int ng = rows * (k / 32);
    hipLaunchKernelGGL(k_dequant_fp4, dim3(grid_for((size_t)ng, 256)), dim3(256), 0, st, (const uint8_t *)codes,
                       (const uint8_t *)scales, ng, out);
    return abi_status(hipGetLastError(), "dequant_fp4 launch");
}

int stbl_amd_dequant_gguf17(float *out, const void *w, int rows, int k, hipStream_t st) {
    if (!out || !w || rows <= 0 || k <= 0 || k % 32) return abi_fail(hipErrorInvalidValue, "dequant_gguf17: need k %% 32 == 0");
    const int nb = rows * (k / 32);
    hipLaunchKernelGGL(k_dequant_gguf17, dim3(grid_for((size_t)nb, 256)), dim3(256), 0, st, (const uint8_t *)w, nb, out);
    return abi_status(hipGetLastError(), "dequant_gguf17 launch");
}

int stbl_amd_dequant_fp8(float *out, const void *codes, const void *scales, int rows, int k, int scale_e8m0,
                         hipStream_t st) {
    if (!out || !codes || !scales || rows <= 0 || k <= 0 || k % 16 || (scale_e8m0 && k % 32))
        return abi_fail(hipErrorInvalidValue, "dequant_fp8: need k %% 16 == 0 (k %% 32 for E8M0 scales)");
    if (!aligned16(codes) || !aligned16(out)) return abi_fail(hipErrorInvalidValue, "dequant_fp8: codes and out must be 16-byte aligned");
    hipLaunchKernelGGL(k_dequant_fp8, dim3(grid_for((size_t)rows * k / 16, 256)), dim3(256), 0, st,
                       (const uint8_t *)codes, scales, rows, k, scale_e8m0, out);
    return abi_status(hipGetLastError(), "dequant_fp8 launch");
}

}  // extern "C"
