// Which kernel a GEMM call takes, and the workspace it needs: plain host C++, so that the rules can be
// checked against each other without a GPU. operand_group is called by k_gemm_one and k_gemm_waves too.
#pragma once

#include <algorithm>
#include <cstdint>

#ifdef __HIPCC__
#define STBL_HD __host__ __device__ __forceinline__
#else
#define STBL_HD inline
#endif

namespace stbl {

constexpr int kGemmMaxM = 64;
constexpr int kGemmMaxN = 1 << 20;
constexpr int kGemmMaxRows = 8192;  // of stbl_amd_gemm_rows

// Kernel, tile shape and split of K, chosen per shape (each choice measured fastest for its shape). Calls of
// up to 64 rows:
//   kOne64, k_gemm_one with 32 x 64 tiles on 4 waves of 4 steps, when K % 512 == 0, K <= 2048, m > 32
//     and the tiles give >= 192 workgroups (7168 x 2048: 6.6 us);
//   kOne32, k_gemm_one with 16 x 32 tiles on up to 8 waves of 8 steps (FP4 weights: 8.2 -> 7.9 us
//     against 16 waves of 4, 8.9 with 4 waves of 16) or 16 waves of 4 steps (FP8), when K % 512 == 0,
//     K <= 8192, m > 32 and the tiles give >= 192 workgroups (2048 x 7168: 11.7 -> 8.3 us against
//     kSplit);
//   kWaves24, k_gemm_waves with 32 x 64 tiles, when K <= 2048, m > 32 and these give >= 192 workgroups
//     (unaligned scales or K % 512 != 0; 64 x 7168 x 1920: 7.6 us FP4, 8.3 FP8; with 16 waves of one
//     step 7.6 and 9.6);
//   kWaves22, k_gemm_waves with 32 x 32 tiles, for other K of up to kSplitSteps steps;
//   kSplit otherwise, k_gemm with 64 x 64 tiles and 8 waves of one step each, K split into slices of <= 8
//     steps, as many as it takes to give >= 200 workgroups (2048 x 7168: 7 slices, 224 workgroups),
//     and k_gemm_reduce: with few tiles and many steps the waves of one workgroup are too few
//     (64 x 512 x 4096: 9.7 us, 13.3 with k_gemm_waves; x 3072: 10.0 and 8.5; 10 x 2048 x 3584: 9.0 and 7.5).
// Calls of more rows: kWaves22 while its 32 x 32 tiles give at most one workgroup per CU, kWaves24 up to
// twice that (700 x 512 x 4096 FP8: 15.1 us, 19.2 with 32 x 32 and 20.8 with k_gemm_tile), then k_gemm_tile
// with 64 x 64 tiles (kTile64) or, from one of those per CU on, 64 x 128 tiles on twice the waves (kTile128:
// 600 x 2048 x 7168 31.4 -> 29.5 us, 1024 x 7168 x 2048 33.2 -> 31.1; 300 x 2048 x 7168 23.9 -> 27.6).
enum GemmKernel { kSplit, kWaves22, kWaves24, kOne32, kOne64, kTile64, kTile128 };

constexpr int kSplitSteps = 26;
constexpr int kCUs = 256;

struct GemmPlan {
    GemmKernel kernel;
    bool chain;  // how the call sums K (k_gemm_tile): steps in groups of `group`, chained or not
    int group;
    int slices;  // kSplit: of `group` steps
};

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// aligned: the scale arrays are 16-byte aligned (k_gemm_one and chained sums load 4 steps' scales at once).
// Rows of a call of more than 64 are summed as those of a call of 64, whatever the kernel.
inline GemmPlan gemm_plan(int fmt, int m, int n, int k, bool aligned) {
    const int ks = k / 128, mc = std::min(m, kGemmMaxM);
    GemmPlan p = {};
    if (aligned && ks % 4 == 0 && ks <= 16 && mc > 32 && ceil_div(n, 64) * ceil_div(mc, 32) >= 192) {
        p = {kOne64, true, 4, 1};
    } else if (aligned && ks % 4 == 0 && ks <= 64 && mc > 32 && ceil_div(n, 32) * ceil_div(mc, 16) >= 192) {
        p = {kOne32, true, fmt == 0 ? 8 : 4, 1};
    } else if (ks <= 16 && mc > 32 && 2 * ceil_div(n, 64) >= 192) {
        p = {kWaves24, false, 1, 1};
    } else if (ks <= 16 && ceil_div(n, 32) >= 192) {
        p = {kWaves22, false, 1, 1};
    } else {
        const int tiles = ceil_div(n, 64);
        const int want = std::max(ceil_div(ks, 8), std::min(ks, ceil_div(200, tiles)));
        p.group = ceil_div(ks, want), p.slices = ceil_div(ks, p.group);
        p.kernel = ks > kSplitSteps ? kSplit : kWaves22;
        if (p.slices == 1) p.group = 1;  // one running sum over the steps
    }
    if (m <= kGemmMaxM) return p;
    const int64_t t32 = (int64_t)ceil_div(m, 32) * ceil_div(n, 32), t64 = (int64_t)ceil_div(m, 64) * ceil_div(n, 64);
    p.kernel = t32 <= kCUs ? kWaves22 : t32 <= 2 * kCUs ? kWaves24 : t64 < kCUs ? kTile64 : kTile128;
    return p;
}

// Rows of a kernel's output tiles.
constexpr int tile_rows(GemmKernel kernel) {
    return kernel == kOne32 ? 16 : kernel == kOne64 || kernel == kWaves22 || kernel == kWaves24 ? 32 : 64;
}

inline bool is_tile(const GemmPlan &p) { return p.kernel == kTile64 || p.kernel == kTile128; }

inline uint64_t a256(uint64_t v) { return (v + 255) & ~(uint64_t)255; }

// Bytes the partial tiles of a call of up to 64 rows take at the front of `work`. The split of K does not
// depend on m, and a call whose scale arrays are not 16-byte aligned may split where an aligned one does
// not, so the size is that of the plan without alignment.
inline uint64_t part_reserve(int n, int k) {
    const GemmPlan p = gemm_plan(0, 1, n, k, false);
    return p.kernel == kSplit ? a256((uint64_t)ceil_div(n, 64) * p.slices * (4 * 4 * 64) * 16) : 0;
}

// Rows of the activation codes in the workspace: a whole number of 16-row groups (operand order).
inline uint64_t aq_bytes(int m, int k) { return a256((uint64_t)ceil_div(m, 16) * 16 * k); }

// The 16-row group of activations in operand order that m-tile mt of the output tile at row m0 reads:
// past the call's last group that group again, as the workspace holds no further one (aq_bytes).
STBL_HD int operand_group(int m0, int mt, int m) {
    const int group = (m0 >> 4) + mt, last = (m - 1) >> 4;
    return group < last ? group : last;
}

// The workspace of a call of more than 64 rows: activation codes in operand order, then their scales (bytes
// [m][k / block] for the kernels that read those, dwords [k / 128][m] for k_gemm_tile), then the FP4
// weights' scale dwords.
inline uint64_t rows_work_bytes(int m, int n, int k) {
    return aq_bytes(m, k) + a256((uint64_t)m * (k / 32)) + a256((uint64_t)n * (k / 32));
}

inline uint64_t gemm_work_bytes(int m, int n, int k) {
    if (m < 1 || n < 1 || k < 128) return 256;
    const uint64_t few = part_reserve(n, k) + aq_bytes(std::min(m, kGemmMaxM), k) + a256((uint64_t)std::min(m, kGemmMaxM) * (k / 32)) + 256;
    return m > kGemmMaxM ? std::max(few, rows_work_bytes(m, n, k)) : few;
}

}  // namespace stbl
