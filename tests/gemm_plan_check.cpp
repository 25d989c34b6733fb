// gemm_plan.hpp's rules against each other, over both formats, aligned and unaligned scales, every m up to 64
// and larger ones around whole tiles: no tile reads an activation group that the workspace does not hold, and
// the parts of the workspace fit its size. Prints the first call that breaks a rule. Built as a library, it
// tells the GPU tests which kernel a call takes.
#include <cstdio>

#include "gemm_plan.hpp"

using namespace stbl;

static int check(int fmt, int m, int n, int k, bool aligned) {
    const GemmPlan p = gemm_plan(fmt, m, n, k, aligned);
    const int rows = tile_rows(p.kernel);
    const uint64_t codes = aq_bytes(m, k), front = m <= kGemmMaxM ? part_reserve(n, k) : 0;
    const uint64_t scales = is_tile(p) ? a256((uint64_t)m * (k / 32)) + (uint64_t)n * (k / 32) : (uint64_t)m * (k / 32);
    const char *broken = nullptr;
    for (int m0 = 0; m0 < m && p.kernel != kSplit; m0 += rows)  // kSplit reads codes row by row
        for (int mt = 0; mt < rows / 16; mt++)
            if ((uint64_t)(operand_group(m0, mt, m) + 1) * 16 * k > codes) broken = "activation group past the workspace's";
    if (front + codes + scales > gemm_work_bytes(m, n, k)) broken = "workspace too small";
    if (broken) printf("%s: kernel %d, fmt %d, %d x %d x %d, aligned %d\n", broken, p.kernel, fmt, m, n, k, aligned);
    return broken ? 1 : 0;
}

// Per call: the kernel (GemmKernel), whether sums chain, and the steps of a group.
extern "C" void gemm_plan_of(int fmt, int m, int n, int k, int aligned, int *out) {
    const GemmPlan p = gemm_plan(fmt, m, n, k, aligned != 0);
    out[0] = p.kernel, out[1] = p.chain, out[2] = p.group;
}

int main() {
    const int ns[] = {1, 16, 64, 200, 512, 1536, 2048, 3072, 4096, 6080, 6096, 6144, 6160, 7168, 12288, 16384};
    const int ks[] = {128, 256, 384, 512, 1024, 1536, 1920, 2048, 2176, 3328, 3456, 4096, 6656, 7168, 8192, 8704};
    for (int n : ns)
        for (int k : ks)
            for (int fmt = 0; fmt < 2; fmt++)
                for (int aligned = 0; aligned < 2; aligned++) {
                    for (int m = 1; m <= 64; m++)
                        if (check(fmt, m, n, k, aligned)) return 1;
                    for (int m : {65, 79, 80, 81, 97, 128, 129, 300, 321, 1000, 1024, 8191, 8192})
                        if (check(fmt, m, n, k, aligned)) return 1;
                }
    return 0;
}
