// moe_plan.hpp's rules at measured sizes: the way that was faster.
#include <cstdio>

#include "moe_plan.hpp"

int main() {
    const struct {
        bool fp4;
        int tokens, dim, inter;
        bool once;
    } steps[] = {{true, 4, 1024, 512, false},   {true, 15, 1024, 512, false},   {true, 4, 2048, 1024, false},
                 {true, 8, 3072, 1024, false},  {true, 10, 4096, 1536, false},  {true, 13, 5120, 512, false},
                 {true, 10, 2304, 2304, true},  {true, 25, 5120, 512, true},    {true, 15, 7168, 2048, true},
                 {true, 19, 5120, 2304, true},  {true, 25, 5120, 2304, true},   {false, 33, 5120, 512, false},
                 {false, 12, 7168, 2048, false}, {false, 49, 3072, 1024, false}, {false, 137, 2048, 1024, true},
                 {false, 25, 5120, 2304, true}, {true, 272, 16384, 16384, true}, {true, 0, 16384, 16384, false}};
    for (const auto &s : steps)
        if (stbl::quantize_once(s.fp4, s.tokens, s.dim, s.inter) != s.once) {
            printf("fp4 %d, %d tokens, %d x %d: not %d\n", s.fp4, s.tokens, s.dim, s.inter, s.once);
            return 1;
        }
    const struct {
        int n_exp, t, score_fn;
        bool split;
    } routers[] = {{64, 1, 1, false},   {128, 1, 0, false},   {128, 1, 1, true},    {256, 1, 1, true},    {256, 1024, 1, true},
                   {256, 2048, 1, false}, {257, 1, 0, true},  {384, 2, 1, true},    {512, 1024, 0, true}, {1024, 2048, 1, true},
                   {384, 8192, 0, false}, {1024, 8192, 1, false}};
    for (const auto &r : routers)
        if (stbl::route_split(r.n_exp, r.t, r.score_fn) != r.split) {
            printf("router of %d experts, %d tokens, score %d: not %d\n", r.n_exp, r.t, r.score_fn, r.split);
            return 1;
        }
    return 0;
}
