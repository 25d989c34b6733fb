// Rules of an MoE step: plain host C++, so that they can be checked without a GPU.
#pragma once

#include <cstdint>

namespace stbl {

// Whether a step quantizes x and its SwiGLU outputs in two launches of their own (k_moe_act_quant), or every
// workgroup its tokens' chunks in registers. The launches cost about 2.7 us whatever the size. What they
// save grows with the waves that would quantize, times the tokens of each: 4 rows of gate and up, 8 of down a
// workgroup, a wave per 2048 values of K. Only jobs of several tokens count (`tokens`: the sum of theirs): a
// one-token job's quantization hides behind its weights. FP8 experts stream twice the bytes per product
// and hide more. In registers -> in launches, us (top-k, tokens of a step; waves x tokens):
//   FP4 routed  1024 x 512 top-4, 2       10.5 -> 13.3 (1024)    3072 x 1024 top-6, 2   19.9 -> 21.3 (7168)
//               4096 x 1536 top-8, 2      30.2 -> 32.1 (12800)   5120 x 512 top-6, 3    27.7 -> 29.1 (13312)
//               2304 x 2304 top-8, 2      36.2 -> 33.5 (17280)   5120 x 512 top-8, 4    47.2 -> 45.0 (25600)
//               7168 x 2048 top-8, 3      84.5 -> 80.0 (44160)   5120 x 2304 top-8, 4  100.8 -> 88.5 (75200)
//   FP8 routed  5120 x 512 top-6, 6       40.0 -> 41.9 (33792)   3072 x 1024 top-8, 6   39.7 -> 42.4 (43904)
//               2048 x 1024 top-6, 16     46.8 -> 46.3 (54272)   2048 x 1024 top-8, 16  66.9 -> 61.8 (70144)
// Against the better of both ways the line costs a tenth at worst in 900 such steps, 0.2% on average.
inline bool quantize_once(bool fp4, int64_t tokens, int dim, int inter) {
    const int64_t gate_up = (int64_t)((dim + 2047) / 2048) * ((inter + 3) / 4);
    const int64_t down = (int64_t)((inter + 2047) / 2048) * ((dim + 7) / 8);
    return tokens * (gate_up + down) >= (fp4 ? 14000 : 50000);
}

// Whether the router takes a workgroup a token, whose four waves share the scores, instead of a wave (k_route).
// Few tokens leave the GPU idle, and a wave's scores then take longer than its top-k: from 5 a lane on, or
// from 2 with the longer sqrt(softplus) (score_fn 1). Many tokens fill it either way, and three of
// the four waves only wait. A wave -> a workgroup, us, top-1:
//   1 token:      384 experts 2.9 -> 2.5, with sqrt(softplus) 4.4 -> 3.2; 1024 8.7 -> 4.5; 256 3.3 -> 2.4
//   2048 tokens:  384 experts 3.6 -> 3.7, with sqrt(softplus) 5.8 -> 5.6; 1024 11.7 -> 10.3; 256 (1024 tokens) 4.0 -> 3.7
//   8192 tokens:  384 experts 6.4 -> 7.7, with sqrt(softplus) 12.5 -> 13.5; 256 9.0 -> 11.9
inline bool route_split(int n_exp, int t, int score_fn) {
    return n_exp > 256 ? t <= 2048 : n_exp > 64 && score_fn == 1 && t <= 1024;
}

}  // namespace stbl
