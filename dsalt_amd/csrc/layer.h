// Integer windows and score weights of a DSALT attention layer.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

namespace dsalt {

struct SelectorsParams {
    int total_len, n_heads, dtype;
    const void* gate;     // [T] window-gate logits
    int64_t gate_st;
    const void* alpha_w;  // [H]
    float n_min, n_span;  // n_span = n_max - n_min
    int32_t* w;           // [T] out
    float* alpha;         // [H] out
};

hipError_t selectors_launch(const SelectorsParams& p, hipStream_t stream);

}  // namespace dsalt
