// w = max(floor(n_min + sigmoid(gate) (n_max - n_min)), 1) per token and alpha = sigmoid(alpha_w)
// per head, each operation rounded to the tensor type as the elementwise expression evaluated one
// operation at a time (this file is compiled without fused multiply-adds).  A few KB of work, so
// one launch in place of ten is all there is to gain: 997 tokens, bf16, about 17 us of a layer's
// GPU time -> 2.6 us, and the host time of nine launches (the layer call 303 -> 183 us with the
// score outputs, conversions and plan launch it no longer asks for).
#include "layer.h"

#include "common.h"
#include "timing.h"

namespace dsalt {

namespace {

template <typename T>
__device__ __forceinline__ float rounded(float x) {
    return to_float(from_float<T>(x));
}
template <typename T>
__device__ __forceinline__ float sigmoid_of(T x) {
    return rounded<T>(1.0f / (1.0f + expf(-to_float(x))));
}

template <typename T>
__global__ __launch_bounds__(256) void selectors_kernel(SelectorsParams p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < p.total_len) {
        const float s = sigmoid_of(((const T*)p.gate)[(int64_t)i * p.gate_st]);
        const float w = rounded<T>(__fadd_rn(rounded<T>(__fmul_rn(s, p.n_span)), p.n_min));
        p.w[i] = max((int)floorf(w), 1);
    } else if (i - p.total_len < p.n_heads) {
        p.alpha[i - p.total_len] = sigmoid_of(((const T*)p.alpha_w)[i - p.total_len]);
    }
}

}  // namespace

hipError_t selectors_launch(const SelectorsParams& p, hipStream_t stream) {
    const int n = p.total_len + p.n_heads;
    if (n == 0) return hipSuccess;
    const dim3 grid(ceil_div(n, 256));
    switch (p.dtype) {
        case 0: DSALT_LAUNCH("selectors", selectors_kernel<float>, grid, dim3(256), 0, stream, p); break;
        case 1: DSALT_LAUNCH("selectors", selectors_kernel<bf16>, grid, dim3(256), 0, stream, p); break;
        default: DSALT_LAUNCH("selectors", selectors_kernel<f16>, grid, dim3(256), 0, stream, p); break;
    }
    return hipGetLastError();
}

}  // namespace dsalt
