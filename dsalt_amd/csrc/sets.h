// Landmark sets handed in by a caller, put into the order the attention kernels read.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

namespace dsalt {

struct SortSetsParams {
    int64_t n_sets;
    int k;              // slots per set, at most kMaxLandmarks
    int idx64;          // positions are int64 (else int32)
    const void* idx;    // [n_sets, k]
    int32_t* out;       // [n_sets, k] ascending, -1 last
    int64_t* perm;      // [n_sets, k] source slot of each output slot
    const void* bias;   // [n_sets, k] of bias_bytes each (2 or 4), or null
    void* bias_out;
    int bias_bytes;
};

hipError_t sort_sets_launch(const SortSetsParams& p, hipStream_t stream);

}  // namespace dsalt
