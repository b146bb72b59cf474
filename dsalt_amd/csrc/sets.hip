// Sets of landmark positions in any order -> ascending with -1 last, the source slot of each
// output slot, and the slots' biases in the same order.
//
// One block per set.  Sets a selection made are already in order: the block compares
// neighbours and copies.  Else each slot counts the slots that come before it (equal
// positions keep their order), k^2 / threads LDS reads: the sets are small (usually at most 128
// slots), so one launch is bound by its latency, where a general radix sort with the selects,
// conversions and gathers around it took eleven launches (8 sets of 64 slots: 21.7 of about 45 us
// on the GPU in the sort alone, with their host time more than the attention forward beside
// them).  From about 512 slots on the count is the slower way for sets out of order (8 sets of
// 1024: 214 us against 57), and a caller with such sets sorts them otherwise.
#include "sets.h"

#include "common.h"
#include "timing.h"

namespace dsalt {

namespace {

constexpr int kSortThreads = 256;
constexpr int64_t kSortLast = 0x7fffffff;  // key of an empty slot: after every position

__global__ __launch_bounds__(kSortThreads) void sort_sets_kernel(SortSetsParams p) {
    __shared__ int64_t key[kMaxLandmarks];
    const int tid = threadIdx.x, K = p.k;
    for (int64_t set = blockIdx.x; set < p.n_sets; set += gridDim.x) {
        const int64_t o = set * K;
        for (int i = tid; i < K; i += kSortThreads) {
            const int64_t v = p.idx64 ? ((const int64_t*)p.idx)[o + i] : (int64_t)((const int32_t*)p.idx)[o + i];
            key[i] = v < 0 ? kSortLast : v;
        }
        __syncthreads();
        int unsorted = 0;
        for (int i = tid; i + 1 < K; i += kSortThreads) unsorted |= key[i] > key[i + 1];
        unsorted = __syncthreads_or(unsorted);
        for (int i = tid; i < K; i += kSortThreads) {
            const int64_t x = key[i];
            int r = i;
            if (unsorted) {
                r = 0;
                for (int j = 0; j < K; ++j) r += key[j] < x || (key[j] == x && j < i);
            }
            p.out[o + r] = x == kSortLast ? -1 : (int32_t)x;
            p.perm[o + r] = i;
            if (p.bias_bytes == 4) ((uint32_t*)p.bias_out)[o + r] = ((const uint32_t*)p.bias)[o + i];
            else if (p.bias_bytes == 2) ((uint16_t*)p.bias_out)[o + r] = ((const uint16_t*)p.bias)[o + i];
        }
        __syncthreads();  // the next set reuses the keys
    }
}

}  // namespace

hipError_t sort_sets_launch(const SortSetsParams& p, hipStream_t stream) {
    if (p.n_sets == 0 || p.k == 0) return hipSuccess;
    const int64_t blocks = p.n_sets < (1 << 16) ? p.n_sets : (1 << 16);
    DSALT_LAUNCH("sort_sets", sort_sets_kernel, dim3((unsigned)blocks), dim3(kSortThreads), 0, stream, p);
    return hipGetLastError();
}

}  // namespace dsalt
