// attn_common.h -- the window and cache-row arithmetic that the attention
// kernels share.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

namespace mrml {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ size_t cache_row_of(int t, int capacity) { return (size_t)(capacity > 0 ? t % capacity : t); }

// The window: the last min(n_past + 1, limit) positions, limit = the cache
// capacity or, below it, the sliding window (cuda.rs:2658-2697 sliding_window;
// kernels.rs:1398-1404).  Cache rows stay position % capacity.
__device__ __forceinline__ void attn_window(const int32_t *d_pos, int n_past_arg, int limit, int &window, int &start)
{
    const int n_past = d_pos ? *d_pos : n_past_arg;
    const int count = n_past + 1;
    window = (limit > 0 && count > limit) ? limit : count;
    start = count - window;
}

}  // namespace mrml
