// Document starts of packed rows from their position ids: out[b][i] = index of the last token at or before i whose position
// does not follow its predecessor's by one (the convention transformers detects packing by, masking_utils.py:728-757).
//
// What bounds it: latency.  A row is a few thousand integers; written with tensor operations it was nine launches (55 us at
// 8192 tokens, half of it one scan over the row).  A workgroup takes 1024 tokens: their own boundaries by a maximum
// scan in registers and LDS, and what reaches into them from the left by looking backwards, 1024 tokens at a time, until
// the first boundary (a document's length away).  One launch, 5.5 us.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gptoss {

constexpr int kDocTokens = 1024;      // tokens per workgroup, four per thread

template <typename T>
__global__ __launch_bounds__(256) void doc_start_kernel(const T *pos, int64_t row_stride, int S, int32_t *out) {
    __shared__ int wave_max[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const T *row = pos + (int64_t)blockIdx.y * row_stride;
    // the largest boundary among the four tokens from i0 on, -1 without one (own[k]: up to token k)
    auto boundaries = [&](int i0, int (&own)[4]) __attribute__((always_inline)) {
        T p[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const int i = i0 - 1 + k;
            p[k] = i >= 0 && i < S ? row[i] : T(0);
        }
        int last = -1;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = i0 + k;
            if (i < S && (i == 0 || p[k + 1] - p[k] != T(1))) last = i;
            own[k] = last;
        }
        return last;
    };
    auto block_max = [&](int x) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) x = max(x, __shfl_xor(x, d));
        __syncthreads();
        if (lane == 0) wave_max[w] = x;
        __syncthreads();
        return max(max(wave_max[0], wave_max[1]), max(wave_max[2], wave_max[3]));
    };
    const int base = blockIdx.x * kDocTokens;
    int left = -1, own[4];
    for (int b0 = base - kDocTokens; b0 >= 0 && left < 0; b0 -= kDocTokens) left = block_max(boundaries(b0 + 4 * tid, own));
    int scan = boundaries(base + 4 * tid, own);
    // exclusive maximum over the threads before this one
    int incl = scan;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(incl, d);
        if (lane >= d) incl = max(incl, y);
    }
    __syncthreads();
    if (lane == 63) wave_max[w] = incl;
    __syncthreads();
    int before = __shfl_up(incl, 1);
    before = max(left, lane == 0 ? -1 : before);
    for (int k = 0; k < w; ++k) before = max(before, wave_max[k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int i = base + 4 * tid + k;
        if (i < S) out[(int64_t)blockIdx.y * S + i] = max(before, own[k]);
    }
}

}  // namespace gptoss
