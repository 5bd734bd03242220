// wgscan.h -- exclusive scan of a short array by one workgroup of 1024.
#pragma once
#include "wave.h"

namespace lstc {

// put(i, sum of get(0 .. i - 1), get(i)) for every i < n; returns the total.  All
// 1024 threads call it.  What put writes may be what get has read (each round's
// reads come before its writes, and no element is read twice).
template <class Get, class Put>
__device__ __forceinline__ uint64_t wg_scan(uint64_t n, Get get, Put put) {
    __shared__ uint64_t s_w[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint64_t carry = 0;
    for (uint64_t base = 0; base < n; base += 4096) {
        const uint64_t i0 = base + 4 * tid;
        uint64_t v[4], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            v[k] = i0 + k < n ? get(i0 + k) : 0;
            sum += v[k];
        }
        const uint64_t incl = wave_incl_scan64(sum, lane);
        __syncthreads();
        if (lane == 63) s_w[wv] = incl;
        __syncthreads();
        uint64_t run = carry + incl - sum;
        for (uint32_t w = 0; w < 16; ++w) {
            const uint64_t x = s_w[w];
            run += w < wv ? x : 0;
            carry += x;
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            if (i0 + k < n) put(i0 + k, run, v[k]);
            run += v[k];
        }
    }
    return carry;
}

}  // namespace lstc
