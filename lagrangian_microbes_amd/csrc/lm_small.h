// Small populations: one workgroup of 16 wavefronts holds a whole step in its
// LDS (lm_pairs.hip, lm_rps.hip), so a batch takes one launch per phase where
// the general path takes about twenty-five.
#pragma once

#include "lm_common.h"
#include "lm_scan.h"

namespace lm {

constexpr int kSmallBlock = 1024;
// Positions, indices and a bucket table of this many particles fill a CU's
// 160 KB of LDS.
constexpr int64_t kSmallMax = 12288;

// Workgroup-wide exclusive scan over kSmallBlock threads; *total gets the sum.
__device__ inline uint32_t small_exclusive_scan(uint32_t x, uint32_t* lds /* >= 16 */, uint32_t* total) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t inc = wave_inclusive_scan(x);
    __syncthreads();
    if (lane == 63) lds[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kSmallBlock / 64; ++w) {
        const uint32_t v = lds[w];
        before += w < wave ? v : 0u;
        all += v;
    }
    *total = all;
    return before + inc - x;
}

// In-place exclusive scan of v[0 .. count) in LDS, `per` consecutive entries
// per thread; every thread must call it.
__device__ inline void small_scan_array(uint32_t* v, uint32_t count, uint32_t* lds) {
    const uint32_t per = (count + kSmallBlock - 1) / kSmallBlock;
    const uint32_t a = min(threadIdx.x * per, count), b = min(a + per, count);
    uint32_t sum = 0, all;
    for (uint32_t k = a; k < b; ++k) sum += v[k];
    uint32_t acc = small_exclusive_scan(sum, lds, &all);
    for (uint32_t k = a; k < b; ++k) {
        const uint32_t c = v[k];
        v[k] = acc;
        acc += c;
    }
    __syncthreads();
}

}  // namespace lm
