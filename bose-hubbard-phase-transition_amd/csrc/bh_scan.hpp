// bh_scan.hpp -- block-level scan helper shared by the basis and Hamiltonian builders.
#pragma once

#include "bh_internal.hpp"

// Exclusive scan of a wave64 block of BLOCK threads.  lds must hold BLOCK/64 + 1 values.
template <int BLOCK>
__device__ __forceinline__ int64_t bh_block_exclusive_scan(int64_t v, int64_t* lds, int64_t* total) {
    const int lane = threadIdx.x & 63;
    const int wid = threadIdx.x >> 6;
    int64_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t run = 0;
        for (int w = 0; w < BLOCK / 64; ++w) {
            int64_t t = lds[w];
            lds[w] = run;
            run += t;
        }
        lds[BLOCK / 64] = run;
    }
    __syncthreads();
    const int64_t res = lds[wid] + x - v;
    if (total) *total = lds[BLOCK / 64];
    __syncthreads();
    return res;
}
