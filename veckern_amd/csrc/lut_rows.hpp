// One block's share of the plain per-query lookup tables lut[q][s][c] (lut.hip, and the probe of an inverted-file
// search, which builds them in the same launch).
#pragma once

#include "device.hpp"

namespace vk {

// kLutQueries queries q0 .. of sub-space s: thread c reads centroid c of sub-space s once (DSUB
// known at compile time: one or two 16-byte loads) and produces its entry for each of the queries, each store
// coalesced over c. A block per (s, query) would reread the centroid row once per query and leave each thread one entry.
constexpr int kLutQueries = 8;

template <int DSUB>
__device__ __forceinline__ void lut_rows(const float* __restrict__ queries, const float* __restrict__ centroids, int d,
                                         int m, int dsub_rt, int nq, float* __restrict__ lut, int s, int q0, int c) {
#pragma clang fp contract(off)
    const int dsub = DSUB ? DSUB : dsub_rt;
    const float* cent = centroids + (static_cast<size_t>(s) * KSUB + c) * dsub;
    float cv[DSUB ? DSUB : 1];
    if constexpr (DSUB > 0) {
#pragma unroll
        for (int j = 0; j < DSUB; ++j) cv[j] = cent[j];
    }
#pragma unroll
    for (int qq = 0; qq < kLutQueries; ++qq) {
        const int q = q0 + qq;
        if (q >= nq) break;  // block-uniform
        const float* x = queries + static_cast<size_t>(q) * d + static_cast<size_t>(s) * dsub;
        float acc = 0.f;
        if constexpr (DSUB > 0) {
#pragma unroll
            for (int j = 0; j < DSUB; ++j) {
                const float diff = x[j] - cv[j];
                acc += diff * diff;
            }
        } else {
            for (int j = 0; j < dsub; ++j) {
                const float diff = x[j] - cent[j];
                acc += diff * diff;
            }
        }
        lut[(static_cast<size_t>(q) * m + s) * KSUB + c] = acc;
    }
}

}  // namespace vk
