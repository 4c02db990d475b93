// Top-k selection (reference: select_kernel, kernels.cuh:179-202, launched by searcher.cu:285-296).
// One block per query. Each wave streams its share of the candidates into a wave-cooperative sorted list
// (threshold test per candidate, rare inserts), then the four wave lists are merged by rank. Two candidate
// sources share the kernel:
//   mode 0 — a row of n distances, ids are column indices (unfused scans);
//   mode 1 — bx partial K-lists per query laid out [q][bx][K] (per-thread-list fused scans).
// Empty slots ({+inf, INT32_MAX}) are skipped, like the reference skips id < 0, and the output turns any that
// remain into {+inf, -1}.
#include "kernels.hpp"

namespace vk {

template <int S>
__global__ void __launch_bounds__(256) select_kernel(SelectArgs a) {
    constexpr int T = 256, W = T / WAVE;
    __shared__ Pair buf[(W + 1) * WAVE * S];
    const int64_t q = blockIdx.x;
    const int tid = threadIdx.x, lane = __lane_id(), wave = tid / WAVE;
    const int K = a.K;

    WaveList<S, true> list;  // bulk admission: a row's first chunks admit most of their lanes
    list.init();
    if (a.mode == 0) {
        stream_row<S, W>(list, a.dists + q * a.len, a.len, K, wave, lane);
    } else {
        const Pair* first = a.part + q * a.bx * K;
        const int64_t all = a.bx * K;
        for (int64_t base = static_cast<int64_t>(wave) * WAVE; base < all; base += W * WAVE) {
            const int64_t e = base + lane;
            Pair p{INFINITY, kEmptyId};
            if (e < all) p = first[e];
            list.offer(p.d, p.i, p.i != kEmptyId, K);
        }
    }

    Pair* merged = buf + W * K;
    list.store(buf + wave * K, K);
    __syncthreads();
    merge_lists(buf, W, K, merged, tid, T);
    __syncthreads();
    for (int j = tid; j < a.k; j += T) {
        const Pair p = merged[j];
        a.out[q * a.k + j] = p.i == kEmptyId ? Pair{INFINITY, -1} : p;
    }
}

hipError_t launch_select(const SelectArgs& a, int nq, hipStream_t stream) {
    if (a.K <= WAVE) hipLaunchKernelGGL(select_kernel<1>, dim3(nq), dim3(256), 0, stream, a);
    else if (a.K <= 2 * WAVE) hipLaunchKernelGGL(select_kernel<2>, dim3(nq), dim3(256), 0, stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace vk
