// Exact re-ranking of search candidates on the GPU: the step after the PQ search (reference rerank_exact,
// cpu_ref.cpp:66-77, used by bench --rerank, bench_main.cpp:145-153). For each query, the full-precision squared
// L2 distance to each candidate's base vector, then the k smallest by (dist, id).
//
// One block per query, one wave per 64 candidates (at most eight waves, which then take several rounds). A lane sums
// its candidate's distance alone, in dimension order j = 0..d-1 with a separate multiply and add, exactly like l2sq
// (common.hpp:27-34), so distances are bit-identical to the CPU's; the query's values are wave-uniform scalar loads.
// The wave lists are merged through LDS.
//
// The work is a random gather of r rows of d floats per query, bound by memory latency and by the addresses a CU can
// process. Two ways to read the rows, chosen by launch_rerank:
//  - rows: a lane reads its own row with 16-byte loads, eight in flight;
//  - slices: 32 floats of 64 rows at a time, 8 consecutive lanes on a 128-byte slice of a row, through LDS to the lane that
//    sums them, with the next slice's loads in flight meanwhile. A lane that reads its own row touches a line of its own
//    with every load, 64 lines per instruction, which costs where many rows are read; a slice costs a pass through LDS
//    each, 30 in a row for d = 960.
// us per call over 1M rows that no cache holds, rows / slices: d = 128, 100 x 100 21.8 / 23.3, 1000 x 100 29.3 / 28.6,
// 2000 x 100 39.2 / 37.3, 300 x 300 34.0 / 29.0; d = 96, 2000 x 20 21.1 / 22.5, 1000 x 200 33.8 / 32.0; d = 200, 1000 x 100
// 38.7 / 34.8, 200 x 1000 65.7 / 53.1, one query x 1000 58.6 / 45.7, 2000 x 20 25.1 / 30.3. In the caches: d = 960, 2000 x 10
// 37 / 66, one query x 100 29 / 50, 1000 x 200 147 / 131. Rows that are not 16-byte aligned by 4-byte loads: d = 130, 1000 x
// 100 38.4, by slices of 4-byte loads 52.4. One wave per query reading rows lane by lane: d = 128, 2000 x 100 58.
#include <type_traits>

#include "kernels.hpp"

namespace vk {

namespace {

constexpr int kSliceFloats = 32;
constexpr int kMaxRerankWaves = 8;
constexpr int kSliceBytes = WAVE * kSliceFloats * 4;  // LDS per wave

// One wave's slices of its 64 rows (d % 4 == 0 and an aligned base: 16-byte loads).
// LDS holds row-major 16-byte chunks, chunk c of row r at r * 8 + (c ^ ((r >> 1) & 7)): the 16 lanes that read the
// same chunk of 16 consecutive rows in one pass then fall on all 16 bank groups.
struct SliceLoader {
    static constexpr int kLoads = 8, kLanesPerRow = 8, kRows = WAVE / kLanesPerRow;
    float4 v[kLoads];

    __device__ __forceinline__ void load(const float* base, int d, int32_t id, bool use, int first, int lane) {
        const int at = first + lane % kLanesPerRow * 4;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int32_t rid = __shfl(use ? id : -1, i * kRows + lane / kLanesPerRow);
            float4 x{};
            if (rid >= 0 && at < d) x = *reinterpret_cast<const float4*>(base + static_cast<int64_t>(rid) * d + at);
            v[i] = x;
        }
    }
    __device__ __forceinline__ void store(float* lds, int lane) const {
        const int c = lane % kLanesPerRow;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int row = i * kRows + lane / kLanesPerRow;
            *reinterpret_cast<float4*>(lds + (row * 8 + (c ^ ((row >> 1) & 7))) * 4) = v[i];
        }
    }
};

__device__ __forceinline__ void wave_lds_fence() {  // LDS written by other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The distance of one candidate by its own lane, which reads the row with loads of its own, eight in flight.
template <bool VEC4>
__device__ __forceinline__ float row_distance(const float* x, const float* row, int d) {
#pragma clang fp contract(off)
    float acc = 0.f;
    auto add = [&](float xv, float bv) {
        const float diff = xv - bv;
        acc += diff * diff;
    };
    if constexpr (VEC4) {
#pragma unroll 8
        for (int j = 0; j < d; j += 4) {
            const float4 v = *reinterpret_cast<const float4*>(row + j);
            add(x[j], v.x);
            add(x[j + 1], v.y);
            add(x[j + 2], v.z);
            add(x[j + 3], v.w);
        }
    } else {
#pragma unroll 8
        for (int j = 0; j < d; ++j) add(x[j], row[j]);
    }
    return acc;
}

enum class Read { kFloats, kRows, kSlices };  // a lane's row by 4- or by 16-byte loads, or slices

template <int S, Read READ>
__global__ void __launch_bounds__(kMaxRerankWaves * WAVE) rerank_kernel(RerankArgs a) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int lane = __lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / WAVE);
    const int waves = static_cast<int>(blockDim.x) / WAVE;
    const int64_t q = blockIdx.x;
    const float* x = a.queries + q * a.d;
    const Pair* cand = a.candidates ? a.candidates + q * a.r : nullptr;
    float* const slice = reinterpret_cast<float*>(lds_raw + wave * kSliceBytes);
    WaveList<S, true> list;
    list.init();
    bool bad = false;
    for (int64_t base = static_cast<int64_t>(wave) * WAVE; base < a.r; base += static_cast<int64_t>(waves) * WAVE) {
        const int64_t j = base + lane;
        const int32_t id = j < a.r ? (cand ? cand[j].i : static_cast<int32_t>(j)) : -1;
        bad |= id >= a.n;  // an id past the base: reported, never read
        const bool use = id >= 0 && id < a.n;
        float acc = 0.f;
        if constexpr (READ != Read::kSlices) {
            if (use) acc = row_distance<READ == Read::kRows>(x, a.base + static_cast<int64_t>(id) * a.d, a.d);
        } else {
            SliceLoader next;
            next.load(a.base, a.d, id, use, 0, lane);
            for (int first = 0; first < a.d; first += kSliceFloats) {
                wave_lds_fence();  // the previous slice has been read
                next.store(slice, lane);
                wave_lds_fence();
                if (first + kSliceFloats < a.d) next.load(a.base, a.d, id, use, first + kSliceFloats, lane);
                auto chunk = [&](int c) {
                    return *reinterpret_cast<const float4*>(slice + (lane * 8 + (c ^ ((lane >> 1) & 7))) * 4);
                };
                auto add = [&](float xv, float bv) {
                    const float diff = xv - bv;
                    acc += diff * diff;
                };
                const int width = a.d - first;
                if (width >= kSliceFloats) {
#pragma unroll
                    for (int c = 0; c < kSliceFloats / 4; ++c) {
                        const float4 v = chunk(c);
                        const float* xs = x + first + c * 4;
                        add(xs[0], v.x);
                        add(xs[1], v.y);
                        add(xs[2], v.z);
                        add(xs[3], v.w);
                    }
                } else {
                    for (int c = 0; c * 4 < width; ++c) {
                        const float4 v = chunk(c);
                        const float* xs = x + first + c * 4;
                        add(xs[0], v.x);
                        add(xs[1], v.y);
                        add(xs[2], v.z);
                        add(xs[3], v.w);
                    }
                }
            }
        }
        list.offer(use ? acc : INFINITY, id, use, a.K);
    }
    if (__builtin_amdgcn_ballot_w64(bad) && lane == 0)
        __hip_atomic_store(a.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (waves > 1) {
        __syncthreads();  // every wave has finished with its slices
        Pair* const lists = reinterpret_cast<Pair*>(lds_raw);
        list.store(lists + wave * a.K, a.K);
        __syncthreads();
        if (wave != 0) return;
        list.init();
        stream_partials(list, lists, 0, 1, waves, a.K, lane);
    }
    Pair* out = a.out + q * a.k;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int p = s * WAVE + lane;
        if (p < a.k) out[p] = list.id[s] == kEmptyId ? Pair{INFINITY, -1} : Pair{list.d[s], list.id[s]};
    }
}

}  // namespace

hipError_t launch_rerank(const RerankArgs& a, hipStream_t stream) {
    if (a.K > 2 * WAVE) return hipErrorInvalidValue;
    // A launch dimension holds fewer than 2^32 threads: very many queries go in several launches.
    constexpr int64_t kMaxBlocks = int64_t{1} << 22;
    const int waves = static_cast<int>(a.r < WAVE * kMaxRerankWaves ? (a.r + WAVE - 1) / WAVE : kMaxRerankWaves);
    const dim3 threads(static_cast<unsigned>(waves * WAVE));
    // Slices where a query has many candidates, or more than one wave's and the call gathers 64 MB: there the address
    // processing counts, below it the latency of the slices' passes through LDS.
    const bool vec4 = a.d % 4 == 0 && reinterpret_cast<uintptr_t>(a.base) % 16 == 0;
    const bool slices = vec4 && a.d >= 16 && a.r > WAVE &&
                        (a.r > 4 * WAVE || a.nq >= (int64_t{1} << 24) / (a.r * a.d));
    // The slices' buffers also hold the wave lists (K <= 128 pairs a wave); without slices the lists alone.
    const size_t lds = static_cast<size_t>(waves) * (slices ? kSliceBytes : a.K * sizeof(Pair));
    static_assert(2 * WAVE * sizeof(Pair) <= kSliceBytes, "a wave's list fits its slice buffer");
    for (int64_t q0 = 0; q0 < a.nq; q0 += kMaxBlocks) {
        RerankArgs b = a;
        b.nq = a.nq - q0 < kMaxBlocks ? a.nq - q0 : kMaxBlocks;
        b.queries = a.queries + q0 * a.d;
        if (a.candidates) b.candidates = a.candidates + q0 * a.r;
        b.out = a.out + q0 * a.k;
        const dim3 grid(static_cast<unsigned>(b.nq));
        auto launch = [&](auto sc) {
            constexpr int S = decltype(sc)::value;
            if (slices) hipLaunchKernelGGL((rerank_kernel<S, Read::kSlices>), grid, threads, lds, stream, b);
            else if (vec4) hipLaunchKernelGGL((rerank_kernel<S, Read::kRows>), grid, threads, lds, stream, b);
            else hipLaunchKernelGGL((rerank_kernel<S, Read::kFloats>), grid, threads, lds, stream, b);
        };
        if (a.K <= WAVE) launch(std::integral_constant<int, 1>{});
        else launch(std::integral_constant<int, 2>{});
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace vk
