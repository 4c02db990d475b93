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
// process: a lane that reads its own row touches a line of its own with every load, 64 lines per instruction. The
// rows therefore come in 32-float slices that consecutive lanes read together (8 lanes per 128-byte slice of a row)
// and go through LDS to the lane that sums them, with the next slice's loads in flight meanwhile (1000 queries x 100
// candidates, d = 128: 50.8 us per call with one wave per query reading rows lane by lane, 45.7 so).
#include <type_traits>

#include "kernels.hpp"

namespace vk {

namespace {

constexpr int kSliceFloats = 32;
constexpr int kMaxRerankWaves = 8;
constexpr int kSliceBytes = WAVE * kSliceFloats * 4;  // LDS per wave

// One wave's slices of its 64 rows. VEC4: 16-byte loads (d % 4 == 0: rows are 16-byte aligned); otherwise 4-byte.
// LDS holds row-major 16-byte chunks, chunk c of row r at r * 8 + (c ^ ((r >> 1) & 7)): the 16 lanes that read the
// same chunk of 16 consecutive rows in one pass then fall on all 16 bank groups.
template <bool VEC4>
struct SliceLoader {
    static constexpr int kLoads = VEC4 ? 8 : 32;
    using T = std::conditional_t<VEC4, float4, float>;
    T v[kLoads];

    __device__ __forceinline__ void load(const float* base, int d, int32_t id, bool use, int first, int lane) {
        constexpr int kLanesPerRow = VEC4 ? 8 : 32, kRows = WAVE / kLanesPerRow, kWidth = VEC4 ? 4 : 1;
        const int at = first + (lane % kLanesPerRow) * kWidth;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int row = i * kRows + lane / kLanesPerRow;
            const int32_t rid = __shfl(use ? id : -1, row);
            T x{};
            if (rid >= 0 && at < d) x = *reinterpret_cast<const T*>(base + static_cast<int64_t>(rid) * d + at);
            v[i] = x;
        }
    }
    __device__ __forceinline__ void store(float* lds, int lane) const {
        constexpr int kLanesPerRow = VEC4 ? 8 : 32, kRows = WAVE / kLanesPerRow;
        const int c = lane % kLanesPerRow;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int row = i * kRows + lane / kLanesPerRow;
            if constexpr (VEC4) {
                *reinterpret_cast<float4*>(lds + (row * 8 + (c ^ ((row >> 1) & 7))) * 4) = v[i];
            } else {
                lds[(row * 8 + ((c >> 2) ^ ((row >> 1) & 7))) * 4 + (c & 3)] = v[i];
            }
        }
    }
};

__device__ __forceinline__ void wave_lds_fence() {  // LDS written by other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int S, bool VEC4>
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
        SliceLoader<VEC4> next;
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
                    if (c * 4 + 1 < width) add(xs[1], v.y);
                    if (c * 4 + 2 < width) add(xs[2], v.z);
                    if (c * 4 + 3 < width) add(xs[3], v.w);
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
    const size_t lds = static_cast<size_t>(waves) * kSliceBytes;  // also holds the wave lists (K <= 128 pairs a wave)
    static_assert(2 * WAVE * sizeof(Pair) <= kSliceBytes, "a wave's list fits its slice buffer");
    const bool vec4 = a.d % 4 == 0 && reinterpret_cast<uintptr_t>(a.base) % 16 == 0;
    for (int64_t q0 = 0; q0 < a.nq; q0 += kMaxBlocks) {
        RerankArgs b = a;
        b.nq = a.nq - q0 < kMaxBlocks ? a.nq - q0 : kMaxBlocks;
        b.queries = a.queries + q0 * a.d;
        if (a.candidates) b.candidates = a.candidates + q0 * a.r;
        b.out = a.out + q0 * a.k;
        const dim3 grid(static_cast<unsigned>(b.nq));
        if (a.K <= WAVE) {
            if (vec4) hipLaunchKernelGGL((rerank_kernel<1, true>), grid, threads, lds, stream, b);
            else hipLaunchKernelGGL((rerank_kernel<1, false>), grid, threads, lds, stream, b);
        } else {
            if (vec4) hipLaunchKernelGGL((rerank_kernel<2, true>), grid, threads, lds, stream, b);
            else hipLaunchKernelGGL((rerank_kernel<2, false>), grid, threads, lds, stream, b);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace vk
