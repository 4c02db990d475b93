// Nearest-centroid assignment on the GPU: the PQ encoder and the assignment step of k-means training (reference
// ProductQuantizer::encode / train, pq.cpp:11-22, 31-76). For sub-vector x of sub-space s it returns the first c
// in 0..255 with the smallest l2sq(x, C[s][c]), scanning c in order from a best distance of FLT_MAX exactly as
// nearest_centroid does, with l2sq's dimension order and separate multiply and add, so codes are identical to the
// CPU's, ties included.
//
// Sub-vector widths with an instance below go through the matrix cores as a filter: |c|^2 - 2 x.c of every centroid
// from bf16 products, the two smallest of them per vector, and a bound on the error of both the products and the
// exact fp32 sums. Where the gap between the two exceeds the bound, the smallest is the exact arithmetic's only
// minimum; the other vectors (about one in a hundred; ties, NaN, infinities and extreme magnitudes among them) are
// compared with all 256 centroids in the exact arithmetic. Every other width takes the exact comparison directly, and so do small inputs of two dimensions per sub-space.
#include <cfloat>

#include "kernels.hpp"

namespace vk {

namespace {

constexpr int kAssignThreads = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// min(a, b) in one instruction (fminf first quietens operands that come from integer operations).
__device__ __forceinline__ float min_bits(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Any width: one lane per (vector, sub-space), a block's lanes on one sub-space (grid y).
__global__ void __launch_bounds__(kAssignThreads) nearest_kernel(NearestArgs a) {
#pragma clang fp contract(off)
    const int s = blockIdx.y;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kAssignThreads + threadIdx.x;
    if (i >= a.n) return;
    const int dsub = a.dsub;
    const float* xr = a.x + i * a.x_stride + static_cast<int64_t>(s) * dsub;
    const float* cent = a.centroids + static_cast<int64_t>(s) * KSUB * dsub;
    int best = 0;
    float best_dist = FLT_MAX;
    for (int c = 0; c < KSUB; ++c) {
        float acc = 0.f;
        for (int j = 0; j < dsub; ++j) {
            const float diff = xr[j] - cent[c * dsub + j];
            acc += diff * diff;
        }
        if (acc < best_dist) {
            best_dist = acc;
            best = c;
        }
    }
    if (a.codes) a.codes[i * a.m + s] = static_cast<uint8_t>(best);
    if (a.assign) a.assign[i] = static_cast<uint32_t>(best);
}

// The exact comparison of one vector per lane with the sub-space's codebook in LDS, centroids in order: every lane reads
// the same centroid at the same time (an LDS broadcast, 16-byte reads when DSUB % 4 == 0).
template <int DSUB>
__device__ __forceinline__ int nearest_of_all(const float (&x)[DSUB], const float* cent) {
#pragma clang fp contract(off)
    int best = 0;
    float best_dist = FLT_MAX;
    for (int c = 0; c < KSUB; ++c) {
        float cv[DSUB];
        if constexpr (DSUB % 4 == 0) {
#pragma unroll
            for (int e = 0; e < DSUB; e += 4)
                *reinterpret_cast<f32x4*>(cv + e) = *reinterpret_cast<const f32x4*>(cent + c * DSUB + e);
        } else {
#pragma unroll
            for (int e = 0; e < DSUB; ++e) cv[e] = cent[c * DSUB + e];
        }
        float acc = 0.f;
#pragma unroll
        for (int e = 0; e < DSUB; ++e) {
            const float diff = x[e] - cv[e];
            acc += diff * diff;
        }
        if (acc < best_dist) {
            best_dist = acc;
            best = c;
        }
    }
    return best;
}

// The exact comparison alone, for the width and sizes where the filter does not earn back the splitting of the codebook
// (launch_nearest): a block stages one sub-space's codebook (grid y) and each lane takes a vector.
template <int DSUB>
__global__ void __launch_bounds__(kAssignThreads) nearest_exact_kernel(NearestArgs a) {
    __shared__ __align__(16) float cent[KSUB * DSUB];
    const int s = blockIdx.y;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kAssignThreads + threadIdx.x;
    const float* src = a.centroids + static_cast<int64_t>(s) * KSUB * DSUB;
    for (int e = threadIdx.x; e < KSUB * DSUB; e += kAssignThreads) cent[e] = src[e];
    const float* xr = a.x + min<int64_t>(i, a.n - 1) * a.x_stride + static_cast<int64_t>(s) * DSUB;
    float x[DSUB];
#pragma unroll
    for (int e = 0; e < DSUB; ++e) x[e] = xr[e];
    __syncthreads();
    const int best = nearest_of_all<DSUB>(x, cent);
    if (i >= a.n) return;
    if (a.codes) a.codes[i * a.m + s] = static_cast<uint8_t>(best);
    if (a.assign) a.assign[i] = static_cast<uint32_t>(best);
}

// The filtered form. A block takes one sub-space and `chunk` vectors; a wave takes 64 vectors at a time as four
// groups of 16 columns against 16 tiles of 16 centroids.
//
// Products. Both sides are first moved by the mean of a few centroids, x = x_in - mean and c = c_in - mean (rounded), so that
// the error bound follows the spread of the data and not its distance from the origin. x' = -2x and c are split into two
// bf16 parts each, x' = xh + xm + rest with |rest| <= 2^-17 |x'|; the
// four kinds of part products fill the K = 32 of one v_mfma_f32_16x16x32_bf16 for 8 dimensions: the lanes of k-group
// g (lane / 16) hold part g & 1 of the centroid and part g >> 1 of the vector, and the accumulators start at |c|^2.
// A lane ends up with the values of 64 centroids (tile t, row 4 g + i) for its column, and keeps the two smallest.
// The value's low 6 bits are replaced by 4 t + i, so the minimum carries its index: three VALU operations per value
// (and-or, med3, min) against 3 * dsub + 3 for the exact comparison.
//
// Error bound, with X = |x|, C = the largest |c| of the sub-space: the splits drop at most 2 * 2^-17 of X C each way
// on 2 x.c (2^-15 X C together), the accumulation of NK * 32 products and |c|^2 errs by at most 2^-23 NK 32 times
// the sum of their magnitudes (2^-16 X C + 2^-17 C^2 at NK = 2), the index bits 2^-17 of the value. Exact sums err by
// at most (dsub + 3) 2^-24 of the distance, at most (X + C)^2; rounding x and c moves x - c by at most 2^-24 (X + C),
// the distance by 2^-23 (X + C)^2. The gap must exceed both values' errors.
//
// Vectors whose two smallest values are closer than that are compared exactly: one at a time by the whole wave where a step
// of 64 has few of them (about one in a hundred on the mixture), otherwise each by its own lane, all 64 at once. A
// codebook with repeated centroids, or data with many ties, leaves most vectors undecided; a wave whose step had more
// than kMostUndecided then leaves the filter out for the rest of its chunk, since it would cost more than it saves.
// 500k vectors of 128 dimensions, m = 64: 1167 us, the exact comparison alone 1317; every centroid twice 1315 (4380 without
// that rule). All values moved by 20 per dimension: 1167, without the mean 4080 (m = 16: 353, 725).
//
// What bounds it: the VALU work per value (at 1M x d128, m = 16: 4.1e9 values; 680 us, the exact comparison of every
// centroid took 1850).
// Blocks of the same vectors and consecutive sub-spaces run on the same XCD (block b runs on XCD b % 8), so that a
// 128-byte line of x, which holds several sub-spaces, is read into one L2 once.
constexpr int kXcds = 8;

// Centroids whose mean both sides are moved by (any point near the codebook does).
constexpr int kMeanOf = 4;

// Undecided vectors of 64 from which comparing all of them exactly, a lane each, costs no more than the filter and the
// comparisons one at a time. Measured at 500k vectors of 128 (96) dimensions, us: filter / exact, all / one at a time,
// all: dsub 2 1150 / 1360 / 3220, dsub 3 600 / 945 / 1650, dsub 4 610 / 1130 / 1730, dsub 8 365 / 985 / 1385, dsub 12
// 240 / 783 / 850, dsub 16 517 / 1880 / 2420.
template <int DSUB>
constexpr int kMostUndecided = DSUB <= 2 ? 6 : DSUB == 3 ? 14 : DSUB == 4 ? 18 : DSUB == 12 ? 38 : 28;

template <int DSUB>
__global__ void __launch_bounds__(kAssignThreads) nearest_filter_kernel(NearestArgs a, int chunk) {
#pragma clang fp contract(off)
    constexpr int NK = (DSUB + 7) / 8;  // K steps of 8 dimensions (the last one zero-padded)
    constexpr int G = 4;                // groups of 16 vectors per wave
    __shared__ bf16x8 split[NK][2][KSUB];
    __shared__ __align__(16) float norm[KSUB];
    __shared__ __align__(16) float cent[KSUB * DSUB];
    __shared__ unsigned cmax_bits;
    const int tid = threadIdx.x, lane = __lane_id(), col = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int64_t j = blockIdx.x / kXcds;
    const int s = static_cast<int>(j % a.m);
    const int64_t first = ((j / a.m) * kXcds + blockIdx.x % kXcds) * chunk;
    if (first >= a.n) return;  // block-uniform
    const int64_t last = min<int64_t>(a.n, first + chunk);

    if (tid == 0) cmax_bits = 0u;
    const float* const book = a.centroids + static_cast<int64_t>(s) * KSUB * DSUB;
    float mu[DSUB];
#pragma unroll
    for (int e = 0; e < DSUB; ++e) {
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < kMeanOf; ++r) sum += book[r * (KSUB / kMeanOf) * DSUB + e];
        mu[e] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sum * (1.f / kMeanOf))));
    }
    {
        const float* src = book + tid * DSUB;
        float sum = 0.f;
        bf16x8 hi[NK], mid[NK];
#pragma unroll
        for (int e = 0; e < NK * 8; ++e) {
            float v = 0.f;
            if (e < DSUB) {
                cent[tid * DSUB + e] = src[e];
                v = src[e] - mu[e];
            }
            sum += v * v;
            const __bf16 h = static_cast<__bf16>(v);
            hi[e / 8][e % 8] = h;
            mid[e / 8][e % 8] = static_cast<__bf16>(v - static_cast<float>(h));
        }
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            split[k][0][tid] = hi[k];
            split[k][1][tid] = mid[k];
        }
        norm[tid] = sum;
        __syncthreads();
        atomicMax(&cmax_bits, __float_as_uint(sum) & 0x7fffffffu);  // norms are >= 0; a NaN norm is the largest
        __syncthreads();
    }
    const float c2 = __uint_as_float(cmax_bits);
    const float cn = sqrtf(c2) * 1.0001f;
    constexpr float kHuge = 0x1p80f, kTiny = 0x1p-80f;  // squares whose products stay far from overflow and underflow

    bool filter = true;  // wave-uniform
    for (int64_t v0 = first + wave * WAVE; v0 < last; v0 += kAssignThreads) {  // wave-uniform, no barrier inside
        uint64_t redo = ~uint64_t{0};  // bit l: vector v0 + l takes the exact comparison
        int code = 0;                  // lane l: the code of vector v0 + l
        if (filter) {
            bf16x8 b[G][NK];
            float x2[G], m1[G], m2[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int64_t i = min<int64_t>(v0 + g * 16 + col, a.n - 1);
                const float* xr = a.x + i * a.x_stride + static_cast<int64_t>(s) * DSUB;
                float sum = 0.f;
#pragma unroll
                for (int e = 0; e < NK * 8; ++e) {
                    const float v = e < DSUB ? xr[e] - mu[e] : 0.f;
                    sum += v * v;
                    const float w = -2.f * v;
                    const __bf16 h = static_cast<__bf16>(w);
                    const __bf16 mid = static_cast<__bf16>(w - static_cast<float>(h));
                    b[g][e / 8][e % 8] = kg >= 2 ? mid : h;
                }
                x2[g] = sum;
                m1[g] = INFINITY;
                m2[g] = INFINITY;
            }
#pragma unroll
            for (int t = 0; t < KSUB / 16; ++t) {
                const f32x4 nv = *reinterpret_cast<const f32x4*>(&norm[t * 16 + 4 * kg]);
                bf16x8 av[NK];
#pragma unroll
                for (int k = 0; k < NK; ++k) av[k] = split[k][kg & 1][t * 16 + col];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    f32x4 acc = nv;
#pragma unroll
                    for (int k = 0; k < NK; ++k)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[k], b[g][k], acc, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float key = __uint_as_float((__float_as_uint(acc[r]) & ~63u) | (4 * t + r));
                        m2[g] = __builtin_amdgcn_fmed3f(key, m1[g], m2[g]);
                        m1[g] = min_bits(m1[g], key);
                    }
                }
            }
            redo = 0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int tr = static_cast<int>(__float_as_uint(m1[g]) & 63u);
                int c = (tr >> 2) * 16 + kg * 4 + (tr & 3);
                float lo = m1[g], next = m2[g];
#pragma unroll
                for (int o = 16; o < WAVE; o <<= 1) {  // the column's four lanes
                    const float olo = __shfl_xor(lo, o), onext = __shfl_xor(next, o);
                    const int oc = __shfl_xor(c, o);
                    next = fminf(fminf(next, onext), fmaxf(lo, olo));
                    c = olo < lo ? oc : c;
                    lo = fminf(lo, olo);
                }
                const float xn = sqrtf(x2[g]) * 1.0001f;
                const float reach = (xn + cn) * (xn + cn);
                const float err = 1.25f * (xn * cn * (0x1p-15f + NK * 0x1p-17f) + c2 * (NK * 0x1p-18f) +
                                           fmaxf(fabsf(lo), fabsf(next)) * 0x1p-17f);
                const float tau = 2.f * err + reach * (4 * (DSUB + 5) * 0x1p-24f);
                const bool sure = next - lo > tau && c2 < kHuge && x2[g] < kHuge && reach > kTiny;
                redo |= (__builtin_amdgcn_ballot_w64(!sure) & 0xffffu) << (16 * g);
                code = kg == g ? c : code;
            }
        }
        const int64_t i = v0 + lane;
        if (last - v0 < WAVE) redo &= (uint64_t{1} << (last - v0)) - 1;
        if (__popcll(redo) > kMostUndecided<DSUB>) {  // wave-uniform: each lane its vector, centroids in order
            filter = false;
            const float* xr = a.x + min<int64_t>(i, last - 1) * a.x_stride + static_cast<int64_t>(s) * DSUB;
            float xv[DSUB];
#pragma unroll
            for (int e = 0; e < DSUB; ++e) xv[e] = xr[e];
            code = nearest_of_all<DSUB>(xv, cent);
            redo = 0;
        }
        while (redo) {  // wave-uniform: lane l compares centroids l, l + 64, l + 128, l + 192
            const int v = __ffsll(static_cast<unsigned long long>(redo)) - 1;
            redo &= redo - 1;
            const float* xr = a.x + (v0 + v) * a.x_stride + static_cast<int64_t>(s) * DSUB;
            float xv[DSUB];
#pragma unroll
            for (int e = 0; e < DSUB; ++e) xv[e] = xr[e];
            uint64_t best = uint64_t{__float_as_uint(FLT_MAX)} << 32;  // (distance bits, centroid); distances are >= 0
#pragma unroll
            for (int r = 0; r < KSUB / WAVE; ++r) {
                const int c = r * WAVE + lane;
                float acc = 0.f;
#pragma unroll
                for (int e = 0; e < DSUB; ++e) {
                    const float diff = xv[e] - cent[c * DSUB + e];
                    acc += diff * diff;
                }
                const uint64_t key = (uint64_t{__float_as_uint(acc)} << 32) | static_cast<unsigned>(c);
                if (acc < FLT_MAX && key < best) best = key;
            }
            auto nearer = [&](auto jc) {
                constexpr int o = decltype(jc)::value;
                const uint64_t other =
                    (static_cast<uint64_t>(static_cast<uint32_t>(xor_lane<o>(static_cast<int>(best >> 32)))) << 32) |
                    static_cast<uint32_t>(xor_lane<o>(static_cast<int>(static_cast<uint32_t>(best))));
                best = other < best ? other : best;
            };
            nearer(std::integral_constant<int, 1>{});
            nearer(std::integral_constant<int, 2>{});
            nearer(std::integral_constant<int, 4>{});
            nearer(std::integral_constant<int, 8>{});
            nearer(std::integral_constant<int, 16>{});
            nearer(std::integral_constant<int, 32>{});
            if (lane == v) code = static_cast<int>(best & 0xffu);
        }
        if (i < last) {
            if (a.codes) a.codes[i * a.m + s] = static_cast<uint8_t>(code);
            if (a.assign) a.assign[i] = static_cast<uint32_t>(code);
        }
    }
}

// Two-dimensional sub-vectors: the exact comparison takes 9 VALU operations per value against the filter's 3, and the
// filter's set-up is paid back from about this many codes (exact / filter, us: m = 64, 30k vectors 99 / 108, 100k 303 /
// 272, 1M 2770 / 2420; m = 1, 1M vectors 56 / 66).
constexpr int64_t kFilterPairs = int64_t{1} << 22;

template <int DSUB>
hipError_t launch_filter(const NearestArgs& a, hipStream_t stream) {
    // Vectors per block: 2048 or 1024 where that still gives every CU many blocks, fewer for small inputs (a block first
    // splits its codebook, so it takes at least one pass of its four waves).
    int64_t chunk = 2048;
    while (chunk > kAssignThreads && (a.n + chunk - 1) / chunk * a.m < 4096) chunk /= 2;
    auto blocks_of = [&](int64_t vectors) {
        return ((a.n + vectors - 1) / vectors + kXcds - 1) / kXcds * kXcds * static_cast<int64_t>(a.m);
    };
    // A launch dimension holds fewer than 2^32 threads.
    while (blocks_of(chunk) * kAssignThreads >= int64_t{1} << 31 && chunk < int64_t{1} << 30) chunk *= 2;
    const int64_t blocks = blocks_of(chunk);
    if (blocks * kAssignThreads >= int64_t{1} << 31) return hipErrorInvalidValue;
    hipLaunchKernelGGL(nearest_filter_kernel<DSUB>, dim3(static_cast<unsigned>(blocks)), dim3(kAssignThreads), 0, stream,
                       a, static_cast<int>(chunk));
    return hipGetLastError();
}

}  // namespace

hipError_t launch_nearest(const NearestArgs& a, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((a.n + kAssignThreads - 1) / kAssignThreads), static_cast<unsigned>(a.m));
    if (a.dsub == 2 && a.n * a.m < kFilterPairs) {
        hipLaunchKernelGGL(nearest_exact_kernel<2>, grid, dim3(kAssignThreads), 0, stream, a);
        return hipGetLastError();
    }
    switch (a.dsub) {
        case 2: return launch_filter<2>(a, stream);
        case 3: return launch_filter<3>(a, stream);
        case 4: return launch_filter<4>(a, stream);
        case 6: return launch_filter<6>(a, stream);
        case 8: return launch_filter<8>(a, stream);
        case 12: return launch_filter<12>(a, stream);
        case 16: return launch_filter<16>(a, stream);
        default: break;
    }
    hipLaunchKernelGGL(nearest_kernel, grid, dim3(kAssignThreads), 0, stream, a);
    return hipGetLastError();
}

}  // namespace vk
