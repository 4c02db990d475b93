// One-time code layout transforms, run on the GPU when a variant first needs them (reference:
// build_interleaved_bytes / build_interleaved_words, searcher.cu:103-119, formulas kernels.cuh:92-94, 238-240).
// Tiles are 64 vectors (one wave64) instead of the reference's 32. Every output element is written once, with
// coalesced stores; the strided row-major reads are a one-off cost.
#include "kernels.hpp"

namespace vk {

__global__ void __launch_bounds__(256)
    build_words_kernel(const uint8_t* __restrict__ codes, int64_t n, int words, int64_t total, uint4* __restrict__ out) {
    for (int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; o < total;
         o += static_cast<int64_t>(gridDim.x) * 256) {
        const int64_t lane = o % WAVE, w = (o / WAVE) % words, tile = o / (static_cast<int64_t>(WAVE) * words);
        const int64_t i = tile * WAVE + lane;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (i < n) v = *reinterpret_cast<const uint4*>(codes + (i * words + w) * 16);
        out[o] = v;
    }
}

__global__ void __launch_bounds__(256)
    build_bytes_kernel(const uint8_t* __restrict__ codes, int64_t n, int m, int64_t total, uint8_t* __restrict__ out) {
    for (int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; o < total;
         o += static_cast<int64_t>(gridDim.x) * 256) {
        const int64_t lane = o % WAVE, s = (o / WAVE) % m, tile = o / (static_cast<int64_t>(WAVE) * m);
        const int64_t i = tile * WAVE + lane;
        out[o] = i < n ? codes[i * m + s] : 0;
    }
}

static int layout_grid(int64_t total) {
    const int64_t blocks = (total + 255) / 256;
    return static_cast<int>(blocks < 4096 ? (blocks > 0 ? blocks : 1) : 4096);
}

hipError_t launch_build_words(const uint8_t* codes, int64_t n, int m, int64_t n_pad, uint4* out, hipStream_t stream) {
    const int words = m / 16;
    const int64_t total = n_pad * words;  // uint4 elements
    hipLaunchKernelGGL(build_words_kernel, dim3(layout_grid(total)), dim3(256), 0, stream, codes, n, words, total, out);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256)
    build_sorted_words_kernel(const uint8_t* __restrict__ codes, int64_t n, int words, int64_t total,
                              const uint32_t* __restrict__ slot_ids, const uint8_t* __restrict__ rows,
                              uint4* __restrict__ out) {
    for (int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; o < total;
         o += static_cast<int64_t>(gridDim.x) * 256) {
        const int64_t lane = o % WAVE, w = (o / WAVE) % words, tile = o / (static_cast<int64_t>(WAVE) * words);
        const int64_t slot = tile * WAVE + lane;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (slot < n) {
            const int64_t i = slot_ids[(tile >> 2) * 256 + lane * 4 + (tile & 3)];
            if (i < n) v = *reinterpret_cast<const uint4*>(codes + (i * words + w) * 16);  // ids are < n
            if (rows) {  // code byte j of the word (sub-space 16 w + j) -> its table row
                const uint8_t* r = rows + w * 16 * 256;
                uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    uint32_t y = 0;
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        y |= static_cast<uint32_t>(r[(k * 4 + b) * 256 + ((x[k] >> (8 * b)) & 0xffu)]) << (8 * b);
                    x[k] = y;
                }
                v = make_uint4(x[0], x[1], x[2], x[3]);
            }
        }
        out[o] = v;
    }
}

hipError_t launch_build_sorted_words(const uint8_t* codes, int64_t n, int m, int64_t n_pad, const uint32_t* slot_ids,
                                     const uint8_t* rows, uint4* out, hipStream_t stream) {
    const int words = m / 16;
    const int64_t total = n_pad * words;
    hipLaunchKernelGGL(build_sorted_words_kernel, dim3(layout_grid(total)), dim3(256), 0, stream, codes, n, words, total,
                       slot_ids, rows, out);
    return hipGetLastError();
}

hipError_t launch_build_bytes(const uint8_t* codes, int64_t n, int m, int64_t n_pad, uint8_t* out,
                              hipStream_t stream) {
    const int64_t total = n_pad * m;
    hipLaunchKernelGGL(build_bytes_kernel, dim3(layout_grid(total)), dim3(256), 0, stream, codes, n, m, total, out);
    return hipGetLastError();
}

// Sets count words to zero with vector stores (used where a hipMemsetAsync node is unwanted, e.g. in work a
// caller may capture into a graph).
__global__ void __launch_bounds__(256) zero_words_kernel(unsigned* __restrict__ p, int64_t count) {
    for (int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; o < count;
         o += static_cast<int64_t>(gridDim.x) * 256)
        p[o] = 0u;
}

hipError_t launch_zero_words(unsigned* p, int64_t count, hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_words_kernel, dim3(layout_grid(count)), dim3(256), 0, stream, p, count);
    return hipGetLastError();
}

namespace {

__global__ void build_heads_kernel(const uint32_t* words, int m, int64_t granules, int head_words, uint4* out) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;  // (granule, h, lane)
    if (e >= granules * head_words * WAVE) return;
    const int lane = static_cast<int>(e % WAVE), h = static_cast<int>(e / WAVE % head_words);
    const int64_t tile0 = e / WAVE / head_words * 4;
    auto part = [&](int u) {
        return words[(((tile0 + u) * (m / 16) + h / 4) * WAVE + lane) * 4 + h % 4];
    };
    out[e] = make_uint4(part(0), part(1), part(2), part(3));
}

// One block per sampled tile of the slot order and four sub-spaces past the sort key (grid y): squared distances between the
// codewords of neighbouring lanes' vectors, and of each lane's vector and one half the database away.
__global__ void __launch_bounds__(WAVE)
    tile_spread_kernel(const uint8_t* codes, const uint32_t* slot_ids, const float* centroids, int m, int dsub,
                       int64_t tiles, int64_t stride, double* sums) {
    const int64_t tile = static_cast<int64_t>(blockIdx.x) * stride, far_tile = (tile + tiles / 2) % tiles;
    const int lane = threadIdx.x;
    auto row = [&](int64_t t, int l) {
        return codes + static_cast<int64_t>(slot_ids[(t >> 2) * 256 + l * 4 + (t & 3)]) * m;
    };
    const uint8_t* const own = row(tile, lane);
    const uint8_t* const next = row(tile, lane ^ 1);
    const uint8_t* const other = row(far_tile, lane);
    float close = 0.f, apart = 0.f;
    const int s0 = 4 + 4 * static_cast<int>(blockIdx.y);
    for (int s = s0; s < m && s < s0 + 4; ++s) {
        const float* c = centroids + static_cast<int64_t>(s) * KSUB * dsub;
        for (int j = 0; j < dsub; ++j) {
            const float x = c[own[s] * dsub + j], dn = x - c[next[s] * dsub + j], df = x - c[other[s] * dsub + j];
            close += dn * dn;
            apart += df * df;
        }
    }
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        close += __shfl_xor(close, o);
        apart += __shfl_xor(apart, o);
    }
    if (lane == 0) {
        atomicAdd(&sums[0], static_cast<double>(close));
        atomicAdd(&sums[1], static_cast<double>(apart));
    }
}

}  // namespace

hipError_t launch_build_heads(const uint4* words, int m, int64_t n_pad, int head_words, uint4* out,
                              hipStream_t stream) {
    const int64_t granules = n_pad / 256, threads = granules * head_words * WAVE;
    hipLaunchKernelGGL(build_heads_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, stream,
                       reinterpret_cast<const uint32_t*>(words), m, granules, head_words, out);
    return hipGetLastError();
}

hipError_t launch_tile_spread(const uint8_t* codes, const uint32_t* slot_ids, const float* centroids, int m, int dsub,
                              int64_t tiles, int64_t stride, double* sums, hipStream_t stream) {
    const int64_t blocks = (tiles + stride - 1) / stride;
    if (blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(tile_spread_kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>((m - 1) / 4)),
                       dim3(WAVE), 0, stream, codes, slot_ids, centroids, m, dsub, tiles, stride, sums);
    return hipGetLastError();
}

}  // namespace vk
