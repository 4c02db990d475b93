// Instances of the fused wave-list scan that abandon tiles, fp32 tables, m = 64.
#include "fused_wave.inl"

namespace vk {
WaveScanKernel abandon_kernel_m64(int q, int threads, bool vote) {
    return select_abandon_kernel<64, false>(q, threads, vote);
}
}  // namespace vk
