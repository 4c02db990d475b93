// Instances of the fused wave-list scan that abandon tiles, fp32 tables, m = 48.
#include "fused_wave.inl"

namespace vk {
WaveScanKernel abandon_kernel_m48(int q, int threads, bool vote) {
    return select_abandon_kernel<48, false>(q, threads, vote);
}
}  // namespace vk
