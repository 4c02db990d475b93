// Instances of the fused wave-list scan that abandon tiles, fp16 tables, m = 48.
#include "fused_wave.inl"

namespace vk {
WaveScanKernel abandon_kernel_h48(int q, int threads, bool vote) {
    return select_abandon_kernel<48, true>(q, threads, vote);
}
}  // namespace vk
