// Instances of the fused wave-list scan for m = 48.
#include "fused_wave.inl"

namespace vk {
WaveScanKernel fused_wave_kernel_m48(int qg, int ng, int ilp, int segments, bool bulk, int threads) {
    return select_wave_kernel<48, false>(qg, ng, ilp, segments, bulk, threads);
}
}  // namespace vk
