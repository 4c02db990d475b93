// Inverted-list (IVF) instances of the fused wave-list scan for m = 48.
#include "fused_wave.inl"

namespace vk {
WaveScanKernel ivf_kernel_m48(int segments) { return select_ivf_kernel<48>(segments); }
}  // namespace vk
