// nfft_k_mix_f32.hip -- one-pass mixed-radix lines, FP32
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_mix_line<float, false>(MixArgs);
template __global__ void k_mix_line<float, true>(MixArgs);
}  // namespace nfft
