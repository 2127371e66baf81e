// nfft_k_mix_f32.hip -- mixed-radix lines and tiles, FP32
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_mix_line<float, false, double2>(MixArgs);
template __global__ void k_mix_line<float, false, float2>(MixArgs);
template __global__ void k_mix_line<float, true, float2>(MixArgs);
template __global__ void k_mix_tile<float, false>(MixTileArgs);
template __global__ void k_mix_tile<float, true>(MixTileArgs);
}  // namespace nfft
