// nfft_k_mix_f64.hip -- mixed-radix lines and tiles, FP64
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_mix_line<double, false, double2>(MixArgs);
template __global__ void k_mix_line<double, true, double2>(MixArgs);
template __global__ void k_mix_tile<double, false>(MixTileArgs);
}  // namespace nfft
