// nfft_k_mix_f64.hip -- one-pass mixed-radix lines, FP64
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_mix_line<double, false>(MixArgs);
template __global__ void k_mix_line<double, true>(MixArgs);
}  // namespace nfft
