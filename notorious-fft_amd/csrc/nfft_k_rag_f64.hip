// nfft_k_rag_f64.hip -- kernels of ragged batches, FP64
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_rag_group<double, false>(RagArgs);
template __global__ void k_rag_group<double, true>(RagArgs);
template __global__ void k_rag_tile<double>(RagArgs);
}  // namespace nfft
