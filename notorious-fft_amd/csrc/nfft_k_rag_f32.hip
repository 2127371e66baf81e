// nfft_k_rag_f32.hip -- kernels of ragged batches, FP32
#include "nfft_kernels_mix.h"

namespace nfft {
template __global__ void k_rag_group<float, false>(RagArgs);
template __global__ void k_rag_group<float, true>(RagArgs);
template __global__ void k_rag_tile<float>(RagArgs);
}  // namespace nfft
