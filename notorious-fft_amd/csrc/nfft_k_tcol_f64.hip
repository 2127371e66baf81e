// nfft_k_tcol_f64.hip -- DCT / DST along strided axes, FP64
#include "nfft_launch_impl.h"
#include "nfft_tcol_impl.h"

namespace nfft {
template hipError_t tcol_impl<double>(int, int, const TrigColArgs &, hipStream_t, bool);
}  // namespace nfft
