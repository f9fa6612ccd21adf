// The PME grid's forward FFT, convolution and inverse FFT in FP64.
#include "pmx_fft.h"

namespace pmx {

hipError_t launch_pme_fft64(const FftArgs &f, hipStream_t st) { return launch_fft_t<double>(f, st); }

}  // namespace pmx
