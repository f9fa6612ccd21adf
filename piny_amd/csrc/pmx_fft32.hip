// The PME grid's forward FFT, convolution and inverse FFT in FP32.
#include "pmx_fft.h"

namespace pmx {

hipError_t launch_pme_fft32(const FftArgs &f, hipStream_t st) { return launch_fft_t<float>(f, st); }

}  // namespace pmx
