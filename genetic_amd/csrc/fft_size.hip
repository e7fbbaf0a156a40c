// The passes of one precision and size (GIC_FFT_T, GIC_FFT_N), a unit of its
// own so that the sizes compile side by side.
#include "fft_fused.h"

namespace gic {

template <> const FftApi<GIC_FFT_T> &fft_api<GIC_FFT_T, GIC_FFT_N>() {
  static const FftApi<GIC_FFT_T> a = fft_api_of<GIC_FFT_T, GIC_FFT_N>();
  return a;
}

}  // namespace gic
