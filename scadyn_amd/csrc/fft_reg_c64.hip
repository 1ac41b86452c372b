// Two-stage register line FFT, complex64.
#include "fft_reg_kernel.hpp"

namespace scadyn {

template void launch_line_reg<cf>(const LinePass &, const cf *, cf *, const cf *, int, const cf *, const ConvInfo &,
                                  int, hipStream_t);

}  // namespace scadyn
