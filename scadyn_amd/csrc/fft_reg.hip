// Two-stage register line FFT, complex128.
#include "fft_reg_kernel.hpp"

namespace scadyn {

bool reg_radix_ok(int r) {
    switch (r) {
#define OK(R) case R:
        REG_RADICES(OK)
#undef OK
        return true;
        default: return false;
    }
}

template void launch_line_reg<cd>(const LinePass &, const cd *, cd *, const cd *, int, const cd *, const ConvInfo &,
                                  int, hipStream_t);

}  // namespace scadyn
