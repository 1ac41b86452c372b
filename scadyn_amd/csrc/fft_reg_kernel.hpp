// Kernel and launcher of the two-stage register line FFT (the algebra and the
// per-thread stages are in fft_reg_core.hpp, shared with the host self-test).
// Included by one translation unit per element type.
#pragma once

#include "fft_reg_core.hpp"

namespace scadyn {
namespace regfft {

__device__ inline size_t wave_uniform(size_t v) {
    return (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v) |
           (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32)) << 32;
}
// split an address into the wave's first lane's and this lane's distance to it
// in bytes (lane 0 has the smallest: items and columns ascend with the lane)
template <typename C>
__device__ inline void wave_base(size_t &base, unsigned &lane) {
    const size_t b = wave_uniform(base);
    lane = (unsigned)((base - b) * sizeof(C));
    base = b;
}

// SH: log2 of the tile width, with 32-bit lane offsets; -1: any width, 64-bit addresses.
// RMAX, the largest radix compiled in, sets the registers and so the waves per SIMD, of
// the any-width instance too: narrow batches run it on the x passes (105 points, 1
// vector, complex128: 18 us with radices up to 20 compiled in, 13 with up to 16)
template <int MODE, typename C, int RMAX, int SH>
__global__ __launch_bounds__(sizeof(C) <= 8 ? 1024 : 512) void k_line_reg(const C *__restrict__ in,
                                                                          C *__restrict__ out, LinePass p,
                                                                          const C *__restrict__ twg, int sign,
                                                                          const C *__restrict__ fg, ConvInfo ci) {
    extern __shared__ char smraw[];
    C *tw = reinterpret_cast<C *>(smraw);
    C *lds = tw + p.L;
    for (int m = threadIdx.x; m < p.L; m += blockDim.x) tw[m] = twg[m];
    // neighbouring tiles of a line row share cache lines (rows need not be
    // 128-byte aligned): give them to one XCD
    Ctx x = make_ctx(p, xcd_remap(blockIdx.x, gridDim.x), threadIdx.x);
    if constexpr (SH >= 0) {
        wave_base<C>(x.in0, x.in_lane);
        wave_base<C>(x.out0, x.out_lane);
    }
    C v[RMAX];
    line_reg_phase<MODE, C, RMAX, SH>(0, in, out, lds, tw, fg, ci, p, x, sign, v);
    __syncthreads();
    line_reg_phase<MODE, C, RMAX, SH>(1, in, out, lds, tw, fg, ci, p, x, sign, v);
    if (MODE == 1) {
        __syncthreads();  // every stage-2 read of LDS is done
        line_reg_phase<MODE, C, RMAX, SH>(2, in, out, lds, tw, fg, ci, p, x, sign, v);
        __syncthreads();
        line_reg_phase<MODE, C, RMAX, SH>(3, in, out, lds, tw, fg, ci, p, x, sign, v);
    }
}

template <int MODE, typename C, int SH>
static void launch_sh(int rm, dim3 grid, dim3 block, size_t lds, hipStream_t s, const C *in, C *out,
                      const LinePass &p, const C *tw, int sign, const C *fg, const ConvInfo &ci) {
    switch (rm) {
#define INST(R)                                                                                              \
    case R:                                                                                                  \
        hipLaunchKernelGGL((k_line_reg<MODE, C, R, SH>), grid, block, lds, s, in, out, p, tw, sign, fg, ci); \
        break;
        INST(12) INST(14) INST(16) INST(18) INST(20)
#undef INST
    }
}

}  // namespace regfft

template <typename C>
void launch_line_reg(const LinePass &p, const C *in, C *out, const C *tw, int sign, const C *fg, const ConvInfo &ci,
                     int mode, hipStream_t s) {
    using namespace regfft;
    const long long tiles = (p.inner + p.ti - 1) / p.ti;
    const long long blocks = tiles * p.outer;
    if (blocks <= 0) return;
    if (blocks > 0x7fffffffLL) fail(SCADYN_ERR_UNSUPPORTED, "FFT grid too large");
    const size_t lds = line_pass_lds(p, sizeof(C));
    if (p.threads > reg_max_threads(sizeof(C))) fail(SCADYN_ERR_UNSUPPORTED, "FFT tile exceeds the thread bound");
    if (lds > 65536) fail(SCADYN_ERR_UNSUPPORTED, "FFT tile exceeds 64 KiB of LDS");
    const dim3 grid((unsigned)blocks), block(p.threads);
    const int rm = reg_rmax(p);
    constexpr int S0 = sizeof(C) == 16 ? 3 : 4;
    const int sh = reg_shift(p, ci, mode, sizeof(C));
#define GO(M, S) launch_sh<M, C, S>(rm, grid, block, lds, s, in, out, p, tw, sign, fg, ci)
    if (mode == 0) {
        if (sh == S0)
            GO(0, S0);
        else if (sh == S0 + 1)
            GO(0, S0 + 1);
        else
            GO(0, -1);
    } else {
        if (sh == 3)
            GO(1, 3);
        else if (sh == 4)
            GO(1, 4);
        else
            GO(1, -1);
    }
#undef GO
    HIP_CHECK(hipGetLastError());
}

}  // namespace scadyn
