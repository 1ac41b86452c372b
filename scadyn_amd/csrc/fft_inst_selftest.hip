// Host self-test of the register line FFT's compiled instances: the one that the
// launcher picks for a pass (reg_shift: tile width fixed at compile time, 32-bit
// lane offsets from a wave's first lane) run lane by lane, a wave's addresses split
// as the kernel splits them.
//
//  * transforms and the fused convolution at the planner's own widths, full, partial
//    and single tiles, against the 64-bit instance: the same operations, so the
//    same bits;
//  * convolutions whose octant of FFT(G) is larger than 2 GiB and 4 GiB (wide flat
//    boxes), against a direct long-double DFT.  The octant is reserved, not
//    filled: only the columns of the tile are written and read.
//
// Exit status 0 when every case passes.
#include <sys/mman.h>

#include <array>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "fft_reg_core.hpp"

using namespace scadyn;
using namespace scadyn::regfft;
typedef std::complex<long double> cl;

static const long double PI_L = 3.141592653589793238462643383279502884L;
static int failures = 0, cases = 0;

template <typename C>
static std::vector<C> twiddles(int L) {
    std::vector<C> t(L);
    for (int m = 0; m < L; ++m) {
        const cl w = std::polar(1.0L, -2.0L * PI_L * m / L);
        t[m].x = (typename Prec<C>::real)w.real();
        t[m].y = (typename Prec<C>::real)w.imag();
    }
    return t;
}

// one workgroup (the register bound RMAX changes no operation: the largest for all);
// shift: columns added to the one that fixes the octant's row
template <int MODE, typename C, int SH>
static void block(const LinePass &p, long long b, const C *in, C *out, const C *tw, int sign, const C *fg,
                  const ConvInfo &ci, long long shift) {
    std::vector<C> lds((size_t)p.L * p.ti);
    std::vector<std::array<C, 20>> regs(p.threads);
    for (int ph = 0; ph < (MODE == 0 ? 2 : 4); ++ph)
        for (int t = 0; t < p.threads; ++t) {
            Ctx x = make_ctx(p, b, t);
            x.i += shift;
            if (SH >= 0) {
                const Ctx first = make_ctx(p, b, t & ~63);
                x.in_lane = (unsigned)((x.in0 - first.in0) * sizeof(C));
                x.out_lane = (unsigned)((x.out0 - first.out0) * sizeof(C));
                x.in0 = first.in0;
                x.out0 = first.out0;
            }
            line_reg_phase<MODE, C, 20, SH>(ph, in, out, lds.data(), tw, fg, ci, p, x, sign, regs[t].data());
        }
}
template <int MODE, typename C, int SH>
static void blocks(const LinePass &p, const C *in, C *out, const C *tw, int sign, const C *fg, const ConvInfo &ci,
                   long long shift) {
    const long long n = (p.inner + p.ti - 1) / p.ti * p.outer;
    for (long long b = 0; b < n; ++b) block<MODE, C, SH>(p, b, in, out, tw, sign, fg, ci, shift);
}
template <int MODE, typename C>
static void run(int sh, const LinePass &p, const C *in, C *out, const C *tw, int sign, const C *fg, const ConvInfo &ci,
                long long shift = 0) {
    constexpr int S0 = MODE == 1 || sizeof(C) == 16 ? 3 : 4;
    if (sh == S0)
        blocks<MODE, C, S0>(p, in, out, tw, sign, fg, ci, shift);
    else if (sh == S0 + 1)
        blocks<MODE, C, S0 + 1>(p, in, out, tw, sign, fg, ci, shift);
    else
        blocks<MODE, C, -1>(p, in, out, tw, sign, fg, ci, shift);
}

template <typename C>
static void fill(std::vector<C> &v, std::mt19937_64 &rng) {
    std::normal_distribution<double> nd;
    for (auto &z : v) z.x = (typename Prec<C>::real)nd(rng), z.y = (typename Prec<C>::real)nd(rng);
}

template <typename C>
static void same_bits(const char *what, const LinePass &p, int sh, const std::vector<C> &a, const std::vector<C> &b) {
    ++cases;
    bool ok = true;
    for (size_t i = 0; i < a.size(); ++i) ok &= a[i].x == b[i].x && a[i].y == b[i].y;
    if (!ok) {
        ++failures;
        std::printf("%s %s L=%d ti=%d instance %d: differs from the 64-bit instance\n", what,
                    sizeof(C) == 16 ? "c128" : "c64", p.L, p.ti, sh);
    }
}

template <typename C>
static void planned(int L, long long inner, std::mt19937_64 &rng) {
    std::vector<C> tw = twiddles<C>(L);
    for (int sign = -1; sign <= 1; sign += 2) {
        const int n_in = sign < 0 ? L / 2 + 1 : L, n_out = sign < 0 ? L : L / 2 + 1;
        LinePass p;
        plan_transform(p, L, n_in, n_out, inner, 2, sizeof(C), true);
        const int sh = reg_shift(p, ConvInfo(), 0, sizeof(C));
        std::vector<C> in((size_t)2 * n_in * inner), a((size_t)2 * n_out * inner), b(a.size());
        fill(in, rng);
        run<0, C>(sh, p, in.data(), a.data(), tw.data(), sign, nullptr, ConvInfo());
        run<0, C>(-1, p, in.data(), b.data(), tw.data(), sign, nullptr, ConvInfo());
        same_bits(sign < 0 ? "fwd" : "inv", p, sh, a, b);
        // and the widest tiles against the definition
        if (inner < 64) continue;
        std::vector<cl> w(L);
        for (int q = 0; q < L; ++q) w[q] = std::polar(1.0L, sign * 2.0L * PI_L * q / L);
        long double num = 0, den = 0;
        for (int c = 0; c < inner; c += 7)
            for (int k = 0; k < n_out; ++k) {
                cl r = 0;
                for (int n = 0; n < n_in; ++n) r += cl(in[(size_t)n * inner + c].x, in[(size_t)n * inner + c].y) * w[(n * k) % L];
                const C o = a[(size_t)k * inner + c];
                num += std::norm(cl(o.x, o.y) - r);
                den += std::norm(r);
            }
        ++cases;
        if (!(std::sqrt(num / den) < (sizeof(C) == 16 ? 1e-14 : 2e-6))) {
            ++failures;
            std::printf("%d points, %d columns: rel.err %.2Le\n", L, p.ti, std::sqrt(num / den));
        }
    }
    const int Nz = L / 2;
    LinePass p;
    plan_conv(p, L, Nz, inner, sizeof(C), true);
    ConvInfo ci;
    ci.Lx = (int)inner, ci.Ly = 1, ci.Lz = L, ci.Hx = (int)inner / 2 + 1, ci.Hy = 1, ci.nb = 1;
    const int sh = reg_shift(p, ci, 1, sizeof(C));
    std::vector<C> in((size_t)Nz * inner), a(in.size()), b(in.size()), fg((size_t)ci.Hx * (L / 2 + 1));
    fill(in, rng);
    fill(fg, rng);
    run<1, C>(sh, p, in.data(), a.data(), tw.data(), -1, fg.data(), ci);
    run<1, C>(-1, p, in.data(), b.data(), tw.data(), -1, fg.data(), ci);
    same_bits("conv", p, sh, a, b);
}

// the planner's widths: {length, columns, complex128 transform, complex64 transform,
// complex128 convolution, complex64 convolution}
static void widths() {
    const int want[][6] = {
        {105, 1 << 20, 16, 32, 16, 16}, {160, 1 << 20, 16, 32, 16, 16}, {168, 1 << 20, 16, 32, 16, 16},
        {210, 1 << 20, 16, 32, 8, 16},  // 16 columns of complex128 exceed 48 KiB
        {270, 1 << 20, 8, 16, 8, 16},   // and here 64 KiB, as do 32 of complex64
        {360, 1 << 20, 8, 16, 8, 16},  {400, 1 << 20, 8, 16, 8, 8},   // not below 8 columns
        {20, 1 << 20, 32, 32, 32, 32}, {75, 1 << 20, 32, 32, 32, 32}, // five thread rows: twice as wide
        {20, 16, 16, 16, 16, 16},                                     // the inner extent bounds it
        {168, 4, 4, 4, 4, 4},          {168, 8, 8, 8, 8, 8},
        {168, 12, 4, 8, 4, 8},         {168, 20, 8, 16, 8, 16}, // a quarter of the columns beyond the extent
        {168, 48, 16, 16, 16, 16},     {168, 36, 16, 16, 16, 16}, {168, 28, 16, 16, 16, 16}};
    for (auto &q : want) {
        LinePass p[4];
        plan_transform(p[0], q[0], q[0] / 2, q[0], q[1], 3, 16, true);
        plan_transform(p[1], q[0], q[0] / 2, q[0], q[1], 3, 8, true);
        plan_conv(p[2], q[0], q[0] / 2, q[1], 16, true);
        plan_conv(p[3], q[0], q[0] / 2, q[1], 8, true);
        for (int i = 0; i < 4; ++i) {
            ++cases;
            if (p[i].ti != q[2 + i] || !p[i].reg || line_pass_lds(p[i], i % 2 ? 8 : 16) > 64 * 1024 ||
                p[i].threads > reg_max_threads(i % 2 ? 8 : 16)) {
                ++failures;
                std::printf("%d points, %d columns, plan %d: %d columns a tile, not %d\n", q[0], q[1], i, p[i].ti, q[2 + i]);
            }
        }
        // the Stockham kernel: two buffers of 64 columns at most in 64 KiB, transform and convolution alike
        plan_transform(p[0], q[0], q[0] / 2, q[0], q[1], 1, 16, false);
        plan_conv(p[2], q[0], q[0] / 2, q[1], 16, false);
        ++cases;
        if (p[0].ti != p[2].ti || p[0].reg || p[2].reg) ++failures, std::printf("%d points: Stockham widths %d, %d\n", q[0], p[0].ti, p[2].ti);
    }
}

// The tile of the columns around (Lx / 2, Ly / 2), the octant's last row, of a grid
// Lx x Ly x Lz.  16 columns, 4 to a grid point.
template <typename C>
static void wide(int Lx, int Ly, int Lz, std::mt19937_64 &rng, double tol) {
    const int Nz = Lz / 2, nb = 4;
    const long long inner = 16;
    LinePass p;
    plan_conv(p, Lz, Nz, inner, sizeof(C), true);
    ConvInfo ci;
    ci.Lx = Lx, ci.Ly = Ly, ci.Lz = Lz, ci.Hx = Lx / 2 + 1, ci.Hy = Ly / 2 + 1, ci.nb = nb;
    const size_t zs = (size_t)ci.Hx * ci.Hy, bytes = zs * (Lz / 2 + 1) * sizeof(C);
    void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) {
        std::printf("no address space for an octant of %zu bytes\n", bytes);
        ++failures;
        return;
    }
    C *fg = (C *)m;
    const long long shift = nb * ((long long)Lx * (Ly / 2) + Lx / 2 - 2);
    std::normal_distribution<double> nd;
    auto row = [&](int c, int kz) {
        const long long xy = (shift + c) / nb;
        const int gx = (int)(xy % Lx), gy = (int)(xy / Lx);
        return (size_t)kz * zs + (size_t)std::min(gy, Ly - gy) * ci.Hx + std::min(gx, Lx - gx);
    };
    for (int c = 0; c < inner; c += nb)
        for (int kz = 0; kz <= Lz / 2; ++kz) {
            C &f = fg[row(c, kz)];
            if (f.x == 0) f.x = (typename Prec<C>::real)nd(rng), f.y = (typename Prec<C>::real)nd(rng);
        }
    std::vector<C> tw = twiddles<C>(Lz), in((size_t)Nz * inner), out(in.size());
    fill(in, rng);
    const int sh = reg_shift(p, ci, 1, sizeof(C));
    run<1, C>(sh, p, in.data(), out.data(), tw.data(), -1, fg, ci, shift);
    std::vector<cl> w(Lz);
    for (int q = 0; q < Lz; ++q) w[q] = std::polar(1.0L, -2.0L * PI_L * q / Lz);
    long double num = 0, den = 0;
    for (int c = 0; c < inner; ++c) {
        std::vector<cl> X(Lz);
        for (int k = 0; k < Lz; ++k) {
            cl a = 0;
            for (int n = 0; n < Nz; ++n) a += cl(in[(size_t)n * inner + c].x, in[(size_t)n * inner + c].y) * w[(n * k) % Lz];
            const C f = fg[row(c, std::min(k, Lz - k))];
            X[k] = a * cl(f.x, f.y);
        }
        for (int n = 0; n < Nz; ++n) {
            cl a = 0;
            for (int k = 0; k < Lz; ++k) a += X[k] * std::conj(w[(n * k) % Lz]);
            const C o = out[(size_t)n * inner + c];
            num += std::norm(cl(o.x, o.y) - a);
            den += std::norm(a);
        }
    }
    munmap(m, bytes);
    ++cases;
    const double err = (double)std::sqrt(num / den);
    const bool ok = err < tol;
    if (!ok) ++failures;
    std::printf("octant %.2f GiB, %d x %d x %d %s, ti=%d, instance %d: rel.err %.2e %s\n", bytes / 1073741824.0, Lx, Ly,
                Lz, sizeof(C) == 16 ? "c128" : "c64", p.ti, sh, err, ok ? "ok" : "FAIL");
}

int main() {
    std::mt19937_64 rng(77);
    widths();
    for (int L : {20, 24, 35, 75, 90, 105, 112, 160, 168, 210, 270, 360, 400})
        for (long long inner : {4, 12, 16, 20, 33, 64}) {
            planned<cd>(L, inner, rng);
            planned<cf>(L, inner, rng);
        }
    // below 2 GiB, where the running offsets still fit or just do not, and beyond 2 and 4 GiB
    wide<cd>(1120, 1120, 400, rng, 1e-14);
    wide<cd>(1176, 1176, 400, rng, 1e-14);
    wide<cd>(1680, 1680, 400, rng, 1e-14);
    wide<cd>(2400, 2400, 400, rng, 1e-14);
    wide<cd>(2400, 2400, 225, rng, 1e-14);
    wide<cf>(2400, 2400, 400, rng, 2e-6);
    wide<cf>(3360, 3360, 400, rng, 2e-6);
    std::printf("%d cases, %d failures\n", cases, failures);
    return failures != 0;
}
