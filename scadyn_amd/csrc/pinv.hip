// Pseudo-inverse of the equivalent-source fit (host code).
//
// Hestenes one-sided Jacobi SVD; replaces ZGESVD in pinv (src/possu.f90:369-422):
// pinv = V diag(1/s) U^H.  All 60 sweeps over the 351 column pairs are latency and
// issue on one core, and they are the largest host part of an operator's
// creation.  The fit is ill-conditioned enough that another order of its sums shows
// at 1e-9 in entries of the T-matrix that are small by symmetry, so every
// element's operations and the order of every sum are those of the plain loops;
// what they are evaluated with changed: four rows per vector, a pair's four sums in
// the lanes of one accumulator, and up to four pairs at a time, whose
// chains of dependent adds and divisions run side by side.  The AVX2 build of the
// same source (no FMA, so no other rounding) is taken where the processor has it.
// 98 x 27 on one core of an EPYC host: 4.1 ms before, now 1.9 (3.2 without AVX2).
#include <algorithm>
#include <cmath>

#include "internal.hpp"

namespace scadyn {
namespace {

typedef double V4 __attribute__((vector_size(32), aligned(8), may_alias));
#define ALWAYS_INLINE inline __attribute__((always_inline))
#define AT(p) (*(const V4 *)(p))
#define SHUF(a, b, i, j, k, l) __builtin_shufflevector(a, b, i, j, k, l)

// columns of complex numbers: real parts, then imaginary parts, each zero padded to
// a multiple of four rows
struct Mat {
    int rows, ld;
    std::vector<double> a;
    Mat(int rows, int cols) : rows(rows), ld((rows + 3) & ~3), a(2 * (size_t)ld * cols, 0.0) {}
    double *re(int j) { return &a[2 * (size_t)ld * j]; }
    double *im(int j) { return re(j) + ld; }
};

// acc = x^H x, y^H y, re x^H y, im x^H y, summed row by row: four rows' terms of each
// are transposed into one vector per row
ALWAYS_INLINE void add_products(V4 *acc, const double *x, const double *y, int ld) {
    const V4 xr = AT(x), xi = AT(x + ld), yr = AT(y), yi = AT(y + ld);
    const V4 a = xr * xr + xi * xi, b = yr * yr + yi * yi, c = xr * yr + xi * yi, d = xr * yi - xi * yr;
    const V4 ab0 = SHUF(a, b, 0, 4, 2, 6), ab1 = SHUF(a, b, 1, 5, 3, 7);
    const V4 cd0 = SHUF(c, d, 0, 4, 2, 6), cd1 = SHUF(c, d, 1, 5, 3, 7);
    V4 t = *acc;
    t += SHUF(ab0, cd0, 0, 1, 4, 5);
    t += SHUF(ab1, cd1, 0, 1, 4, 5);
    t += SHUF(ab0, cd0, 2, 3, 6, 7);
    t += SHUF(ab1, cd1, 2, 3, 6, 7);
    *acc = t;
}

// (x, y) <- (c x - s (ph y), s x + c (ph y))
ALWAYS_INLINE void rotate(double *__restrict__ x, double *__restrict__ y, int ld, double phx, double phy, double c,
                          double s) {
    const V4 pr = {phx, phx, phx, phx}, pi = {phy, phy, phy, phy}, vc = {c, c, c, c}, vs = {s, s, s, s};
    for (int i = 0; i < ld; i += 4) {
        const V4 xr = AT(x + i), xi = AT(x + ld + i), yr = AT(y + i), yi = AT(y + ld + i);
        const V4 br = yr * pr - yi * pi, bi = yr * pi + yi * pr;
        *(V4 *)(x + i) = xr * vc - br * vs;
        *(V4 *)(x + ld + i) = xi * vc - bi * vs;
        *(V4 *)(y + i) = xr * vs + br * vc;
        *(V4 *)(y + ld + i) = xi * vs + bi * vc;
    }
}

// K pairs of disjoint columns (p, q), (p + 1, q - 1), ...; returns the largest cosine
template <int K>
ALWAYS_INLINE double step(Mat &A, Mat &V, int p, int q) {
    V4 g[K];
    const double *x[K], *y[K];
    for (int k = 0; k < K; ++k) {
        g[k] = V4{0, 0, 0, 0};
        x[k] = A.re(p + k);
        y[k] = A.re(q - k);
    }
    for (int i = 0; i < A.ld; i += 4)
        for (int k = 0; k < K; ++k) add_products(&g[k], x[k] + i, y[k] + i, A.ld);
    double off = 0.0, phx[K], phy[K], c[K], s[K];
    bool turn[K];
    for (int k = 0; k < K; ++k) {
        const double alpha = g[k][0], beta = g[k][1], gx = g[k][2], gy = g[k][3];
        const double ag = std::sqrt(gx * gx + gy * gy);
        const double rel = ag == 0.0 ? 0.0 : ag / std::sqrt(alpha * beta);
        off = std::max(off, rel);
        turn[k] = !(ag == 0.0 || rel < 1e-17);
        // phase so that ap^H (aq e^{-i phi}) is real positive
        phx[k] = gx / ag;
        phy[k] = -gy / ag;
        const double zeta = (beta - alpha) / (2.0 * ag);
        const double t = (zeta >= 0 ? 1.0 : -1.0) / (std::fabs(zeta) + std::sqrt(1.0 + zeta * zeta));
        c[k] = 1.0 / std::sqrt(1.0 + t * t);
        s[k] = c[k] * t;
    }
    for (int k = 0; k < K; ++k) {
        if (!turn[k]) continue;
        rotate(A.re(p + k), A.re(q - k), A.ld, phx[k], phy[k], c[k], s[k]);
        rotate(V.re(p + k), V.re(q - k), V.ld, phx[k], phy[k], c[k], s[k]);
    }
    return off;
}

// Cyclic sweeps over the pairs p < q, row by row.  The pairs of one p + q share no
// column, and all that a pair has to follow, (p, q - 1) and (p - 1, q), lie on the
// diagonal before: going by diagonals is the same arithmetic.
ALWAYS_INLINE void sweeps(Mat &A, Mat &V, int n) {
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0.0;
        for (int d = 1; d <= 2 * n - 3; ++d) {
            int p = std::max(0, d - (n - 1));
            for (; p + 3 < d - p - 3; p += 4) off = std::max(off, step<4>(A, V, p, d - p));
            if (p + 1 < d - p - 1) {
                off = std::max(off, step<2>(A, V, p, d - p));
                p += 2;
            }
            if (p < d - p) off = std::max(off, step<1>(A, V, p, d - p));
        }
        if (off < 1e-16) break;
    }
}

ALWAYS_INLINE void pinv_body(Mat &A, Mat &V, Mat &P, int m, int n, double thr) {
    sweeps(A, V, n);
    // P(:, i) += V(:, j) conj(a_ij) / s_j^2
    for (int j = 0; j < n; ++j) {
        const double *ar = A.re(j), *ai = A.im(j), *v = V.re(j);
        double s2 = 0;
        for (int i = 0; i < m; ++i) s2 += ar[i] * ar[i] + ai[i] * ai[i];
        const double s = std::sqrt(s2);
        if (!(s > thr)) continue;
        const double f = 1.0 / (s * s);
        for (int i = 0; i < m; ++i) {
            const double ux = ar[i] * f, uy = -ai[i] * f;
            const V4 ur = {ux, ux, ux, ux}, ui = {uy, uy, uy, uy};
            double *o = P.re(i);
            for (int r = 0; r < P.ld; r += 4) {
                const V4 vr = AT(v + r), vi = AT(v + V.ld + r);
                *(V4 *)(o + r) += vr * ur - vi * ui;
                *(V4 *)(o + P.ld + r) += vr * ui + vi * ur;
            }
        }
    }
}

void pinv_any(Mat &A, Mat &V, Mat &P, int m, int n, double thr) { pinv_body(A, V, P, m, n, thr); }
__attribute__((target("avx2"))) void pinv_avx2(Mat &A, Mat &V, Mat &P, int m, int n, double thr) {
    pinv_body(A, V, P, m, n, thr);
}

}  // namespace

// A column-major m x n, m >= n; the result column-major n x m
std::vector<cd> pinv_jacobi(const std::vector<cd> &A0, int m, int n, double thr, bool wide) {
    Mat A(m, n), V(n, n), P(n, m);
    for (int j = 0; j < n; ++j) {
        for (int i = 0; i < m; ++i) {
            A.re(j)[i] = A0[(size_t)j * m + i].x;
            A.im(j)[i] = A0[(size_t)j * m + i].y;
        }
        V.re(j)[j] = 1.0;
    }
    if (wide && __builtin_cpu_supports("avx2"))
        pinv_avx2(A, V, P, m, n, thr);
    else
        pinv_any(A, V, P, m, n, thr);
    std::vector<cd> out((size_t)n * m);
    for (int i = 0; i < m; ++i)
        for (int r = 0; r < n; ++r) out[(size_t)i * n + r] = cmk(P.re(i)[r], P.im(i)[r]);
    return out;
}

}  // namespace scadyn
