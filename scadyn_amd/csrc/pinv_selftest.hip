// Host self-test of the pseudo-inverse: the vector evaluation (AVX2 and the plain
// target) against the plain loops below, bit for bit, on even and odd shapes,
// rank-deficient matrices and the equivalent-source fit's own kind.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "internal.hpp"

using namespace scadyn;

static std::vector<cd> plain(const std::vector<cd> &A0, int m, int n, double thr) {
    std::vector<cd> A = A0, V((size_t)n * n, cmk(0, 0));
    for (int i = 0; i < n; ++i) V[(size_t)i * n + i] = cmk(1, 0);
    auto col = [&](std::vector<cd> &M, int rows, int j) { return &M[(size_t)j * rows]; };
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0.0;
        for (int p = 0; p < n - 1; ++p)
            for (int q = p + 1; q < n; ++q) {
                cd *ap = col(A, m, p), *aq = col(A, m, q);
                double alpha = 0, beta = 0;
                cd gam = cmk(0, 0);
                for (int i = 0; i < m; ++i) {
                    alpha += cabs2(ap[i]);
                    beta += cabs2(aq[i]);
                    gam = cadd(gam, cmulc(ap[i], aq[i]));
                }
                double ag = std::sqrt(cabs2(gam));
                if (ag == 0.0) continue;
                double rel = ag / std::sqrt(alpha * beta);
                off = std::max(off, rel);
                if (rel < 1e-17) continue;
                // phase so that ap^H (aq e^{-i phi}) is real positive
                cd ph = cmk(gam.x / ag, -gam.y / ag);
                double zeta = (beta - alpha) / (2.0 * ag);
                double t = (zeta >= 0 ? 1.0 : -1.0) / (std::fabs(zeta) + std::sqrt(1.0 + zeta * zeta));
                double c = 1.0 / std::sqrt(1.0 + t * t), s = c * t;
                for (int i = 0; i < m; ++i) {
                    cd x = ap[i], y = cmul(aq[i], ph);
                    ap[i] = csub(cscale(x, c), cscale(y, s));
                    aq[i] = cadd(cscale(x, s), cscale(y, c));
                }
                cd *vp = col(V, n, p), *vq = col(V, n, q);
                for (int i = 0; i < n; ++i) {
                    cd x = vp[i], y = cmul(vq[i], ph);
                    vp[i] = csub(cscale(x, c), cscale(y, s));
                    vq[i] = cadd(cscale(x, s), cscale(y, c));
                }
            }
        if (off < 1e-16) break;
    }
    // pinv (n x m) = sum_j v_j (1/s_j) u_j^H, u_j = a_j / s_j
    std::vector<cd> P((size_t)n * m, cmk(0, 0));
    for (int j = 0; j < n; ++j) {
        cd *aj = col(A, m, j);
        double s2 = 0;
        for (int i = 0; i < m; ++i) s2 += cabs2(aj[i]);
        double s = std::sqrt(s2);
        if (!(s > thr)) continue;
        cd *vj = col(V, n, j);
        for (int i = 0; i < m; ++i) {
            cd u = cscale(cconj(aj[i]), 1.0 / (s * s));  // conj(u_i)/s
            for (int r = 0; r < n; ++r) P[(size_t)i * n + r] = cadd(P[(size_t)i * n + r], cmul(vj[r], u));
        }
    }
    return P;
}

int main() {
    int bad = 0, n_cases = 0;
    std::mt19937 rng(5);
    std::normal_distribution<double> nd;
    auto check = [&](const std::vector<cd> &A, int m, int n, double thr, const char *what) {
        const auto ref = plain(A, m, n, thr);
        for (int wide = 0; wide < 2; ++wide) {
            const auto got = pinv_jacobi(A, m, n, thr, wide != 0);
            int diff = got.size() != ref.size();
            // == takes the two zeros as equal: a padded row may add +0 to a sum of -0
            for (size_t i = 0; !diff && i < ref.size(); ++i) diff = !(got[i].x == ref[i].x && got[i].y == ref[i].y);
            if (diff) std::printf("%s %d x %d wide %d: differs\n", what, m, n, wide);
            bad += diff;
            ++n_cases;
        }
    };
    const int shapes[][2] = {{1, 1}, {2, 1}, {3, 2}, {4, 4}, {5, 5}, {7, 3}, {27, 27}, {31, 8}, {98, 27}};
    for (auto &sh : shapes) {
        const int m = sh[0], n = sh[1];
        std::vector<cd> A((size_t)m * n);
        for (auto &z : A) z = cmk(nd(rng), nd(rng));
        check(A, m, n, 1e-6, "random");
        if (n > 1) {  // a repeated column and a zero column
            std::copy(A.begin(), A.begin() + m, A.begin() + (size_t)(n - 1) * m);
            check(A, m, n, 1e-6, "repeated");
            std::fill(A.begin(), A.begin() + m, cmk(0, 0));
            check(A, m, n, 1e-6, "zero column");
        }
    }
    for (double kd : {0.05, 0.4, 1.5}) {  // 98 points around 27 nodes, as the fit
        std::vector<cd> A;
        for (int u = 0; u < 27; ++u)
            for (int i = 0; i < 98; ++i) {
                const double z = 1.0 - (2.0 * i + 1.0) / 98.0, r = std::sqrt(1.0 - z * z), f = 2.399963229728653 * i;
                const double d[3] = {2.5 * r * std::cos(f) - (u % 3 - 1), 2.5 * r * std::sin(f) - (u / 3 % 3 - 1),
                                     2.5 * z - (u / 9 - 1)};
                const double R = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
                A.push_back(cmk(std::cos(kd * R) / R, std::sin(kd * R) / R));
            }
        check(A, 98, 27, 1e-6, "fit");
    }
    std::printf("%d cases, %d failures\n", n_cases, bad);
    return bad != 0;
}
