// Host self-test of the narrow scatter: the kernel's own per-lane steps
// (scatter_core.hpp) over exact-size buffers, workgroup by workgroup as the kernel
// strides over the nodes, against the sum written out; and the launch geometry on
// grids beyond 2^26 nodes.
//
// Exit status 0 when every case is within tolerance.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "scatter_core.hpp"

using namespace scadyn;
using namespace scadyn::score;

static int failures = 0, cases = 0;

template <typename C>
struct Data {
    ScatterArgs<C> a;
    std::vector<C> xin, S4, grid;
    std::vector<long long> off;
    std::vector<int> cs;
};

template <typename C>
static void make(Data<C> &d, int ncx, int ncy, int ncz, int B, std::mt19937_64 &rng) {
    std::normal_distribution<double> nd;
    d.cs.assign(1, 0);
    for (int c = 0; c < ncx * ncy * ncz; ++c) d.cs.push_back(d.cs.back() + (int)(rng() % 5) * (int)(rng() % 4));
    const int N = d.cs.back();
    auto fill = [&](std::vector<C> &v, size_t n) {
        v.resize(n);
        for (auto &z : v) z.x = (typename Prec<C>::real)nd(rng), z.y = (typename Prec<C>::real)nd(rng);
    };
    fill(d.xin, (size_t)3 * N * B);
    fill(d.S4, (size_t)108 * N);
    d.off.assign(B, 0);
    // one plane of nodes beyond the last box along x, as grids of even node counts have
    const int Nx = 2 * ncx + 2, Ny = 2 * ncy + 1, Nz = 2 * ncz + 1;
    d.grid.assign((size_t)Nx * Ny * Nz * 4 * B, C{9, 9});
    d.a = {d.xin.data(), d.off.data(), B, d.cs.data(), d.S4.data(), Nx, Ny, Nz, ncx, ncy, ncz, d.grid.data()};
}

// the kernel's loop for a launch of nwg workgroups; the groups' sums are added in order
template <typename C, int SB, int G>
static void emulate(const ScatterArgs<C> &s, unsigned nwg) {
    constexpr int PER = nodes_per_group<SB, G>();
    const long long nodes = (long long)s.Nx * s.Ny * s.Nz;
    for (unsigned w = 0; w < nwg; ++w)
        for (int q = 0; q < PER; ++q)
            for (long long p = (long long)w * PER + q; p < nodes; p += (long long)nwg * PER)
                for (int b = 0; b < SB; ++b) {
                    C sum[4] = {};
                    for (int g = 0; g < G; ++g) {
                        C a[4];
                        node_share<C, G>(s, p, b < s.B ? b : s.B - 1, g, a);
                        for (int c = 0; c < 4; ++c) sum[c] = cadd(sum[c], a[c]);
                    }
                    if (b < s.B) write_node(s, p, b, sum);
                }
}

// one thread per (node, slot)
template <typename C>
static void emulate_flat(const ScatterArgs<C> &s) {
    for (long long p = 0; p < (long long)s.Nx * s.Ny * s.Nz; ++p)
        for (int b = 0; b < s.B; ++b) {
            C a[4];
            node_share<C, 1>(s, p, b, 0, a);
            write_node(s, p, b, a);
        }
}

template <typename C>
static double error(const Data<C> &d) {
    const ScatterArgs<C> &s = d.a;
    long double num = 0, den = 0;
    for (int pz = 0; pz < s.Nz; ++pz)
        for (int py = 0; py < s.Ny; ++py)
            for (int px = 0; px < s.Nx; ++px)
                for (int b = 0; b < s.B; ++b) {
                    cd r[4] = {};
                    for (int c = 0; c < s.ncx * s.ncy * s.ncz; ++c) {
                        const int jx = px - 2 * (c % s.ncx), jy = py - 2 * (c / s.ncx % s.ncy), jz = pz - 2 * (c / (s.ncx * s.ncy));
                        if (jx < 0 || jx > 2 || jy < 0 || jy > 2 || jz < 0 || jz > 2) continue;
                        for (int t = d.cs[c]; t < d.cs[c + 1]; ++t) {
                            const C *w = &d.S4[((size_t)t * 27 + jx + 3 * jy + 9 * jz) * 4];
                            for (int q = 0; q < 3; ++q) {
                                const cd x = Prec<cd>::from(d.xin[(size_t)(3 * t + q) * s.B + b]);
                                r[q] = cadd(r[q], cmul(Prec<cd>::from(w[0]), x));
                                r[3] = cadd(r[3], cmul(Prec<cd>::from(w[1 + q]), x));
                            }
                        }
                    }
                    const size_t p = px + (size_t)s.Nx * (py + (size_t)s.Ny * pz);
                    for (int q = 0; q < 4; ++q) {
                        const cd g = Prec<cd>::from(d.grid[(p * 4 + q) * s.B + b]);
                        num += cabs2(csub(g, r[q]));
                        den += cabs2(r[q]);
                    }
                }
    return (double)std::sqrt(num / den);
}

template <typename C, int SB, int G>
static void one(int B, std::mt19937_64 &rng) {
    Data<C> d;
    make(d, 3, 2, 4, B, rng);
    const long long nodes = (long long)d.a.Nx * d.a.Ny * d.a.Nz;
    for (unsigned nwg : {grid_for(nodes, nodes_per_group<SB, G>()), 3u}) {
        std::fill(d.grid.begin(), d.grid.end(), C{9, 9});
        emulate<C, SB, G>(d.a, nwg);
        const double e = error(d);
        ++cases;
        if (!(e < (sizeof(C) == 16 ? 1e-14 : 2e-6))) {
            ++failures;
            std::printf("%s B=%d SB=%d G=%d, %u workgroups: rel.err %.2e\n", sizeof(C) == 16 ? "c128" : "c64", B, SB, G, nwg, e);
        }
    }
}
template <typename C>
static void flat(int B, std::mt19937_64 &rng) {
    Data<C> d;
    make(d, 3, 2, 4, B, rng);
    emulate_flat(d.a);
    ++cases;
    const double e = error(d);
    if (!(e < (sizeof(C) == 16 ? 1e-14 : 2e-6))) {
        ++failures;
        std::printf("%s B=%d, thread per slot: rel.err %.2e\n", sizeof(C) == 16 ? "c128" : "c64", B, e);
    }
}

// the rule's groups fit a wave, and its kernels are those compiled
template <int SB>
static void picks() {
    for (long long nodes = 1; nodes < 1LL << 40; nodes = nodes * 3 / 2 + 1) {
        const int g = pick_groups<SB>(nodes);
        ++cases;
        if (SB * g > 64 || (g != 2 && g != 4 && g != 8 && g != 16)) {
            ++failures;
            std::printf("SB=%d, %lld nodes: %d groups\n", SB, nodes, g);
        }
    }
}

template <int SB, int G>
static void both(int B, std::mt19937_64 &rng) {
    one<cd, SB, G>(B, rng);
    one<cf, SB, G>(B, rng);
}

// a launch of grid_for workgroups stays below 2^32 threads, and its strides reach
// the last node
static void launch(long long nodes, int per) {
    const unsigned long long nwg = grid_for(nodes, per);
    ++cases;
    const bool all = nwg * (unsigned long long)per >= (unsigned long long)nodes || nwg == 1ULL << 20;
    if (nwg * THREADS >= 1ULL << 32 || !all) {
        ++failures;
        std::printf("%lld nodes, %d a workgroup: %llu workgroups\n", nodes, per, nwg);
    }
}

int main() {
    std::mt19937_64 rng(3);
    both<1, 16>(1, rng);
    both<1, 8>(1, rng);
    both<2, 16>(2, rng);
    both<2, 4>(2, rng);
    for (int B : {3, 4}) both<4, 16>(B, rng), both<4, 4>(B, rng), both<4, 2>(B, rng);
    for (int B : {5, 8}) both<8, 8>(B, rng), both<8, 4>(B, rng), both<8, 2>(B, rng);
    for (int B : {9, 16}) both<16, 4>(B, rng), both<16, 2>(B, rng);
    for (int B : {17, 24}) both<32, 2>(B, rng);
    for (int B : {5, 12, 24}) flat<cd>(B, rng), flat<cf>(B, rng);
    picks<1>(), picks<2>(), picks<4>(), picks<8>(), picks<16>(), picks<32>();
    for (long long nodes : {1LL, 15LL, 17LL, (1LL << 26) - 1, (1LL << 26) + 1, 1LL << 28, (1LL << 28) + 5, 1LL << 33})
        for (int per : {4, 8, 16, 32}) launch(nodes, per);
    std::printf("%d cases, %d failures\n", cases, failures);
    return failures != 0;
}
