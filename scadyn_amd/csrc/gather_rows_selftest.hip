// Host self-test of the row-group gather kernels (k_gather_lds, k_gather_cols): their
// own per-lane steps (gather_core.hpp) on the CPU, one wave at a time with the
// workgroup barriers as phase boundaries, over exact-size buffers (AddressSanitizer
// on the host build reports any access outside them), against a direct evaluation of
//   y_t = sum_j (S_{c+1}[t][j] g3[node_j] - k^2 S[t][j] g_c[node_j])
//       + sum_{near tets v} A(t, v) x_v
// on a lattice of cubes of 0 to 13 tets (row groups of 1 to 6 rows, lane groups past
// the end of a group, near lines longer than a staged chunk), blocks with and without
// the transpose flag, inactive slots (left unwritten), every wave layout that the
// launcher picks, full, partial and single chunks of slots.
//
// Exit status 0 when every case agrees to 1e-13 (complex128) / 1e-5 (complex64).
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <random>
#include <type_traits>
#include <vector>

#include "gather_core.hpp"

using namespace scadyn;
using namespace scadyn::gcore;

static int failures = 0;
constexpr int HT = ROW_GT / 2, VC = ROW_VC;

template <typename C>
static C to(cd a) {
    return Prec<C>::from(a);
}

// gather_pass of matvec.hip
template <typename C, int NT, int SB, int NS>
static void rows_pass(const GatherArgs<C> &g, const Item &it, int chunk, std::vector<cd> &lds) {
    C *sm = (C *)lds.data();
    cf *smb = (cf *)lds.data();
    const int rows = it.t1 - it.t0;
    struct Lane {
        Slots<SB, NS> sl;
        C acc[NT][3][NS];
        long long off[NS];
        int64_t rs0, rs1;
    };
    std::vector<Lane> L(64);
    for (int l = 0; l < 64; ++l) {
        L[l].sl = lane_slots<SB, NS>(g, chunk, l);
        for (auto &u : L[l].acc)
            for (auto &c : u)
                for (auto &z : c) z = Prec<C>::zero();
        for (int i = 0; i < NS; ++i) L[l].off[i] = g.in_off[L[l].sl.s[i]] + L[l].sl.s[i];
        stage_s4(g, it.t0, rows, l, sm);
    }
    for (int l = 0; l < 64; ++l) grid_rows<C, NT, NS>(g, it, L[l].sl.s, sm + L[l].sl.grp * NT * 108, L[l].acc);
    for (int l = 0; l < 64; ++l) {
        L[l].rs0 = lane_row_start<C, HT, VC>(g, it.t0, std::min(rows, HT), l);
        L[l].rs1 = lane_row_start<C, HT, VC>(g, it.t0 + HT, rows - HT, l);
    }
    int q = 0;
    for_near_cubes(g, it, [&](int c0, int c1) {
        for (int v0 = c0; v0 < c1; v0 += VC) {
            const int nv = std::min(VC, c1 - v0);
            for (int l = 0; l < 64; ++l) {
                stage_blocks<C, HT, VC>(g, std::min(rows, HT), nv, q, l, L[l].rs0, smb);
                if (rows > HT) stage_blocks<C, HT, VC>(g, rows - HT, nv, q, l, L[l].rs1, smb + HT * VC * 9);
            }
            for (int l = 0; l < 64; ++l)
                chunk_rows<C, NT, VC, NS>(g, L[l].off, v0, nv, smb + L[l].sl.grp * NT * VC * 9, L[l].acc);
            q += nv;
        }
    });
    for (int l = 0; l < 64; ++l) write_rows<C, NT, SB, NS>(g, it, L[l].sl, L[l].acc);
}

// k_gather_lds, one item per workgroup
template <typename C, int SB, int NS>
static void rows_kernel(const GatherArgs<C> &g) {
    constexpr int G = 64 / SB, NTMAX = (ROW_GT + G - 1) / G;
    std::vector<cd> lds((Shape<C, G * NTMAX, VC>::BYTES + 15) / 16);
    const long long nw = (long long)g.n_groups * ((g.B + SB * NS - 1) / (SB * NS));
    for (long long b = 0; b < nw; ++b) {
        const long long w = xcd_remap(b, nw);
        const int chunk = (int)(w / g.n_groups);
        const Item it = group_item(g, (int)(w - (long long)chunk * g.n_groups));
        const int nt = (it.t1 - it.t0 + G - 1) / G;
        if constexpr (NTMAX >= 1)
            if (nt == 1) rows_pass<C, 1, SB, NS>(g, it, chunk, lds);
        if constexpr (NTMAX >= 2)
            if (nt == 2) rows_pass<C, 2, SB, NS>(g, it, chunk, lds);
        if constexpr (NTMAX >= 3)
            if (nt == 3) rows_pass<C, 3, SB, NS>(g, it, chunk, lds);
        if (nt < 1 || nt > NTMAX) ++failures;
    }
}

// gather_cols of matvec.hip
template <typename C, int NT, int SB>
static void cols_pass(const GatherArgs<C> &g, const Item &it, int tp, int chunk, std::vector<cd> &lds) {
    C *sm = (C *)lds.data();
    cf *smb = (cf *)lds.data();
    struct Lane {
        Slots<SB, 1> sl;
        C acc[NT][3];
        long long off;
        int64_t rs;
    };
    std::vector<Lane> L(64);
    for (int l = 0; l < 64; ++l) {
        L[l].sl = lane_slots<SB, 1>(g, chunk, l);
        zero_acc<C, NT>(L[l].acc);
        L[l].off = g.in_off[L[l].sl.s[0]] + L[l].sl.s[0];
        stage_s4(g, tp, NT, l, sm);
    }
    for (int l = 0; l < 64; ++l) grid_share<C, NT, SB>(g, it, L[l].sl, sm, L[l].acc);
    for (int l = 0; l < 64; ++l) L[l].rs = lane_row_start<C, HT, VC>(g, tp, NT, l);
    int q = 0;
    for_near_cubes(g, it, [&](int c0, int c1) {
        for (int v0 = c0; v0 < c1; v0 += VC) {
            const int nv = std::min(VC, c1 - v0);
            for (int l = 0; l < 64; ++l) stage_blocks<C, HT, VC>(g, NT, nv, q, l, L[l].rs, smb);
            for (int l = 0; l < 64; ++l) chunk_share<C, NT, VC, SB>(g, L[l].sl, L[l].off, v0, nv, smb, L[l].acc);
            q += nv;
        }
    });
    for (int l = 0; l < SB; ++l) {  // lane group 0 writes the groups' sum
        if (!L[l].sl.ok[0] || !g.slot_active[L[l].sl.s[0]]) continue;
        for (int u = 0; u < NT; ++u)
            for (int c = 0; c < 3; ++c) {
                C v = Prec<C>::zero();
                for (int m = l; m < 64; m += SB) v = cadd(v, L[m].acc[u][c]);
                g.y[(size_t)(3 * (tp + u) + c) * g.B + L[l].sl.s[0]] = Prec<cd>::from(v);
            }
    }
}
// k_gather_cols
template <typename C, int SB>
static void cols_kernel(const GatherArgs<C> &g) {
    std::vector<cd> lds((Shape<C, HT, VC>::BYTES + 15) / 16);
    const long long nw = (long long)g.n_groups * 2 * ((g.B + SB - 1) / SB);
    for (long long b = 0; b < nw; ++b) {
        const long long w = xcd_remap(b, nw);
        const int chunk = (int)(w / (2 * g.n_groups)), i = (int)(w - (long long)chunk * 2 * g.n_groups);
        const Item it = group_item(g, i >> 1);
        const int tp = it.t0 + (i & 1 ? HT : 0), nt = std::min(HT, it.t1 - tp);
        if (nt == 1) cols_pass<C, 1, SB>(g, it, tp, chunk, lds);
        if (nt == 2) cols_pass<C, 2, SB>(g, it, tp, chunk, lds);
        if (nt == 3) cols_pass<C, 3, SB>(g, it, tp, chunk, lds);
    }
}

template <typename C, typename K>
static void run_case(const char *what, int B, std::mt19937_64 &rng, K &&kernel) {
    const int ncx = 4, ncy = 3, ncz = 3, Nx = 2 * ncx + 2, Ny = 2 * ncy + 2, Nz = 2 * ncz + 2, nc = ncx * ncy * ncz;
    std::vector<int> cs(1, 0);
    for (int c = 0; c < nc; ++c) cs.push_back(cs.back() + (c % 5 == 0 ? 0 : (int)(rng() % 14)));
    const int N = cs.back();
    std::vector<int> cube(N);
    std::vector<int2> groups;
    for (int c = 0; c < nc; ++c) {
        for (int t = cs[c]; t < cs[c + 1]; ++t) cube[t] = c;
        add_row_groups(groups, c, cs[c], cs[c + 1] - cs[c]);
    }
    std::vector<int64_t> row_start(1, 0);
    std::vector<int> col;
    for (int t = 0; t < N; ++t) {
        for (int o = 0; o < 27; ++o) {
            const int x = cube[t] % ncx + o % 3 - 1, y = cube[t] / ncx % ncy + o / 3 % 3 - 1, z = cube[t] / (ncx * ncy) + o / 9 - 1;
            if (x < 0 || x >= ncx || y < 0 || y >= ncy || z < 0 || z >= ncz) continue;
            const int b = x + ncx * (y + ncy * z);
            for (int v = cs[b]; v < cs[b + 1]; ++v) col.push_back(v);
        }
        row_start.push_back((int64_t)col.size());
    }
    std::normal_distribution<double> nd;
    auto rnd = [&](auto &v) {
        for (auto &z : v) z = Prec<typename std::decay<decltype(z)>::type>::from(cmk(nd(rng), nd(rng)));
    };
    const size_t P = col.size() / 2 + 1;
    std::vector<uint32_t> blk(col.size());
    for (auto &e : blk) e = (uint32_t)(rng() % P) | (rng() & 1 ? 0x80000000u : 0u);
    std::vector<cf> blocks(P * 9);
    std::vector<C> S4((size_t)N * 108), grid((size_t)Nx * Ny * Nz * 4 * B), xin((size_t)2 * 3 * N * B);
    rnd(blocks), rnd(S4), rnd(grid), rnd(xin);
    std::vector<long long> off(B);
    std::vector<int> active(B), none(1, 0);
    for (int b = 0; b < B; ++b) off[b] = b % 3 == 1 ? (long long)3 * N * B : 0, active[b] = b % 7 != 3;
    std::vector<cd> y((size_t)3 * N * B, cmk(-7.0, -7.0));
    GatherArgs<C> g = {grid.data(), xin.data(), off.data(), B, none.data(), 0, cs.data(), S4.data(), Nx, Ny, ncx, ncy, ncz,
                       row_start.data(), blk.data(), blocks.data(), 1.7, active.data(), y.data()};
    g.groups = groups.data();
    g.n_groups = (int)groups.size();
    kernel(g);
    double num = 0.0, den = 0.0;
    bool kept = true;
    for (int t = 0; t < N; ++t) {
        const int cx = cube[t] % ncx, cy = cube[t] / ncx % ncy, cz = cube[t] / (ncx * ncy);
        for (int b = 0; b < B; ++b) {
            cd a[3] = {};
            for (int j = 0; j < 27; ++j) {
                const size_t p = (2 * cx + j % 3) + (size_t)Nx * ((2 * cy + j / 3 % 3) + (size_t)Ny * (2 * cz + j / 9));
                for (int r = 0; r < 3; ++r)
                    a[r] = cadd(a[r], csub(cmul(to<cd>(Prec<cd>::from(S4[((size_t)t * 27 + j) * 4 + 1 + r])), Prec<cd>::from(grid[(p * 4 + 3) * B + b])),
                                           cscale(cmul(Prec<cd>::from(S4[((size_t)t * 27 + j) * 4]), Prec<cd>::from(grid[(p * 4 + r) * B + b])), 1.7)));
            }
            for (int64_t e = row_start[t]; e < row_start[t + 1]; ++e)
                for (int i = 0; i < 3; ++i)
                    for (int j = 0; j < 3; ++j) {
                        const cf *m = &blocks[(size_t)(blk[e] & 0x7fffffffu) * 9];
                        a[i] = cadd(a[i], cmul(Prec<cd>::from(blk[e] >> 31 ? m[j + 3 * i] : m[i + 3 * j]),
                                               Prec<cd>::from(xin[off[b] + (size_t)(3 * col[e] + j) * B + b])));
                    }
            for (int r = 0; r < 3; ++r) {
                const cd got = y[(size_t)(3 * t + r) * B + b];
                if (!active[b]) {
                    kept &= got.x == -7.0 && got.y == -7.0;
                    continue;
                }
                num += cabs2(csub(got, a[r]));
                den += cabs2(a[r]);
            }
        }
    }
    const double err = std::sqrt(num / den);
    const bool ok = err < (sizeof(C) == 16 ? 1e-13 : 1e-5) && kept;
    if (!ok) ++failures;
    std::printf("%s %s B=%3d, %zu row groups: rel.err %.2e%s %s\n", what, sizeof(C) == 16 ? "c128" : "c64 ", B, groups.size(), err,
                kept ? "" : ", inactive slots written", ok ? "ok" : "FAIL");
}

template <typename C, int SB, int NS>
static void rows(int B, std::mt19937_64 &rng) {
    char what[32];
    std::snprintf(what, sizeof(what), "rows %2d x %d", SB, NS);
    run_case<C>(what, B, rng, [](const GatherArgs<C> &g) { rows_kernel<C, SB, NS>(g); });
}
template <int SB>
static void cols(int B, std::mt19937_64 &rng) {
    char what[32];
    std::snprintf(what, sizeof(what), "cols %2d", SB);
    run_case<cd>(what, B, rng, [](const GatherArgs<cd> &g) { cols_kernel<cd, SB>(g); });
}

// equal parts of at most ROW_GT rows, each tet once
static void check_groups() {
    for (int n = 0; n <= 40; ++n) {
        std::vector<int2> q;
        add_row_groups(q, 3, 100, n);
        int t = 100;
        bool ok = (int)q.size() == (n + ROW_GT - 1) / ROW_GT;
        for (auto &a : q) {
            ok &= a.x == 3 && a.y >> 3 == t && (a.y & 7) >= 1 && (a.y & 7) <= ROW_GT;
            t += a.y & 7;
        }
        if (!ok || t != 100 + n) ++failures, std::printf("row groups of %d tets FAIL\n", n);
    }
}

int main() {
    std::mt19937_64 rng(17);
    check_groups();
    for (int B : {33, 64, 70, 112}) rows<cd, 32, 2>(B, rng), rows<cf, 32, 2>(B, rng);
    for (int B : {33, 48, 70}) rows<cd, 32, 1>(B, rng);
    for (int B : {17, 32, 48}) rows<cf, 32, 1>(B, rng);
    for (int B : {9, 16}) rows<cf, 16, 1>(B, rng);
    for (int B : {5, 8}) rows<cf, 8, 1>(B, rng);
    cols<2>(1, rng), cols<2>(2, rng), cols<4>(3, rng), cols<4>(4, rng);
    cols<8>(5, rng), cols<8>(8, rng), cols<16>(9, rng), cols<16>(16, rng), cols<32>(17, rng), cols<32>(32, rng);
    std::printf("%d failures\n", failures);
    return failures ? 1 : 0;
}
