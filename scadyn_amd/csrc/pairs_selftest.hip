// Host self-test of the near-zone pair and row kernels' per-lane steps
// (pairs_core.hpp): the pair list, and the rows' column tets and blocks, against the
// reference's loops written out, on grids with empty cubes and cubes of up to 150
// tets; and the share of a lane of two cubes with more pairs than 32 bits count.
//
// Exit status 0 when every list is equal.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>

#include "pairs_core.hpp"

using namespace scadyn;

static int failures = 0, cases = 0;
static void expect(bool ok, const char *what, int a, int b) {
    ++cases;
    if (ok) return;
    ++failures;
    std::printf("%s differs (%d, %d)\n", what, a, b);
}

static void grid(int ncx, int ncy, int ncz, int most, std::mt19937 &rng) {
    GridDesc g = {};
    g.ncx = ncx, g.ncy = ncy, g.ncz = ncz;
    const int nc = ncx * ncy * ncz;
    std::vector<int> cs(1, 0);
    for (int c = 0; c < nc; ++c) cs.push_back(cs.back() + (rng() % 3 ? (int)(rng() % (most + 1)) : 0));
    const int N = cs.back();
    std::vector<int> perm(N);  // reference ids, ascending within a cube
    std::iota(perm.begin(), perm.end(), 0);
    std::shuffle(perm.begin(), perm.end(), rng);
    for (int c = 0; c < nc; ++c) std::sort(perm.begin() + cs[c], perm.begin() + cs[c + 1]);

    // the reference's order: test cube, near cube, test tet, basis tet with id >= the
    // test tet's; and each row's entries by near cube, then column tet
    struct Pair {
        int T, B, o;
    };
    std::vector<Pair> ref;
    std::vector<std::vector<std::pair<int, uint32_t>>> rows(N);
    std::vector<std::vector<std::pair<long long, uint32_t>>> keyed(N);
    for (int c = 0; c < nc; ++c)
        for (int o = 0; o < 27; ++o) {
            const int x = c % ncx + o % 3 - 1, y = c / ncx % ncy + o / 3 % 3 - 1, z = c / (ncx * ncy) + o / 9 - 1;
            if (x < 0 || x >= ncx || y < 0 || y >= ncy || z < 0 || z >= ncz) continue;
            const int b = x + ncx * (y + ncy * z);
            for (int T = cs[c]; T < cs[c + 1]; ++T)
                for (int B = cs[b]; B < cs[b + 1]; ++B) {
                    if (perm[B] < perm[T]) continue;
                    const uint32_t p = (uint32_t)ref.size();
                    ref.push_back({T, B, o});
                    keyed[T].push_back({(long long)o * N + B, p});
                    if (T != B) keyed[B].push_back({(long long)(26 - o) * N + T, p | BLK_TRANSPOSE});
                }
        }
    std::vector<int64_t> row_start(1, 0);
    for (int t = 0; t < N; ++t) {
        std::sort(keyed[t].begin(), keyed[t].end());
        row_start.push_back(row_start.back() + (int64_t)keyed[t].size());
    }

    // the kernels' steps
    std::vector<uint32_t> pos((size_t)27 * N);
    std::vector<Pair> got;
    for (int c = 0; c < nc; ++c) {
        const int t0 = cs[c], n = cs[c + 1] - t0;
        for (int s = 0; s < 27 * n; ++s) {
            int b;
            const int cnt = pairs::kept(cs.data(), perm.data(), pairs::near_cube(c, s / n, g), t0 + s % n, b);
            pos[(size_t)27 * t0 + s] = (uint32_t)got.size();
            for (int i = 0; i < cnt; ++i) got.push_back({t0 + s % n, b + i, s / n});
        }
    }
    bool ok = got.size() == ref.size();
    for (size_t p = 0; ok && p < ref.size(); ++p)
        ok = got[p].T == ref[p].T && got[p].B == ref[p].B && got[p].o == ref[p].o;
    expect(ok, "pair list", N, nc);
    std::vector<int> col((size_t)row_start[N], -1);
    std::vector<uint32_t> blk((size_t)row_start[N], 0xffffffffu);
    for (int c = 0; c < nc; ++c)
        for (int lane = 0; lane < 64; ++lane)
            pairs::fill_rows(cs.data(), perm.data(), g, row_start.data(), pos.data(), col.data(), blk.data(), c, lane);
    ok = true;
    for (int t = 0; t < N; ++t)
        for (size_t e = 0; e < keyed[t].size(); ++e)
            ok &= col[row_start[t] + e] == keyed[t][e].first % N && blk[row_start[t] + e] == keyed[t][e].second;
    expect(ok, "row entries", N, nc);
}

// every 64th of n x m pairs, in order, to the last
static void share(int n, int m, int lane) {
    const long long tot = (long long)n * m;
    long long l = lane;
    bool ok = true;
    pairs::lane_pairs(n, m, lane, [&](int i, int j) {
        ok &= l == (long long)i * m + j;
        l += 64;
    });
    expect(ok && l >= tot && l < tot + 64, "lane's pairs", n, m);
}

int main() {
    std::mt19937 rng(11);
    grid(1, 1, 1, 6, rng);
    grid(4, 3, 5, 9, rng);
    grid(2, 6, 1, 17, rng);
    grid(3, 1, 2, 150, rng);
    for (int n : {1, 5, 63, 64, 65, 200})
        for (int m : {1, 2, 63, 64, 65, 131})
            for (int lane : {0, 1, 37, 63}) share(n, m, lane);
    for (int lane : {0, 63}) {
        share(46341, 46341, lane);  // the first square beyond 2^31
        share(65536, 65536, lane);  // 2^32
    }
    std::printf("%d cases, %d failures\n", cases, failures);
    return failures != 0;
}
