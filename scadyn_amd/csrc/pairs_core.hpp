// Near-zone pairs and row entries (src/precorrection.f90:182-258): the per-lane
// steps of the kernels in setup.hip, host+device so that the host self-test runs
// the same code on the CPU.
#pragma once

#include "internal.hpp"
#include "setup.hpp"

namespace scadyn {
namespace pairs {

#define PR_HD __host__ __device__ inline

// cube o = (dx+1) + 3(dy+1) + 9(dz+1) around cube c, -1 outside the grid
PR_HD int near_cube(int c, int o, const GridDesc &g) {
    const int x = c % g.ncx + o % 3 - 1, y = (c / g.ncx) % g.ncy + (o / 3) % 3 - 1, z = c / (g.ncx * g.ncy) + o / 9 - 1;
    if (x < 0 || x >= g.ncx || y < 0 || y >= g.ncy || z < 0 || z >= g.ncz) return -1;
    return x + g.ncx * (y + g.ncy * z);
}
// first tet of [b, e) whose reference id is >= id
PR_HD int first_from(const int *__restrict__ perm, int b, int e, int id) {
    while (b < e) {
        const int m = (b + e) >> 1;
        if (perm[m] < id)
            b = m + 1;
        else
            e = m;
    }
    return b;
}
// basis tets b .. b + (return value) - 1 that test tet T keeps of cube nc (-1: none)
PR_HD int kept(const int *__restrict__ cs, const int *__restrict__ perm, int nc, int T, int &b) {
    b = 0;
    if (nc < 0) return 0;
    b = first_from(perm, cs[nc], cs[nc + 1], perm[T]);
    return cs[nc + 1] - b;
}

// the lane's share of n x m pairs, 64 lanes, the second index fastest.  The indices
// are advanced, not divided out of a running number: two cubes of more than 46,340
// tets have more pairs than 32 bits count.
template <typename F>
PR_HD void lane_pairs(int n, int m, int lane, F &&f) {
    if (m == 0) return;
    const int di = 64 / m, dj = 64 % m;
    for (int i = lane / m, j = lane % m; i < n;) {
        f(i, j);
        i += di;
        j += dj;
        if (j >= m) j -= m, ++i;
    }
}

// the lane's entries of the rows of cube c; pos: first block of each (near cube,
// test tet), see setup.hip
PR_HD void fill_rows(const int *__restrict__ cs, const int *__restrict__ perm, const GridDesc &g,
                     const int64_t *__restrict__ row_start, const uint32_t *__restrict__ pos,
                     int *__restrict__ ent_col, uint32_t *__restrict__ ent_blk, int c, int lane) {
    const int t0 = cs[c], t1 = cs[c + 1], n = t1 - t0;
    if (n == 0) return;
    int col = 0;  // entries of the near cubes before o
    for (int o = 0; o < 27; ++o) {
        const int nc = near_cube(c, o, g);
        if (nc < 0) continue;
        const int b0 = cs[nc], b1 = cs[nc + 1], m = b1 - b0;
        lane_pairs(n, m, lane, [&](int i, int j) {
            const int T = t0 + i, B = b0 + j;
            uint32_t blk;
            if (perm[B] >= perm[T])
                blk = pos[(size_t)27 * t0 + (size_t)o * n + i] + (uint32_t)(B - first_from(perm, b0, b1, perm[T]));
            else
                blk = (pos[(size_t)27 * b0 + (size_t)(26 - o) * m + j] +
                       (uint32_t)(T - first_from(perm, t0, t1, perm[B]))) |
                      BLK_TRANSPOSE;
            const int64_t r = row_start[T] + col + j;
            ent_col[r] = B;
            ent_blk[r] = blk;
        });
        col += m;
    }
}

}  // namespace pairs
}  // namespace scadyn
