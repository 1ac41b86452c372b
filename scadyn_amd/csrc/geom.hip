// Host-side setup: grid, cube boxes, tet -> cube map, near-zone row offsets,
// the 98x27 pseudo-inverse, and FFT length planning.  Integer/indexing work
// that the reference does serially on the host in src/geometry.f90,
// src/sparse_mat.f90:13-60 and src/precorrection.f90:182-258.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "internal.hpp"
#include "fft.hpp"

namespace scadyn {

static inline void cross3(const double *a, const double *b, double *c) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = -a[0] * b[2] + a[2] * b[0];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

void build_geometry(const scadyn_mesh &mesh, const scadyn_opts &opts, HostGeometry &g) {
    if (mesh.n_tet <= 0 || mesh.n_node <= 0 || !mesh.coord || !mesh.etopol || !mesh.param)
        fail(SCADYN_ERR_ARG, "empty mesh or null array");
    if (opts.M_ex != 2) fail(SCADYN_ERR_UNSUPPORTED, "only stencil order M_ex = 2 is implemented");
    if (opts.near_zone != 1) fail(SCADYN_ERR_UNSUPPORTED, "only near_zone = 1 is implemented");
    if (opts.order != 0) fail(SCADYN_ERR_UNSUPPORTED, "only basis order 0 is implemented");
    const int N = mesh.n_tet, Nn = mesh.n_node;
    if (N >= 1 << 28) fail(SCADYN_ERR_UNSUPPORTED, "more than 2^28 tets");
    g.N = N;
    g.Nnode = Nn;
    const double *X = mesh.coord;
    std::vector<double> tc((size_t)N * 12), vol(N);
    double volsum = 0.0;
    for (int t = 0; t < N; ++t) {
        double p[4][3];
        for (int a = 0; a < 4; ++a) {
            int id = mesh.etopol[4 * (size_t)t + a];
            if (id < 1 || id > Nn)
                fail(SCADYN_ERR_ARG, "etopol entry out of range at tet " + std::to_string(t + 1));
            for (int c = 0; c < 3; ++c) p[a][c] = X[3 * (size_t)(id - 1) + c];
        }
        // gradshape determinant (src/common.f90:460-469)
        double J[3][3];
        for (int c = 0; c < 3; ++c) {
            J[c][0] = p[1][c] - p[0][c];
            J[c][1] = p[2][c] - p[0][c];
            J[c][2] = p[3][c] - p[0][c];
        }
        double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                     J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                     J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
        if (!(det > 0.0))
            fail(SCADYN_ERR_ORIENTATION,
                 "Something is wrong (detJ <= 0) at tet " + std::to_string(t + 1));
        // tetra_volume (src/common.f90:255-267)
        double p41[3], p21[3], p31[3], cr[3];
        for (int c = 0; c < 3; ++c) {
            p41[c] = p[3][c] - p[0][c];
            p21[c] = p[1][c] - p[0][c];
            p31[c] = p[2][c] - p[0][c];
        }
        cross3(p21, p31, cr);
        double dt = p41[0] * cr[0] + p41[1] * cr[1] + p41[2] * cr[2];
        vol[t] = std::sqrt(dt * dt) / 6.0;
        volsum += vol[t];
        std::memcpy(&tc[12 * (size_t)t], p, sizeof(p));
    }
    double mn[3], mx[3];
    for (int c = 0; c < 3; ++c) mn[c] = mx[c] = X[c];
    for (int i = 1; i < Nn; ++i)
        for (int c = 0; c < 3; ++c) {
            mn[c] = std::min(mn[c], X[3 * (size_t)i + c]);
            mx[c] = std::max(mx[c], X[3 * (size_t)i + c]);
        }
    // delta with the default-real exponent 1.0/3.0 (src/geometry.f90:88)
    const double third32 = (double)(1.0f / 3.0f);
    double delta = opts.grid_size * 1.0 / opts.M_ex * std::pow(volsum / (double)N, third32);
    int n[3];
    for (int c = 0; c < 3; ++c) {
        n[c] = (int)std::ceil(std::fabs(mx[c] - mn[c]) / delta) + 1;
        n[c] = n[c] + (n[c] + 1) % 2 + 1;  // src/geometry.f90:94-98
    }
    g.Nx = n[0];
    g.Ny = n[1];
    g.Nz = n[2];
    g.delta = delta;
    g.box_delta = delta * opts.M_ex;
    for (int c = 0; c < 3; ++c) g.min_coord[c] = mn[c];
    g.ncx = (g.Nx - 2) / 2;
    g.ncy = (g.Ny - 2) / 2;
    g.ncz = (g.Nz - 2) / 2;
    g.N_cubes = g.ncx * g.ncy * g.ncz;
    // tet -> cube by centroid (src/geometry.f90:13-55, :342-353)
    std::vector<int> cube_of(N);
    for (int t = 0; t < N; ++t) {
        const double *p = &tc[12 * (size_t)t];
        int M[3];
        for (int c = 0; c < 3; ++c) {
            double cp = (p[c] + p[3 + c] + p[6 + c] + p[9 + c]) / 4;
            M[c] = (int)std::floor((cp - mn[c]) / g.box_delta);
        }
        if (M[0] < 0 || M[1] < 0 || M[2] < 0 || M[0] >= g.ncx || M[1] >= g.ncy || M[2] >= g.ncz)
            fail(SCADYN_ERR_GRID, "something is wrong (Point is not in any cube), tet " +
                                      std::to_string(t + 1));
        cube_of[t] = M[0] + g.ncx * M[1] + g.ncx * g.ncy * M[2];
    }
    // stable counting sort by cube: internal order
    g.cube_start.assign(g.N_cubes + 1, 0);
    for (int t = 0; t < N; ++t) g.cube_start[cube_of[t] + 1]++;
    g.N_tet_cube = 0;
    for (int c = 0; c < g.N_cubes; ++c) {
        g.N_tet_cube = std::max(g.N_tet_cube, g.cube_start[c + 1]);
        g.cube_start[c + 1] += g.cube_start[c];
    }
    std::vector<int> fill(g.cube_start.begin(), g.cube_start.end() - 1);
    g.perm.resize(N);
    g.inv.resize(N);
    for (int t = 0; t < N; ++t) {
        int i = fill[cube_of[t]]++;
        g.perm[i] = t;
        g.inv[t] = i;
    }
    g.tet_cube.resize(N);
    g.tcoord.resize((size_t)N * 12);
    g.vol.resize(N);
    g.param.resize(N);
    for (int i = 0; i < N; ++i) {
        int t = g.perm[i];
        g.tet_cube[i] = cube_of[t];
        std::memcpy(&g.tcoord[12 * (size_t)i], &tc[12 * (size_t)t], 12 * sizeof(double));
        g.vol[i] = vol[t];
        g.param[i] = cmk(mesh.param[2 * (size_t)t], mesh.param[2 * (size_t)t + 1]);
    }
}

void build_near_rows(const HostGeometry &g, NearRows &nr) {
    nr.row_start.assign((size_t)g.N + 1, 0);
    int64_t e = 0;
    for (int c = 0; c < g.N_cubes; ++c) {
        const int t0 = g.cube_start[c], t1 = g.cube_start[c + 1];
        if (t0 == t1) continue;
        const int cx = c % g.ncx, cy = (c / g.ncx) % g.ncy, cz = c / (g.ncx * g.ncy);
        // the near cubes of one (z, y) line are consecutive
        int64_t len = 0;
        for (int zz = std::max(cz - 1, 0); zz <= std::min(cz + 1, g.ncz - 1); ++zz)
            for (int yy = std::max(cy - 1, 0); yy <= std::min(cy + 1, g.ncy - 1); ++yy) {
                const int line = g.ncx * (yy + g.ncy * zz);
                len += g.cube_start[line + std::min(cx + 1, g.ncx - 1) + 1] - g.cube_start[line + std::max(cx - 1, 0)];
            }
        for (int t = t0; t < t1; ++t) {
            nr.row_start[t] = e;
            e += len;
        }
    }
    nr.row_start[g.N] = e;
    nr.P = (e + g.N) / 2;
    if (nr.P >= (long long)BLK_TRANSPOSE) fail(SCADYN_ERR_UNSUPPORTED, "too many near-zone blocks");
}

static bool is_smooth(int L) {
    int r = L;
    for (int p : {2, 3, 5, 7})
        while (r % p == 0) r /= p;
    return r == 1;
}

// L = R1 R2 with both radices in the register FFT's set
static bool reg_splittable(int L) {
    for (int r1 = 2; r1 <= 20; ++r1)
        if (L % r1 == 0 && reg_radix_ok(r1) && reg_radix_ok(L / r1)) return true;
    return false;
}

// FFT length for a zero-padded axis of n >= 2N-1 points: the smallest
// 2,3,5,7-smooth length, or a longer one (at most n/8 more points) that the
// two-stage register FFT covers when the smallest does not
int smooth_length(int n) {
    int s0 = std::max(n, 1);
    while (!is_smooth(s0)) ++s0;
    if (reg_splittable(s0)) return s0;
    for (int L = s0 + 1; L <= n + n / 8; ++L)
        if (is_smooth(L) && reg_splittable(L)) return L;
    return s0;
}

std::vector<int> factor_radices(int L) {
    std::vector<int> rad;
    int r = L;
    while (r % 8 == 0) { rad.push_back(8); r /= 8; }
    while (r % 4 == 0) { rad.push_back(4); r /= 4; }
    while (r % 2 == 0) { rad.push_back(2); r /= 2; }
    for (int p : {7, 5, 3})
        while (r % p == 0) { rad.push_back(p); r /= p; }
    if (r != 1) {
        // a prime factor above 7 (reference 2N lengths): one generic stage
        rad.push_back(r);
    }
    return rad;
}

}  // namespace scadyn
