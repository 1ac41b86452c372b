// Scatter of narrow batches (sparse_T_matmul, src/sparse.f90:13-43, + vec2arr2):
// the per-lane steps, host+device so that the host self-test runs the same code on
// the CPU.  Node p sums the stencil weights of the tets of the <= 8 cubes whose box
// holds p; SB lanes hold a slot each (SB a power of two >= B) and G lane groups
// share the node's tets.
#pragma once

#include "internal.hpp"

namespace scadyn {
namespace score {

#define SC_HD __host__ __device__ inline

template <typename C>
struct ScatterArgs {
    const C *xin;  // element (row, slot b) at xin[in_off[b] + row B + b]
    const long long *in_off;
    int B;
    const int *cube_start;
    const C *S4;
    int Nx, Ny, Nz, ncx, ncy, ncz;
    C *grid;  // [Nz][Ny][Nx][4][B]
};

constexpr int THREADS = 256;
// nodes of a workgroup
template <int SB, int G>
constexpr int nodes_per_group() {
    return THREADS / (SB * G);
}

// group g's share of the sums of node p, slot b
template <typename C, int G>
SC_HD void node_share(const ScatterArgs<C> &s, long long p, int b, int g, C *a) {
    const int px = (int)(p % s.Nx), py = (int)((p / s.Nx) % s.Ny), pz = (int)(p / ((long long)s.Nx * s.Ny));
    const size_t B = (size_t)s.B;
    const C *xb = s.xin + s.in_off[b] + b;
    C a0 = Prec<C>::zero(), a1 = a0, a2 = a0, a3 = a0;
    // cubes c with 2c <= p <= 2c+2 per axis; those of one x line hold consecutive tets
    const int cx0 = px > 0 ? (px - 1) / 2 : 0, cx1 = s.ncx - 1 < px / 2 ? s.ncx - 1 : px / 2;
    const int cy0 = py > 0 ? (py - 1) / 2 : 0, cy1 = s.ncy - 1 < py / 2 ? s.ncy - 1 : py / 2;
    const int cz0 = pz > 0 ? (pz - 1) / 2 : 0, cz1 = s.ncz - 1 < pz / 2 ? s.ncz - 1 : pz / 2;
    for (int cz = cz0; cz <= cz1; ++cz)
        for (int cy = cy0; cy <= cy1; ++cy) {
            const int line = s.ncx * (cy + s.ncy * cz);
            const int t1 = cx1 >= cx0 ? s.cube_start[line + cx1 + 1] : 0, ts = cx1 >= cx0 ? s.cube_start[line + cx1] : 0;
            const int j = 3 * (py - 2 * cy) + 9 * (pz - 2 * cz);
            for (int t = (cx1 >= cx0 ? s.cube_start[line + cx0] : 0) + g; t < t1; t += G) {
                const int jt = j + px - 2 * (t < ts ? cx0 : cx1);
                const C *w = s.S4 + ((size_t)t * 27 + jt) * 4;
                const C x0 = xb[(size_t)(3 * t) * B], x1 = xb[(size_t)(3 * t + 1) * B], x2 = xb[(size_t)(3 * t + 2) * B];
                const C w0 = w[0];
                cfma(a0, w0, x0);
                cfma(a1, w0, x1);
                cfma(a2, w0, x2);
                cfma(a3, w[1], x0);
                cfma(a3, w[2], x1);
                cfma(a3, w[3], x2);
            }
        }
    a[0] = a0, a[1] = a1, a[2] = a2, a[3] = a3;
}

template <typename C>
SC_HD void write_node(const ScatterArgs<C> &s, long long p, int b, const C *a) {
    C *gp = s.grid + (size_t)p * 4 * (size_t)s.B + b;
    for (int c = 0; c < 4; ++c) gp[(size_t)c * s.B] = a[c];
}

}  // namespace score
}  // namespace scadyn
