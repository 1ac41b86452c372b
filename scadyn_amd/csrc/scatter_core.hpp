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

// Which kernel takes a batch of B on a grid of so many nodes.  Few nodes: as many lane
// groups as fit share each node's tets, to keep the chip busy.  Many: they only add
// exchanges, about eight lanes to a node are best; and lanes past B idle, so that
// one thread per (node, slot) wins for widths well below SB.  From 25 slots the
// node blocks of 64-slot chunks.
// us per launch in complex128 (complex64 orders them alike), by grid nodes:
//   3 slots: 16, 8, 4, 2 groups, 99 k nodes 73, 42, 32, 33; 614 k 510, 303, 215, 205;
//     thread per slot 47 and 233
//   5 slots: 8, 4, 2 groups, 50 k 39, 30, 32; 149 k 120, 85, 83; 614 k 531, 372, 335;
//     thread per slot 36, 86 and 306
//   9 slots: 4, 2 groups, 50 k 46, 48; 149 k 141, 133; 614 k 639, 578; thread per slot
//     41, 118 and 456
//   12 slots: 2 groups, 149 k 140, 360 k 328, 614 k 606; thread per slot 142, 375, 565
//   20 slots: 2 groups, 149 k 207, 614 k 942; thread per slot 200 and 840
//   24 slots: 2 groups, 149 k 208, 360 k 508, 614 k 981; thread per slot 219, 547, 922
//   25 slots: 64-slot chunk, 149 k 193; thread per slot 235
// Lines of a multiple of 32 nodes: the narrow kernel's workgroups of 8 or 16 nodes, and
// with them the eight XCDs, keep their place along x from line to line, so that some get
// only the ends of the lines, where a body has few tets (shifting them by one a turn
// took 12 slots below from 430 to 338 us).  A thread per (node, slot) does not where the
// width is no power of two.  64 x 64 x 64 nodes, complex128, us narrow and by threads:
// 3 slots 137 and 114, 5 227 and 148, 7 233 and 183, 12 430 and 234, 24 649 and 412;
// 32 x 32 x 32, 5 slots 32 and 28, 12 48 and 34, 24 75 and 63.
enum Kernel { NARROW, FLAT, BLOCKS };
inline Kernel pick_kernel(int B, long long nodes, int Nx) {
    if (B > 24) return BLOCKS;
    if (Nx % 32 == 0 && nodes >= 1LL << 15 && B >= 3 && (B & (B - 1)) != 0) return FLAT;
    if (nodes >= 1LL << 17 && (B == 9 || B == 10 || (B >= 17 && B <= 20))) return FLAT;
    if (nodes >= 3LL << 17 && (B == 5 || B == 11 || B == 12 || (B >= 21 && B <= 24))) return FLAT;
    return NARROW;
}
// lane groups of the narrow kernel
template <int SB>
inline int pick_groups(long long nodes) {
    if (nodes < 1LL << 15 || SB == 32) return 64 / SB < 16 ? 64 / SB : 16;
    if (SB <= 2) return 8 / SB;
    if (SB == 4) return nodes < 1LL << 19 ? 4 : 2;
    return nodes < 1LL << 16 ? 4 : 2;
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
