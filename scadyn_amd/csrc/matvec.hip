// Batched pFFT matvec y = A x (compute_Ax2, src/gmres_module.f90:57-176).
//
// Multi-vectors are RHS-innermost: element (row, slot b) of a batch of B
// vectors sits at row*B + b, rows being 3*t + c in the internal (cube-sorted)
// tet order.  Grid buffers are [z][y][x][4][B]: channel 0..2 carry S^T x_c
// (the three "Y" convolutions) and channel 3 carries Sx^T x_x + Sy^T x_y +
// Sz^T x_z; by linearity this one convolution replaces the reference's three
// divergence convolutions (:122-144), whose gathered sum it equals.
#include <type_traits>

#include "matvec.hpp"
#include "gather_core.hpp"
#include "scatter_core.hpp"

namespace scadyn {

// ---- narrow batches (up to 32 slots) -------------------------------------------
// One wave per tet (gather) or a few nodes (scatter): the lanes are SB slots (a power
// of two >= B) x groups that share the sum's terms, combined at the end by a fixed
// exchange over the groups.  A few slots leave nothing to hide a
// serial chain of loads behind, so what bounds these kernels is the number of
// dependent rounds: 160 near tets and 27 nodes per row, about 20 tets per node,
// divided by the groups.  With one thread per (row, slot), which walked them all,
// 1,680 tets x 1 vector took 164 us (gather) and 29 us (scatter), now 13 and 10;
// 24,708 tets x 1 206 and 37, now 95 and 21.
template <typename C, int SB, int END = 64>
__device__ inline C group_sum(C v) {
#pragma unroll
    for (int o = SB; o < END; o <<= 1) {
        v.x += __shfl_xor(v.x, o, 64);
        v.y += __shfl_xor(v.y, o, 64);
    }
    return v;
}

// scatter (scatter_core.hpp); the launch caps the grid, a workgroup strides over nodes
template <typename C, int SB, int G>
__global__ __launch_bounds__(score::THREADS) void k_scatter_narrow(score::ScatterArgs<C> s) {
    constexpr int PER = score::nodes_per_group<SB, G>();
    const int b = threadIdx.x & (SB - 1), g = (threadIdx.x / SB) % G;
    const int bl = b < s.B ? b : s.B - 1;  // idle lanes load the last slot and store nothing
    const long long nodes = (long long)s.Nx * s.Ny * s.Nz;
    // a node's lanes leave together
    for (long long p = (long long)blockIdx.x * PER + threadIdx.x / (SB * G); p < nodes; p += (long long)gridDim.x * PER) {
        C a[4];
        score::node_share<C, G>(s, p, bl, g, a);
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = group_sum<C, SB, SB * G>(a[c]);
        if (g == 0 && b < s.B) score::write_node(s, p, b, a);
    }
}

// one thread per (node, slot), the node's tets in order
template <typename C>
__global__ __launch_bounds__(score::THREADS) void k_scatter_flat(score::ScatterArgs<C> s) {
    const long long tot = (long long)s.Nx * s.Ny * s.Nz * s.B;
    for (long long e = blockIdx.x * (long long)score::THREADS + threadIdx.x; e < tot;
         e += (long long)gridDim.x * score::THREADS) {
        const long long p = e / s.B;
        const int b = (int)(e - p * s.B);
        C a[4];
        score::node_share<C, 1>(s, p, b, 0, a);
        score::write_node(s, p, b, a);
    }
}

// gather (sparse_eps_matmul, src/sparse.f90:47-77) + Y_aim = Y2 - k^2 Y (:148-153)
// + symmetric near-zone blocks (matmul_Acorr_const, src/sparse_mat.f90:96-123)
template <typename C, int SB>
__global__ __launch_bounds__(256) void k_gather_narrow(
    const C *__restrict__ grid, const C *__restrict__ xin, const long long *__restrict__ in_off, int B,
    int N, const int *__restrict__ tet_cube, const C *__restrict__ S4, int Nx, int Ny, int ncx, int ncy,
    const int64_t *__restrict__ row_start, const int *__restrict__ ent_col,
    const uint32_t *__restrict__ ent_blk, const cf *__restrict__ blocks, double k2,
    const int *__restrict__ slot_active, cd *__restrict__ y) {
    constexpr int G = 64 / SB;
    typedef typename Prec<C>::real R;
    const int lane = threadIdx.x & 63, b = lane & (SB - 1), g = lane / SB;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int t = blockIdx.x * 4 + wib;
    if (t >= N) return;
    const int bl = b < B ? b : B - 1;
    C a0 = Prec<C>::zero(), a1 = a0, a2 = a0;
    {
        const int c = tet_cube[t];
        const int cx = c % ncx, cy = (c / ncx) % ncy, cz = c / (ncx * ncy);
        const size_t base = (size_t)(2 * cx) + (size_t)Nx * ((size_t)(2 * cy) + (size_t)Ny * (2 * cz));
        const C *s = S4 + (size_t)t * 108;
        const R kk = (R)k2;
        for (int j = g; j < 27; j += G) {
            const C *gp = grid + (base + j % 3 + (size_t)Nx * ((j / 3) % 3 + (size_t)Ny * (j / 9))) * 4 * B + bl;
            const C g3 = gp[(size_t)3 * B];
            const C *sj = s + j * 4;
            const C s0 = cscale(sj[0], -kk);
            cfma(a0, s0, gp[0]);
            cfma(a1, s0, gp[(size_t)B]);
            cfma(a2, s0, gp[(size_t)2 * B]);
            cfma(a0, sj[1], g3);
            cfma(a1, sj[2], g3);
            cfma(a2, sj[3], g3);
        }
    }
    const C *xb = xin + in_off[bl] + bl;
    const int64_t q1 = row_start[t + 1];
#pragma unroll 2
    for (int64_t q = row_start[t] + g; q < q1; q += G) {
        const int col = ent_col[q];
        const uint32_t eb = ent_blk[q];
        const cf *a = blocks + (size_t)(eb & 0x7fffffffu) * 9;
        const C x0 = xb[(size_t)(3 * col) * B], x1 = xb[(size_t)(3 * col + 1) * B], x2 = xb[(size_t)(3 * col + 2) * B];
        // A(i, j) at i + 3 j, or of the transposed block at j + 3 i
        const int si = eb & 0x80000000u ? 3 : 1, sj = 4 - si;
        cfma(a0, Prec<C>::from(a[0]), x0);
        cfma(a0, Prec<C>::from(a[sj]), x1);
        cfma(a0, Prec<C>::from(a[2 * sj]), x2);
        cfma(a1, Prec<C>::from(a[si]), x0);
        cfma(a1, Prec<C>::from(a[4]), x1);
        cfma(a1, Prec<C>::from(a[si + 2 * sj]), x2);
        cfma(a2, Prec<C>::from(a[2 * si]), x0);
        cfma(a2, Prec<C>::from(a[2 * si + sj]), x1);
        cfma(a2, Prec<C>::from(a[8]), x2);
    }
    a0 = group_sum<C, SB>(a0);
    a1 = group_sum<C, SB>(a1);
    a2 = group_sum<C, SB>(a2);
    if (g == 0 && b < B && (!slot_active || slot_active[b])) {  // inactive slots are not written
        cd *yo = y + (size_t)(3 * t) * B + b;
        yo[0] = Prec<cd>::from(a0);
        yo[(size_t)B] = Prec<cd>::from(a1);
        yo[(size_t)2 * B] = Prec<cd>::from(a2);
    }
}

// the same with one thread per (row, slot), the row's terms in order
template <typename C>
__global__ __launch_bounds__(256) void k_gather_flat(
    const C *__restrict__ grid, const C *__restrict__ xin, const long long *__restrict__ in_off, int B,
    int N, const int *__restrict__ tet_cube, const C *__restrict__ S4, int Nx, int Ny, int ncx, int ncy,
    const int64_t *__restrict__ row_start, const int *__restrict__ ent_col,
    const uint32_t *__restrict__ ent_blk, const cf *__restrict__ blocks, double k2,
    const int *__restrict__ slot_active, cd *__restrict__ y) {
    const long long tot = (long long)N * B;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < tot;
         e += (long long)gridDim.x * blockDim.x) {
        const int b = (int)(e % B);
        const int t = (int)(e / B);
        cd *yo = y + (size_t)(3 * t) * B + b;
        if (slot_active && !slot_active[b]) continue;  // inactive slots are not written
        const int c = tet_cube[t];
        const int cx = c % ncx, cy = (c / ncx) % ncy, cz = c / (ncx * ncy);
        const size_t base = (size_t)(2 * cx) + (size_t)Nx * ((size_t)(2 * cy) + (size_t)Ny * (2 * cz));
        const C *s = S4 + (size_t)t * 108;
        C Y0 = Prec<C>::zero(), Y1 = Y0, Y2 = Y0, Z0 = Y0, Z1 = Y0, Z2 = Y0;
        for (int jz = 0; jz < 3; ++jz)
            for (int jy = 0; jy < 3; ++jy)
                for (int jx = 0; jx < 3; ++jx) {
                    const int j = jx + 3 * jy + 9 * jz;
                    const size_t node = base + jx + (size_t)Nx * (jy + (size_t)Ny * jz);
                    const C *g = grid + node * 4 * B + b;
                    const C g0 = g[0], g1 = g[(size_t)B], g2 = g[(size_t)2 * B], g3 = g[(size_t)3 * B];
                    const C *sj = s + j * 4;
                    cfma(Y0, sj[0], g0);
                    cfma(Y1, sj[0], g1);
                    cfma(Y2, sj[0], g2);
                    cfma(Z0, sj[1], g3);
                    cfma(Z1, sj[2], g3);
                    cfma(Z2, sj[3], g3);
                }
        // near zone
        const C *xb = xin + in_off[b] + b;
        C n0 = Prec<C>::zero(), n1 = n0, n2 = n0;
        for (int64_t q = row_start[t]; q < row_start[t + 1]; ++q) {
            const int col = ent_col[q];
            const uint32_t eb = ent_blk[q];
            const cf *a = blocks + (size_t)(eb & 0x7fffffffu) * 9;
            const C x0 = Prec<C>::from(xb[(size_t)(3 * col) * B]),
                    x1 = Prec<C>::from(xb[(size_t)(3 * col + 1) * B]),
                    x2 = Prec<C>::from(xb[(size_t)(3 * col + 2) * B]);
            C m[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) m[i] = Prec<C>::from(a[i]);
            if (eb & 0x80000000u) {
                // transpose: y_i += sum_j A(j,i) x_j ; A(i,j) at i + 3j
                cfma(n0, m[0], x0); cfma(n0, m[1], x1); cfma(n0, m[2], x2);
                cfma(n1, m[3], x0); cfma(n1, m[4], x1); cfma(n1, m[5], x2);
                cfma(n2, m[6], x0); cfma(n2, m[7], x1); cfma(n2, m[8], x2);
            } else {
                cfma(n0, m[0], x0); cfma(n0, m[3], x1); cfma(n0, m[6], x2);
                cfma(n1, m[1], x0); cfma(n1, m[4], x1); cfma(n1, m[7], x2);
                cfma(n2, m[2], x0); cfma(n2, m[5], x1); cfma(n2, m[8], x2);
            }
        }
        typedef typename Prec<C>::real R;
        const R kk = (R)k2;
        yo[0] = Prec<cd>::from(cadd(n0, csub(Z0, cscale(Y0, kk))));
        yo[(size_t)B] = Prec<cd>::from(cadd(n1, csub(Z1, cscale(Y1, kk))));
        yo[(size_t)2 * B] = Prec<cd>::from(cadd(n2, csub(Z2, cscale(Y2, kk))));
    }
}

// ---- on-chip reuse variants (slots in chunks of 64) --------------------------
// Scatter, one wave per 2x2x2 block of grid nodes (2a..2a+1, 2b..2b+1, 2c..2c+1),
// ceil(N/2) blocks per axis:
// every node of the block lies in the boxes of the same <= 8 cubes (a-1..a per
// axis), so the wave loads each of their tets' x once for all 8 nodes, instead
// of once per node.  Per node the sum runs over cubes and tets in the same
// order: z, y, x.
template <typename C>
__global__ __launch_bounds__(256) void k_scatter_blk_w64(const C *__restrict__ xin,
                                                         const long long *__restrict__ in_off, int B,
                                                         const int *__restrict__ cube_start,
                                                         const C *__restrict__ S4, int Nx, int Ny, int Nz,
                                                         int ncx, int ncy, int ncz, C *__restrict__ grid) {
    const int lane = threadIdx.x & 63;
    const int nch = (B + 63) >> 6;  // last chunk may be partial: lanes >= B load slot B-1, store nothing
    // ceil(N/2) blocks per axis cover every node (nodes beyond the cubes' boxes get zeros)
    const int nbx = (Nx + 1) >> 1, nby = (Ny + 1) >> 1, nbz = (Nz + 1) >> 1;
    const long long nw = (long long)nbx * nby * nbz * nch;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // items (node block, slot chunk) with the chunk fastest; a chunk-major order
    // with XCD-contiguous workgroup ranges (as in the gather) measured slower
    for (long long w = (long long)blockIdx.x * 4 + wib; w < nw; w += (long long)gridDim.x * 4) {
        const long long blk = w / nch;
        const int braw = (int)(w - blk * nch) * 64 + lane;
        const bool valid = braw < B;
        const int b = valid ? braw : B - 1;
        const int ba = (int)(blk % nbx), bb = (int)((blk / nbx) % nby), bc = (int)(blk / ((long long)nbx * nby));
        const C *xb = xin + in_off[b] + b;
        C acc[2][2][2][4];
#pragma unroll
        for (int iz = 0; iz < 2; ++iz)
#pragma unroll
            for (int iy = 0; iy < 2; ++iy)
#pragma unroll
                for (int ix = 0; ix < 2; ++ix)
#pragma unroll
                    for (int ch = 0; ch < 4; ++ch) acc[iz][iy][ix][ch] = Prec<C>::zero();
        // cube (ba-1+dx, bb-1+dy, bc-1+dz); node 2ba+ix is in its box when dx = 1
        // (local index ix) or dx = 0 and ix = 0 (local index 2)
#pragma unroll
        for (int dz = 0; dz < 2; ++dz) {
            const int cz = bc - 1 + dz;
            if (cz < 0 || cz >= ncz) continue;
#pragma unroll
            for (int dy = 0; dy < 2; ++dy) {
                const int cy = bb - 1 + dy;
                if (cy < 0 || cy >= ncy) continue;
#pragma unroll
                for (int dx = 0; dx < 2; ++dx) {
                    const int cx = ba - 1 + dx;
                    if (cx < 0 || cx >= ncx) continue;
                    const int c = cx + ncx * (cy + ncy * cz);
                    const int t1 = cube_start[c + 1];
                    for (int t = cube_start[c]; t < t1; ++t) {
                        const C x0 = Prec<C>::from(xb[(size_t)(3 * t) * B]),
                                x1 = Prec<C>::from(xb[(size_t)(3 * t + 1) * B]),
                                x2 = Prec<C>::from(xb[(size_t)(3 * t + 2) * B]);
                        const C *st = S4 + (size_t)t * 108;
#pragma unroll
                        for (int iz = 0; iz < 2; ++iz) {
                            if (dz == 0 && iz == 1) continue;
                            const int jz = dz ? iz : 2;
#pragma unroll
                            for (int iy = 0; iy < 2; ++iy) {
                                if (dy == 0 && iy == 1) continue;
                                const int jy = dy ? iy : 2;
#pragma unroll
                                for (int ix = 0; ix < 2; ++ix) {
                                    if (dx == 0 && ix == 1) continue;
                                    const int jx = dx ? ix : 2;
                                    const C *s = st + (jx + 3 * jy + 9 * jz) * 4;
                                    C *a = acc[iz][iy][ix];
                                    const C s0 = s[0];
                                    cfma(a[0], s0, x0);
                                    cfma(a[1], s0, x1);
                                    cfma(a[2], s0, x2);
                                    cfma(a[3], s[1], x0);
                                    cfma(a[3], s[2], x1);
                                    cfma(a[3], s[3], x2);
                                }
                            }
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int iz = 0; iz < 2; ++iz)
#pragma unroll
            for (int iy = 0; iy < 2; ++iy)
#pragma unroll
                for (int ix = 0; ix < 2; ++ix) {
                    const int px = 2 * ba + ix, py = 2 * bb + iy, pz = 2 * bc + iz;
                    if (!valid || px >= Nx || py >= Ny || pz >= Nz) continue;
                    C *gp = grid + ((size_t)px + (size_t)Nx * ((size_t)py + (size_t)Ny * pz)) * 4 * B + b;
#pragma unroll
                    for (int ch = 0; ch < 4; ++ch) gp[(size_t)ch * B] = acc[iz][iy][ix][ch];
                }
    }
}

// Gather + near zone with the per-tet operands staged in LDS, one 64-thread
// workgroup per (row group of a cube, chunk of slots); the steps are in
// gather_core.hpp (shared with the host self-test of the row groups).  Staging keeps many
// operand fetches in flight (wave-uniform operands read through scalar loads
// would wait on each other).
template <typename C, int NT, int VC, int SB, int NS>
__device__ __forceinline__ void gather_pass(const gcore::GatherArgs<C> &g, const gcore::Item &it, int chunk, int lane,
                                            unsigned char *smraw) {
    C *sm = (C *)smraw;         // S* records of the group's tets
    cf *smb = (cf *)smraw;      // then the near-zone blocks of each chunk
    using namespace gcore;
    const int rows = it.t1 - it.t0;
    const Slots<SB, NS> sl = lane_slots<SB, NS>(g, chunk, lane);
    C acc[NT][3][NS];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < NS; ++i) acc[u][c][i] = Prec<C>::zero();
    long long off[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) off[i] = g.in_off[sl.s[i]] + sl.s[i];
    __syncthreads();  // the previous item's reads of sm are done
    stage_s4(g, it.t0, rows, lane, sm);
    __syncthreads();
    grid_rows<C, NT, NS>(g, it, sl.s, sm + sl.grp * NT * 108, acc);
    // a lane stages one block of the first and one of the last ROW_GT / 2 rows
    constexpr int HT = ROW_GT / 2;
    const int64_t rs0 = lane_row_start<C, HT, VC>(g, it.t0, min(rows, HT), lane),
                  rs1 = lane_row_start<C, HT, VC>(g, it.t0 + HT, rows - HT, lane);
    int q = 0;
    for_near_cubes(g, it, [&](int c0, int c1) {
        for (int v0 = c0; v0 < c1; v0 += VC) {
            const int nv = min(VC, c1 - v0);
            __syncthreads();
            stage_blocks<C, HT, VC>(g, min(rows, HT), nv, q, lane, rs0, smb);
            if (rows > HT) stage_blocks<C, HT, VC>(g, rows - HT, nv, q, lane, rs1, smb + HT * VC * 9);
            __syncthreads();
            chunk_rows<C, NT, VC, NS>(g, off, v0, nv, smb + sl.grp * NT * VC * 9, acc);
            q += nv;
        }
    });
    write_rows<C, NT, SB, NS>(g, it, sl, acc);
}

template <typename C, int VC, int SB, int NS>
__global__ __launch_bounds__(64, 3) void k_gather_lds(gcore::GatherArgs<C> g) {
    using namespace gcore;
    constexpr int G = 64 / SB, NTMAX = (ROW_GT + G - 1) / G;  // lane groups, rows of each
    static_assert(NTMAX <= 3 && ROW_GT / 2 * VC <= 64, "passes below; one block of each half per lane");
    __shared__ __align__(16) unsigned char sm[Shape<C, G * NTMAX, VC>::BYTES];
    const int lane = threadIdx.x;
    const long long nw = (long long)g.n_groups * ((g.B + SB * NS - 1) / (SB * NS));
    for (long long b = blockIdx.x; b < nw; b += gridDim.x) {
        // one item per workgroup when the grid covers all items (the launch
        // below); a grid-stride remainder keeps plain order
        const long long w = nw == gridDim.x ? xcd_remap(b, nw) : b;
        const int chunk = (int)(w / g.n_groups);
        const Item it = group_item(g, (int)(w - (long long)chunk * g.n_groups));
        const int nt = (it.t1 - it.t0 + G - 1) / G;  // wave-uniform
#define PASS(N)                                                                          \
    if constexpr (NTMAX >= N)                                                            \
        if (nt == N) gather_pass<C, N, VC, SB, NS>(g, it, chunk, lane, sm);
        PASS(1) PASS(2) PASS(3)
#undef PASS
    }
}

// complex128, up to 32 slots (up to 4 on large meshes): three rows at a time, the columns shared by the lane
// groups (24,708 tets x 7: 153 us against 231 with the rows shared; complex64 keeps
// the order of its sums)
template <typename C, int NT, int VC, int SB>
__device__ __forceinline__ void gather_cols(const gcore::GatherArgs<C> &g, const gcore::Item &it, int tp, int chunk,
                                            int lane, unsigned char *smraw) {
    C *sm = (C *)smraw;
    cf *smb = (cf *)smraw;
    using namespace gcore;
    const Slots<SB, 1> sl = lane_slots<SB, 1>(g, chunk, lane);
    C acc[NT][3];
    zero_acc<C, NT>(acc);
    const long long off = g.in_off[sl.s[0]] + sl.s[0];
    __syncthreads();  // the previous rows' reads of sm are done
    stage_s4(g, tp, NT, lane, sm);
    __syncthreads();
    grid_share<C, NT, SB>(g, it, sl, sm, acc);
    const int64_t rs = lane_row_start<C, ROW_GT / 2, VC>(g, tp, NT, lane);
    int q = 0;
    for_near_cubes(g, it, [&](int c0, int c1) {
        for (int v0 = c0; v0 < c1; v0 += VC) {
            const int nv = min(VC, c1 - v0);
            __syncthreads();
            stage_blocks<C, ROW_GT / 2, VC>(g, NT, nv, q, lane, rs, smb);
            __syncthreads();
            chunk_share<C, NT, VC, SB>(g, sl, off, v0, nv, smb, acc);
            q += nv;
        }
    });
    const bool write = sl.grp == 0 && sl.ok[0] && (!g.slot_active || g.slot_active[sl.s[0]]);
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const C v = group_sum<C, SB>(acc[u][c]);
            if (write) g.y[(size_t)(3 * (tp + u) + c) * g.B + sl.s[0]] = Prec<cd>::from(v);
        }
}

template <typename C, int VC, int SB>
__global__ __launch_bounds__(64, 3) void k_gather_cols(gcore::GatherArgs<C> g) {
    using namespace gcore;
    constexpr int HT = ROW_GT / 2;
    static_assert(HT == 3 && HT * VC <= 64, "passes below; one block per lane");
    __shared__ __align__(16) unsigned char sm[Shape<C, HT, VC>::BYTES];
    const int lane = threadIdx.x;
    const long long nw = (long long)g.n_groups * 2 * ((g.B + SB - 1) / SB);
    for (long long b = blockIdx.x; b < nw; b += gridDim.x) {
        const long long w = nw == gridDim.x ? xcd_remap(b, nw) : b;
        const int chunk = (int)(w / (2 * g.n_groups));
        const int i = (int)(w - (long long)chunk * 2 * g.n_groups);
        const Item it = group_item(g, i >> 1);
        const int tp = it.t0 + (i & 1 ? HT : 0), nt = min(HT, it.t1 - tp);  // wave-uniform
        if (nt == 1) gather_cols<C, 1, VC, SB>(g, it, tp, chunk, lane, sm);
        if (nt == 2) gather_cols<C, 2, VC, SB>(g, it, tp, chunk, lane, sm);
        if (nt == 3) gather_cols<C, 3, VC, SB>(g, it, tp, chunk, lane, sm);
    }
}

// The complex64 gather with the near-zone product on the matrix cores
// (v_mfma_f32_16x16x4f32, operand algebra in gather_core.hpp): the grid part
// as k_gather_lds, then per near chunk the blocks staged in LDS as the A
// operand and the column tets' x as the B operand, the output tiles exchanged
// through LDS to the lanes that own the slots (opts.gather_kernel = 1).  FP32
// matrix instructions have twice the FP32 vector rate and the stored
// complex64 blocks need no conversion, but each k-step's operand set-up
// (index decode, LDS read, x load) costs about as many vector instructions as
// the FMAs it replaces: measured 23.0 vs 10.8 ms per launch at 824k tets,
// 59 slots, so the vector-FMA kernel stays the default.
typedef float v4f __attribute__((ext_vector_type(4)));

template <int NT, int GT, int VC>
__device__ __forceinline__ void gather_pass_mf(const gcore::GatherArgs<cf> &g, const gcore::Item &it, int tp,
                                               int lane, unsigned char *smraw) {
    using namespace gcore;
    cf *sm = (cf *)smraw;
    cf *smb = (cf *)smraw;
    float *xb = (float *)smraw;
    // near part first (its output tiles in registers), then the tiles through
    // LDS into the lane's accumulators, then the grid part: the two phases'
    // accumulators are never live together
    constexpr int RT = mf_rows(NT);
    v4f D[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int st = 0; st < 4; ++st) D[rt][st] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const int lo = lane & 15, kq = lane >> 4;
    const int s0 = (it.b & ~63) + lo;  // slot of tile 0 for this lane's B operand; tile st adds 16 st
    long long off[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) off[st] = s0 + 16 * st < g.B ? g.in_off[s0 + 16 * st] : 0;
    const int64_t rsu = lane_row_start<cf, GT, VC>(g, tp, NT, lane);
    int q = 0;
    for_near_cubes(g, it, [&](int c0, int c1) {
        for (int v0 = c0; v0 < c1; v0 += VC) {
            const int nv = min(VC, c1 - v0);
            __syncthreads();  // the previous chunk's (or pass's) reads of the buffer are done
            stage_blocks<cf, GT, VC>(g, NT, nv, q, lane, rsu, smb);
            __syncthreads();
            const int S = (6 * nv + 3) / 4;
            // operands fetched one k-step ahead, so that the loads of step s + 1
            // are in flight while the matrix instructions of step s run
            float bn[4], an[RT];
#pragma unroll
            for (int st = 0; st < 4; ++st) bn[st] = mf_b(g, v0, nv, kq, s0 + 16 * st, off[st], s0 + 16 * st < g.B);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) an[rt] = mf_a(smb, NT, nv, VC, 16 * rt + lo, kq);
            for (int s = 0; s < S; ++s) {
                float bo[4], ao[RT];
#pragma unroll
                for (int st = 0; st < 4; ++st) bo[st] = bn[st];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) ao[rt] = an[rt];
                if (s + 1 < S) {
                    const int kp = 4 * (s + 1) + kq;
#pragma unroll
                    for (int st = 0; st < 4; ++st)
                        bn[st] = mf_b(g, v0, nv, kp, s0 + 16 * st, off[st], s0 + 16 * st < g.B);
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) an[rt] = mf_a(smb, NT, nv, VC, 16 * rt + lo, kp);
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int st = 0; st < 4; ++st)
                        D[rt][st] = __builtin_amdgcn_mfma_f32_16x16x4f32(ao[rt], bo[st], D[rt][st], 0, 0, 0);
            }
            q += nv;
        }
    });
    __syncthreads();  // the last chunk's block reads are done
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int e = 0; e < 4; ++e) xb[mf_xidx(lane, e, rt, st)] = D[rt][st][e];
    __syncthreads();
    cf acc[NT][3];
    zero_acc<cf, NT>(acc);
    mf_combine<NT>(xb, lane, acc);
    __syncthreads();  // the exchange is read before the S* records overwrite it
    stage_s4(g, tp, NT, lane, sm);
    __syncthreads();
    grid_part<cf, NT>(g, it, sm, acc);
    write_out<cf, NT>(g, it, tp, acc);
}

template <int GT, int VC>
__global__ __launch_bounds__(64, 3) void k_gather_mf(gcore::GatherArgs<cf> g) {
    using namespace gcore;
    static_assert(GT == 8, "the pass switch below covers 1..8 row tets");
    constexpr int SB = Shape<cf, GT, VC>::BYTES > MF_XBYTES ? Shape<cf, GT, VC>::BYTES : MF_XBYTES;
    __shared__ __align__(16) unsigned char sm[SB];
    const int lane = threadIdx.x;
    const long long nw = (long long)g.n_ne * ((g.B + 63) >> 6);
    for (long long b = blockIdx.x; b < nw; b += gridDim.x) {
        const long long w = nw == gridDim.x ? xcd_remap(b, nw) : b;
        const Item it = make_item(g, w, lane);
        for (int tp = it.t0; tp < it.t1; tp += GT) {
            switch (min(GT, it.t1 - tp)) {  // wave-uniform
                case 1: gather_pass_mf<1, GT, VC>(g, it, tp, lane, sm); break;
                case 2: gather_pass_mf<2, GT, VC>(g, it, tp, lane, sm); break;
                case 3: gather_pass_mf<3, GT, VC>(g, it, tp, lane, sm); break;
                case 4: gather_pass_mf<4, GT, VC>(g, it, tp, lane, sm); break;
                case 5: gather_pass_mf<5, GT, VC>(g, it, tp, lane, sm); break;
                case 6: gather_pass_mf<6, GT, VC>(g, it, tp, lane, sm); break;
                case 7: gather_pass_mf<7, GT, VC>(g, it, tp, lane, sm); break;
                default: gather_pass_mf<8, GT, VC>(g, it, tp, lane, sm); break;
            }
        }
    }
}

// Gather kernels by width and mesh, us per launch at N tets.
//  * One tet a wave to 4 slots: it reads every block by single lanes, which costs more
//    than it saves once the chip is full, so in complex128 only on small meshes
//    (1,680 tets x 3: 17 us against 30 with k_gather_cols; 12.7 k 74 and 62; 201 k
//    1,415 and 911; thread per slot 155, 161, 1,360).  Complex64 keeps it: another
//    order of its sums can move a mixed solve's iteration counts.
//  * Complex64 of 5 to 8 slots: row groups leave lanes idle (six of eight lane groups
//    have a row, and five of eight lanes a slot); on large meshes one thread per slot
//    is faster (5 slots: 24.7 k 179 us in groups, 179 by threads; 98 k 814 and 728;
//    201 k 1,536 and 1,357; 8 slots: 98 k 825 and 815; 201 k 1,557 and 1,498).
//  * Few rows to a group (fine grids, bodies of many half-empty cubes; the default grid
//    has five to six): a group costs about the same whatever its rows, so there one
//    thread per (row, slot) wins, the wider the batch the fewer rows it takes.
//    43,248 tets, us in groups and by threads: 2.0 rows a group complex128 3 slots 295
//    and 125, 12 431 and 254, 24 654 and 475; complex64 5 slots 374 and 134, 12 400 and
//    208, 24 400 and 382; 3.3 rows complex128 5 slots 278 and 260, 8 306 and 351, 17 641
//    and 525; complex64 5 349 and 221, 12 369 and 329, 16 399 and 430; 55,968 tets, 3.9
//    rows complex64 5 521 and 368, 9 534 and 489; 103,536 tets, 4.3 rows 8 939 and 822.
//    Small meshes leave lanes idle either way (5,472 tets, 2 rows, 12 slots 72 and 76).
//  * Else row groups.
enum GatherKernel { GATHER_NARROW, GATHER_FLAT, GATHER_GROUPS };
static bool few_rows(bool wide, int B, int N, int groups) {
    const double rows = (double)N / std::max(groups, 1);
    if (B >= 32) return false;
    if (N < 8192) return wide && B > 16 && rows < 2.5;
    if (!wide) return B >= 5 && B <= (rows < 2.5 ? 24 : rows < 3.5 ? 12 : rows < 4.0 ? 9 : rows < 4.5 ? 8 : 0);
    int lanes = 4;
    while (lanes < B) lanes *= 2;
    return rows < 2.5 || (rows < 3.5 && B >= 3 && (lanes == 4 || 4 * B <= 3 * lanes));
}
template <typename C>
static GatherKernel pick_gather(int B, int N, int groups) {
    const bool wide = sizeof(C) == 16;
    if (few_rows(wide, B, N, groups)) return GATHER_FLAT;
    if (B <= 4) return wide && N >= 8192 ? GATHER_GROUPS : GATHER_NARROW;
    if (!wide && B <= 8 && N >= (B <= 6 ? 1 << 16 : 3 << 16)) return GATHER_FLAT;
    return GATHER_GROUPS;
}

// f(integral constant SB): the lanes' slots of a narrow batch of B
template <typename F>
static void narrow_slots(int B, F &&f) {
    if (B <= 1)
        f(std::integral_constant<int, 1>{});
    else if (B <= 2)
        f(std::integral_constant<int, 2>{});
    else if (B <= 4)
        f(std::integral_constant<int, 4>{});
    else if (B <= 8)
        f(std::integral_constant<int, 8>{});
    else if (B <= 16)
        f(std::integral_constant<int, 16>{});
    else
        f(std::integral_constant<int, 32>{});
}

template <typename C>
void launch_scatter(const MatvecArgs<C> &a, hipStream_t s) {
    const long long nodes = (long long)a.Nx * a.Ny * a.Nz;
    const score::ScatterArgs<C> sa = {a.xin, a.in_off, a.B,   a.cube_start, a.S4,  a.Nx,
                                      a.Ny,  a.Nz,     a.ncx, a.ncy,        a.ncz, a.grid_in};
    const score::Kernel kern = score::pick_kernel(a.B, nodes, a.Nx);
    if (kern == score::BLOCKS) {
        const long long nw = (long long)((a.Nx + 1) / 2) * ((a.Ny + 1) / 2) * ((a.Nz + 1) / 2) * ((a.B + 63) / 64);
        hipLaunchKernelGGL((k_scatter_blk_w64<C>), dim3(grid_for(nw, 4)), dim3(256), 0, s, a.xin, a.in_off, a.B,
                           a.cube_start, a.S4, a.Nx, a.Ny, a.Nz, a.ncx, a.ncy, a.ncz, a.grid_in);
    } else if (kern == score::FLAT) {
        hipLaunchKernelGGL((k_scatter_flat<C>), dim3(grid_for(nodes * a.B, score::THREADS)), dim3(score::THREADS), 0, s,
                           sa);
    } else {
        narrow_slots(a.B, [&](auto sb) {
            constexpr int SB = decltype(sb)::value;
            const int groups = score::pick_groups<SB>(nodes);
            auto go = [&](auto gg) {
                constexpr int G = decltype(gg)::value;
                if constexpr (SB * G <= 64)
                    hipLaunchKernelGGL((k_scatter_narrow<C, SB, G>),
                                       dim3(grid_for(nodes, score::nodes_per_group<SB, G>())), dim3(score::THREADS), 0,
                                       s, sa);
            };
            if (groups == 16)
                go(std::integral_constant<int, 16>{});
            else if (groups == 8)
                go(std::integral_constant<int, 8>{});
            else if (groups == 4)
                go(std::integral_constant<int, 4>{});
            else
                go(std::integral_constant<int, 2>{});
        });
    }
    HIP_CHECK(hipGetLastError());
}

template <typename C>
void launch_gather_near(const MatvecArgs<C> &a, hipStream_t s) {
    const GatherKernel kern = pick_gather<C>(a.B, a.N, a.n_groups);
    if (kern == GATHER_NARROW) {
        narrow_slots(a.B, [&](auto sb) {
            constexpr int SB = decltype(sb)::value;
            if constexpr (SB <= 4)
                hipLaunchKernelGGL((k_gather_narrow<C, SB>), dim3((unsigned)((a.N + 3) / 4)), dim3(256), 0, s,
                                   a.grid_out, a.xin, a.in_off, a.B, a.N, a.tet_cube, a.S4, a.Nx, a.Ny, a.ncx, a.ncy,
                                   a.row_start, a.ent_col, a.ent_blk, a.blocks, a.k2, a.slot_active, a.y);
        });
        HIP_CHECK(hipGetLastError());
        return;
    }
    if (kern == GATHER_FLAT) {
        hipLaunchKernelGGL((k_gather_flat<C>), dim3(grid_for((long long)a.N * a.B, 256)), dim3(256), 0, s, a.grid_out,
                           a.xin, a.in_off, a.B, a.N, a.tet_cube, a.S4, a.Nx, a.Ny, a.ncx, a.ncy, a.row_start,
                           a.ent_col, a.ent_blk, a.blocks, a.k2, a.slot_active, a.y);
        HIP_CHECK(hipGetLastError());
        return;
    }
    gcore::GatherArgs<C> g = {a.grid_out, a.xin,     a.in_off,    a.B,      a.ne_cubes,
                                    a.n_ne,     a.cube_start, a.S4,      a.Nx,     a.Ny,
                                    a.ncx,      a.ncy,       a.ncz,       a.row_start, a.ent_blk,
                                    a.blocks,   a.k2,        a.slot_active, a.y};
    g.groups = a.groups;
    g.n_groups = a.n_groups;
    if constexpr (std::is_same<C, cf>::value) {
        // half full chunks at least: it costs the same for 8 slots as for 64
        if (a.gather_kernel == 1 && (a.B % 64 == 0 || a.B % 64 >= 32)) {
            hipLaunchKernelGGL((k_gather_mf<gcore::GATHER_GT, gcore::GATHER_VC>), dim3(grid_for((long long)a.n_ne * ((a.B + 63) / 64), 1)),
                               dim3(64), 0, s, g);
            HIP_CHECK(hipGetLastError());
            return;
        }
    }
    using gcore::ROW_VC;
    if constexpr (std::is_same<C, cd>::value)
        if (a.B <= 32) {
            auto cols = [&](auto sb) {
                constexpr int SB = decltype(sb)::value;
                hipLaunchKernelGGL((k_gather_cols<C, ROW_VC, SB>), dim3(grid_for(2LL * a.n_groups, 1)), dim3(64), 0, s, g);
            };
            if (a.B > 16)
                cols(std::integral_constant<int, 32>{});
            else if (a.B > 8)
                cols(std::integral_constant<int, 16>{});
            else if (a.B > 4)
                cols(std::integral_constant<int, 8>{});
            else if (a.B > 2)
                cols(std::integral_constant<int, 4>{});
            else
                cols(std::integral_constant<int, 2>{});
            HIP_CHECK(hipGetLastError());
            return;
        }
    auto rows = [&](auto sb, auto ns) {
        constexpr int SB = decltype(sb)::value, NS = decltype(ns)::value;
        const long long nw = (long long)a.n_groups * ((a.B + SB * NS - 1) / (SB * NS));
        hipLaunchKernelGGL((k_gather_lds<C, ROW_VC, SB, NS>), dim3(grid_for(nw, 1)), dim3(64), 0, s, g);
    };
    typedef std::integral_constant<int, 1> one;
    typedef std::integral_constant<int, 32> half;
    // two slots a lane where that still leaves two waves for each of the 1024 SIMDs
    // (24,708 tets, 64 slots: 789 us against 847 with one; 4,686 tets, 48 slots 275
    // against 233)
    if (a.B > 32 && (long long)a.n_groups * ((a.B + 63) / 64) >= 2048)
        rows(half{}, std::integral_constant<int, 2>{});
    else if (sizeof(C) == 16 || a.B > 16)
        rows(half{}, one{});
    else if constexpr (sizeof(C) == 8) {
        if (a.B > 8)
            rows(std::integral_constant<int, 16>{}, one{});
        else
            rows(std::integral_constant<int, 8>{}, one{});
    }
    HIP_CHECK(hipGetLastError());
}

template void launch_scatter<cd>(const MatvecArgs<cd> &, hipStream_t);
template void launch_scatter<cf>(const MatvecArgs<cf> &, hipStream_t);
template void launch_gather_near<cd>(const MatvecArgs<cd> &, hipStream_t);
template void launch_gather_near<cf>(const MatvecArgs<cf> &, hipStream_t);

}  // namespace scadyn
