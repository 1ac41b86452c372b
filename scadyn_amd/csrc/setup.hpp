// Setup-kernel launchers (FP64).
#pragma once

#include "internal.hpp"

namespace scadyn {

struct GridDesc {
    double min[3];
    double delta, box_delta;
    int Nx, Ny, Nz;
    int ncx, ncy, ncz;
};

void upload_tables(hipStream_t s);
const double *host_tet24_p();
const double *host_tet24_w();
const double *host_tri7_p();
const double *host_tri7_w();

// cube98: the 98 sample points, times 2 box_delta
void launch_projection(const double *tcoord, const double *vol, const int *tet_cube, const GridDesc &gd,
                       double k, const cd *WW, const double *cube98, cd *S4, int N, hipStream_t s);
void launch_green_grid(cd *A, const GridDesc &gd, int Lx, int Ly, int Lz, double k, hipStream_t s);
void launch_fg_octant(const cd *F, cd *fg, int Lx, int Ly, int Lz, hipStream_t s);
void launch_pg_table(cd *Gtab, const GridDesc &gd, double k, hipStream_t s);
// Near-zone pairs in the reference's storage order (src/precorrection.f90:182-258:
// test cube, near cube, test tet, basis tet with reference id >= the test
// tet's): internal ids PT[p], PB[p] and cube offset PO[p] = (dx+1) + 3(dy+1) +
// 9(dz+1).  self[t]: the block of tet t with itself.  With ent_blk also the block id
// (| BLK_TRANSPOSE) and column tet of every row entry.  pos (27 N) and tot (N_cubes)
// are scratch.
void launch_near_pairs(const int *cube_start, const int *perm, const int64_t *row_start, const GridDesc &gd,
                       uint32_t *pos, uint32_t *tot, int *PT, int *PB, uint8_t *PO, uint32_t *self,
                       int *ent_col, uint32_t *ent_blk, hipStream_t s);
// reach: a bound on the distance between points of two tets of the near zone
void launch_near_blocks(const int *PT, const int *PB, const uint8_t *POFF, const uint32_t *self, long long P, int N,
                        const double *tcoord, const double *vol, const cd *param, const cd *S4, const cd *Gtab,
                        double k, double reach, cf *blocks, hipStream_t s);
void launch_vswf(const double *tcoord, const double *vol, int N, int Nmax, double k, cd *mat, int ncol,
                 hipStream_t s);

}  // namespace scadyn
