// mg.h -- geometric multigrid preconditioner for the pressure-correction
// system on the Cartesian cell grid.
//
// The reference preconditions its Krylov solvers with ILUT (ilutp.f90,
// solvers.f90:185-199).  Here M^-1 is one V(1,1) cycle:
//   * cell-centred 2x2 coarsening.  The off-diagonal coefficients of a level
//     are about g h dt^2/dx_l^2 times its storage term, a ratio that falls by 4
//     per level; below about 1 a few sweeps act as a level's solve.  The short
//     hierarchy ends at the first level from the fourth on that fits one
//     workgroup; where the ratio there is still above MG_SHORT_RATIO, which
//     leaves the smooth error to Krylov, the deep one goes on to the first level
//     at or below MG_DEEP_RATIO.  (A 200 x 100 grid of 10 m at dt 60 s: 25 x 13
//     cells at ratio 55 and 10.5 pp BiCGStab iterations a solve with the short
//     one, 5.4 with three more levels; 2000 x 1500 cells of 20 m at dt 30 s:
//     63 x 47 at 0.3, where more levels save nothing.)  The FP32 form and the
//     telescoping grids stay with the short one.  With the deep one their pp
//     iterations would fall (200 x 100 FP32 at dt 60 s: 96 -> 51 a step; 301 x 211
//     telescoping at dt 60 s: 86 -> 52) and their results move, by up to 1.8e-10 of
//     a field and 6e-9 of its rms value in a cell over 42 such grids: no further
//     from solves to rtol 1e-13 (1.3e-9 with either) than those of the short one;
//   * smoother: one red-black Gauss-Seidel sweep before (red first, from a zero
//     guess) and after (red first) the coarse correction;
//   * restriction: sum of the children's residuals (the equations are cell
//     integrals); prolongation: the parent's value (short), or linear in the
//     parent and its two nearest coarse neighbours (deep: 1/2, 1/4, 1/4, a
//     neighbour outside the grid is the parent), which takes one in eight of
//     the iterations off;
//   * coarse operators re-discretised from the fine coefficients: the
//     coefficient across a coarse face is half the sum of the fine face
//     coefficients it covers (a 2-D face of twice the length at twice the
//     distance keeps ds/dn), the row excess ap - sum(a) (storage term and the
//     folded open-boundary coefficients) is summed over the children.
// Large levels take two launches each (down: sweep + restriction; up:
// correction + sweep) over LDS tiles; from the first level that fits one
// workgroup (MgTail) the rest of the cycle is a single launch.
// The hierarchy is FP32 throughout; the Krylov vectors, the SpMV and the
// stopping test stay FP64, so the converged solution does not depend on the
// preconditioner's precision.  z is FP32 and the operator is applied to the
// same z that updates x, so the recurrence stays consistent.
//
// Layout: level l has its own ghost ring (pitch nx_l+2), the four directed
// coefficients of a cell side by side (x = N, y = E, z = S, w = W), zero
// toward a neighbour outside the grid and on the ghost ring; dinv = 1/ap
// (zero on the ghost ring and on rows without a diagonal), and zo is zero on
// the ghost ring.  The down sweep leaves the black cells' z only (the red
// ones are replaced by the up sweep before they are read), packed in rows of
// nbx: black cell (i, j) at j nbx + i/2.
#pragma once
#include "common.h"

namespace cms {

constexpr int MG_MAX_LEVELS = 16;
constexpr int MG_SHORT_LEVELS = 4;         // at least
constexpr int MG_SHORT_SWEEPS = 6;         // on the coarsest level
constexpr double MG_SHORT_RATIO = 8.0;
constexpr int MG_DEEP_SWEEPS = 4;
constexpr double MG_DEEP_RATIO = 1.0;

struct MgLevel {
    int nx, ny, nxp, nbx;       // cells, pitch, 2x2 blocks a row
    float4 *a;                  // directed off-diagonal coefficients N, E, S, W
    float *dinv;                // 1/ap
    float *ap;                  // ap (level 0 only: the FP32 operator of the inner solve)
    float *e;                   // row excess ap - sum(a), summed when coarsening
    float *zb;                  // black cells' z after the down sweep, packed
    float *zo, *b;              // cycle output z, right-hand side (zo of level 0 is the caller's
                                // M^-1 x and level 0 takes its b from the caller)
    float w0, w1;               // prolongation weights of the parent and of its neighbours
    __device__ __forceinline__ int idx(int i, int j) const { return (j + 1) * nxp + (i + 1); }
    __device__ __forceinline__ int n() const { return nx * ny; }
};

// The levels of the cycle that run in one workgroup (k_mg_tail): their z and,
// below the first, right-hand sides in LDS.
constexpr int MG_TAIL_NT = 1024;      // threads, and so 2x2 blocks of its first level, at most
constexpr int MG_TAIL_LEVELS = 14;
constexpr unsigned MG_TAIL_LDS = 160 * 1024 - 256;
struct TailLev {
    int nx, ny, nxp, nbx, nblk, npad;
    int oz, ob, oa, od;               // offsets in LDS (floats): z, b, coefficients, dinv
    const float4 *a;
    const float *dinv;
};
struct MgTail {
    int n;                            // levels
    int lds1;                         // first level with its coefficients in LDS (1 or 2)
    int deep;                         // first level run by one wave (>= lds1; n: none)
    int nlds;                         // padded cells of the levels from lds1 on: their coefficients
    const float4 *ga;                 // and dinv, level after level
    const float *gd;
    int sweeps;                       // on the coarsest level
    float w0, w1;                     // prolongation weights
    int zero0, zero1;                 // LDS range cleared at the start (the z and b arrays)
    unsigned lds;                     // bytes
    TailLev L[MG_TAIL_LEVELS];
};

struct Mg {
    int nlev;
    int lt;                           // first level of the tail
    int sweeps;                       // on the coarsest level
    float w0, w1;                     // prolongation weights
    MgLevel L[MG_MAX_LEVELS];
    MgTail tail;
};

}  // namespace cms
