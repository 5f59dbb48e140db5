// mg_kernels.hip -- the V(1,1) cycle of mg.h.
//
// Per level above the tail, one cycle is two launches over LDS tiles:
//   k_mg_down  red-black sweep from z = 0 (red z = b/ap, black
//              z = (b + sum a_k b_nb/ap_nb)/ap) and the coarse right-hand
//              side: the sum over the red children of their residual, which
//              after that sweep is sum a_k z_nb exactly (red z = b/ap cancels
//              b - ap z) and zero on black children
//   (coarser levels, the last of them in k_mg_tail)
//   k_mg_up    red cells: z = (b + sum a_k w_nb)/ap with w = z + P zc on the
//              black cells -- the coarse correction of the red cell itself is
//              replaced by this update, so only the black cells' is needed;
//              then black cells: z = (b + sum a_k z_nb)/ap with the new red
//              values
// The down sweep writes the black z and reads only b; the up sweep reads
// those and the coarse zo and writes zo, so no launch reads values it also
// writes.
#include "mg.h"
#include "krylov.h"

namespace cms {

__device__ __forceinline__ bool mg_thread(const MgLevel &L, int &i, int &j, int &c) {
    const int t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (t >= L.nx * L.ny) return false;
    j = t / L.nx;
    i = t - j * L.nx;
    c = L.idx(i, j);
    return true;
}

// Level 0 from the FP64 pressure-correction system (directed coefficients on
// the padded grid, ap from the solve prologue).
__global__ void __launch_bounds__(BLOCK) k_mg_setup0(Geo g, const double *aN, const double *aE, const double *aS,
                                                     const double *aW, const double *ap, MgLevel L) {
    int i, j, c;
    if (!mg_thread(L, i, j, c)) return;
    const double n_ = j < g.ny - 1 ? aN[c] : 0.0, e_ = i < g.nx - 1 ? aE[c] : 0.0;
    const double s_ = j > 0 ? aS[c] : 0.0, w_ = i > 0 ? aW[c] : 0.0;
    const double d = ap[c];
    L.a[c] = make_float4((float)n_, (float)e_, (float)s_, (float)w_);
    L.dinv[c] = d > 0.0 ? (float)(1.0 / d) : 0.0f;
    L.ap[c] = (float)d;
    L.e[c] = (float)fmax(d - (((n_ + e_) + s_) + w_), 0.0);
}

// Coarse cell (I, J) of level C from its fine level f (children (2I+a, 2J+b),
// a,b in {0,1}).
__device__ __forceinline__ void mg_coarsen_cell(const MgLevel &f, const MgLevel &C, int I, int J) {
    const int i0 = 2 * I, j0 = 2 * J;
    const bool hi = i0 + 1 < f.nx, hj = j0 + 1 < f.ny;
    const int i1 = hi ? i0 + 1 : i0, j1 = hj ? j0 + 1 : j0;
    const int c00 = f.idx(i0, j0), c10 = f.idx(i1, j0), c01 = f.idx(i0, j1), c11 = f.idx(i1, j1);
    const float4 a00 = f.a[c00], a10 = f.a[c10], a01 = f.a[c01], a11 = f.a[c11];
    float e = f.e[c00];
    if (hi) e += f.e[c10];
    if (hj) e += f.e[c01];
    if (hi && hj) e += f.e[c11];
    const float aE = 0.5f * (a10.y + (hj ? a11.y : 0.0f));
    const float aW = 0.5f * (a00.w + (hj ? a01.w : 0.0f));
    const float aN = 0.5f * (a01.x + (hi ? a11.x : 0.0f));
    const float aS = 0.5f * (a00.z + (hi ? a10.z : 0.0f));
    const float ap = e + ((aN + aE) + (aS + aW));
    const int c = C.idx(I, J);
    C.a[c] = make_float4(aN, aE, aS, aW);
    C.e[c] = e;
    C.dinv[c] = ap > 0.0f ? 1.0f / ap : 0.0f;
}
__global__ void __launch_bounds__(BLOCK) k_mg_coarsen(MgLevel f, MgLevel C) {
    int I, J, c;
    if (!mg_thread(C, I, J, c)) return;
    mg_coarsen_cell(f, C, I, J);
}
// Levels l0 .. nlev-1 in turn in one workgroup (each from the one above it).
__global__ void __launch_bounds__(MG_TAIL_NT) k_mg_coarsen_tail(Mg M, int l0) {
    for (int l = l0; l < M.nlev; l++) {
        const MgLevel &C = M.L[l];
        for (int t = threadIdx.x; t < C.nx * C.ny; t += MG_TAIL_NT) {
            const int J = t / C.nx, I = t - J * C.nx;
            mg_coarsen_cell(M.L[l - 1], C, I, J);
        }
        __syncthreads();
    }
}

// sum a_k z_k over the neighbours N, E, S, W
__device__ __forceinline__ float mg_sum(const float4 &a, float zN, float zE, float zS, float zW) {
    return (a.x * zN + a.y * zE) + (a.z * zS + a.w * zW);
}
// Black z of the sweep from zero: (b + sum a_k q_nb)/ap = q + (sum a_k q_nb)/ap,
// q = b/ap (red z).
__device__ __forceinline__ float mg_black(const float4 &a, float qN, float qE, float qS, float qW, float qc, float d) {
    const float s = mg_sum(a, qN, qE, qS, qW);
    return qc + s * d;
}
// z of the sweep after the coarse correction: (b + sum a_k z_nb)/ap.
__device__ __forceinline__ float mg_relax(const float4 &a, float zN, float zE, float zS, float zW, float b, float d) {
    const float s = mg_sum(a, zN, zE, zS, zW);
    return (b + s) * d;
}
// Prolongation: the parent's value and those of the coarse neighbours on the
// child's side in x and in y.
__device__ __forceinline__ float mg_lin(float w0, float w1, float zc, float zx, float zy) {
    return w0 * zc + w1 * (zx + zy);
}

// --- one level over LDS tiles ---------------------------------------------------
// A workgroup owns a tile of TX x TY fine cells; each thread owns NB 2x2
// blocks of it (the children of NB coarse cells), whose coefficients it loads
// once into registers and keeps for both phases of the sweep.  Neighbour
// values come from LDS over the tile and a halo; the halo cells that an owned
// cell reads are recomputed by the same expressions as in the neighbouring
// tile, so they are bitwise the values stored there and the result does not
// depend on the tile shape.  Every global load of the kernel is issued before
// the first wait: on small levels the time is that one round trip, not the
// bytes.
template <int TX, int TY, int NT>
struct MTile {
    static constexpr int NB = TX * TY / 4 / NT;                                // blocks per thread
    static constexpr int SX = TX + 4, SY = TY + 4;                            // staged cells (two-cell halo)
    static constexpr int NS = (SX * SY + NT - 1) / NT;                        // staged per thread (down)
    static constexpr int HX = SX / 2, NH = (HX * SY + NT - 1) / NT;           // staged black cells (up)
    static constexpr int NR = (TX + TY + NT - 1) / NT;                        // halo cells per thread
    // the stop flag is tested first on the large tiles (a launch after the stop
    // must not stream a large level), after the loads are issued on the others
    static constexpr bool EARLY = TX * TY >= 1024;
    static_assert(NB * NT * 4 == TX * TY && TX % 2 == 0 && TY % 2 == 0, "whole blocks per thread");
};

__device__ __forceinline__ bool mg_inside(const MgLevel &L, int i, int j) {
    return i >= 0 && j >= 0 && i < L.nx && j < L.ny;
}
// Padded index of cell (i, j), or 0 -- a corner of the ring, where every array
// of a level and every Krylov vector holds 0 -- outside the grid: the loads
// of a tile and its halo then need no branches, which would each wait for
// their own load.
__device__ __forceinline__ int mg_at(const MgLevel &L, int i, int j) { return mg_inside(L, i, j) ? L.idx(i, j) : 0; }
// Origin of this workgroup's tile.  Tiles are numbered row-major and dealt
// to the XCDs in contiguous runs (xcd_block), so a tile and the neighbours
// whose halo lines it shares mostly run on one XCD and meet in its L2; the
// hardware's own round-robin would put horizontal neighbours on different
// XCDs, each fetching the shared lines from HBM.
template <int TX, int TY>
__device__ __forceinline__ void mg_tile_origin(int &X0, int &Y0) {
    const int nt = (int)(gridDim.x * gridDim.y);
    const int t = xcd_block((int)(blockIdx.y * gridDim.x + blockIdx.x), nt);
    const int ty = t / (int)gridDim.x, tx = t - ty * (int)gridDim.x;
    X0 = tx * TX;
    Y0 = ty * TY;
}
// The halo cells that owned cells of the other colour read: for colour 1 (the
// black cells beside the red ones of the tile's edge) at r < TX/2 south of
// the even columns, then north of the odd ones, west of the even rows, east of
// the odd ones; for colour 0 (red) the other half.
template <int TX, int TY>
__device__ __forceinline__ void mg_halo(int r, int colour, int &fx, int &fy) {
    const int s = colour ^ 1;
    if (r < TX / 2) { fx = 2 * r + s; fy = -1; }
    else if (r < TX) { fx = 2 * (r - TX / 2) + (s ^ 1); fy = TY; }
    else if (r < TX + TY / 2) { fx = -1; fy = 2 * (r - TX) + s; }
    else { fx = TX; fy = 2 * (r - TX - TY / 2) + (s ^ 1); }
}

// Down: pre-smoothing sweep of level f (z of its black cells) and coarse b =
// the sum over the red children of sum a_k z_nb (their residual).
template <int TX, int TY, int NT, class TB>
__global__ void __launch_bounds__(NT) k_mg_down(MgLevel f, const TB *b, MgLevel C, const KryScal *sc) {
    using T = MTile<TX, TY, NT>;
    __shared__ float q[T::SY][T::SX];     // b/ap, then the black cells' z in place
    const bool done = sc->done;
    if (T::EARLY && done) return;
    int X0, Y0;
    mg_tile_origin<TX, TY>(X0, Y0);
    float4 a[T::NB][4], ha[T::NR];
    float dk[T::NB][2], hd[T::NR], sd[T::NS];
    TB sb[T::NS];
#pragma unroll
    for (int k = 0; k < T::NS; k++) {
        const int t = (int)threadIdx.x + k * NT, ly = t / T::SX, lx = t - ly * T::SX;
        const int c = ly < T::SY ? mg_at(f, X0 - 2 + lx, Y0 - 2 + ly) : 0;
        sb[k] = b[c];
        sd[k] = f.dinv[c];
    }
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, i0 = X0 + 2 * (u % (TX / 2)), j0 = Y0 + 2 * (u / (TX / 2));
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int c = mg_at(f, i0 + (s & 1), j0 + (s >> 1));
            a[k][s] = f.a[c];
            if (s == 1 || s == 2) dk[k][s - 1] = f.dinv[c];
        }
    }
#pragma unroll
    for (int k = 0; k < T::NR; k++) {
        const int r = (int)threadIdx.x + k * NT;
        int fx, fy;
        mg_halo<TX, TY>(r, 1, fx, fy);
        const int c = r < TX + TY ? mg_at(f, X0 + fx, Y0 + fy) : 0;
        ha[k] = f.a[c];
        hd[k] = f.dinv[c];
    }
    if (done) return;                     // tested after the loads are issued: its own load overlaps theirs
#pragma unroll
    for (int k = 0; k < T::NS; k++) {
        const int t = (int)threadIdx.x + k * NT, ly = t / T::SX, lx = t - ly * T::SX;
        if (ly < T::SY) q[ly][lx] = (float)sb[k] * sd[k];
    }
    __syncthreads();
    auto black = [&](const float4 &ak, float d, int lx, int ly) {
        return mg_black(ak, q[ly + 1][lx], q[ly][lx + 1], q[ly - 1][lx], q[ly][lx - 1], q[ly][lx], d);
    };
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, fx = 2 * (u % (TX / 2)), fy = 2 * (u / (TX / 2));
        const float z1 = black(a[k][1], dk[k][0], fx + 3, fy + 2), z2 = black(a[k][2], dk[k][1], fx + 2, fy + 3);
        q[fy + 2][fx + 3] = z1;
        q[fy + 3][fx + 2] = z2;
        const int i0 = X0 + fx, j0 = Y0 + fy, I = i0 >> 1;
        if (i0 + 1 < f.nx && j0 < f.ny) f.zb[(size_t)j0 * f.nbx + I] = z1;
        if (i0 < f.nx && j0 + 1 < f.ny) f.zb[(size_t)(j0 + 1) * f.nbx + I] = z2;
    }
#pragma unroll
    for (int k = 0; k < T::NR; k++) {
        const int r = (int)threadIdx.x + k * NT;
        int fx, fy;
        mg_halo<TX, TY>(r, 1, fx, fy);
        if (r < TX + TY) q[fy + 2][fx + 2] = black(ha[k], hd[k], fx + 2, fy + 2);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, fx = 2 * (u % (TX / 2)), fy = 2 * (u / (TX / 2));
        const int I = (X0 + fx) >> 1, J = (Y0 + fy) >> 1, x = fx + 2, y = fy + 2;
        if (I >= C.nx || J >= C.ny) continue;
        // children (0,0) and (1,1), red; coefficients are zero outside the grid
        const float r = mg_sum(a[k][0], q[y + 1][x], q[y][x + 1], q[y - 1][x], q[y][x - 1]) +
                        mg_sum(a[k][3], q[y + 2][x + 1], q[y + 1][x + 2], q[y][x + 1], q[y + 1][x]);
        C.b[C.idx(I, J)] = r;
    }
}

// Up: coarse correction and post-smoothing sweep (red, then black) of level
// L into L.zo.  w = z + P zc of the black cells over the tile + 2 and the new
// red z over the tile + 1 in LDS.
template <int TX, int TY, int NT, class TB>
__global__ void __launch_bounds__(NT) k_mg_up(MgLevel L, const TB *b, MgLevel C, const KryScal *sc) {
    using T = MTile<TX, TY, NT>;
    __shared__ float w[T::SY][T::SX];     // black cells: w; red cells: the new z
    const bool done = sc->done;
    if (T::EARLY && done) return;
    int X0, Y0;
    mg_tile_origin<TX, TY>(X0, Y0);
    float4 a[T::NB][4], ha[T::NR];
    float dd[T::NB][4], hd[T::NR], sz[T::NH], sc0[T::NH], scx[T::NH], scy[T::NH];
    TB bb[T::NB][4], hb[T::NR];
    const bool lin = L.w1 != 0.0f;        // (plain injection reads the parent alone)
    // staged black cells: row ly holds i = X0 - 2 + 2 m + (1 - (ly & 1)) (X0, Y0 even)
#pragma unroll
    for (int k = 0; k < T::NH; k++) {
        const int t = (int)threadIdx.x + k * NT, ly = t / T::HX, m = t - ly * T::HX;
        const int i = min(max(X0 - 2 + 2 * m + 1 - (ly & 1), 0), L.nx - 1), j = min(max(Y0 - 2 + ly, 0), L.ny - 1);
        const int I = i >> 1, J = j >> 1;
        const int Ix = !lin ? I : (i & 1) ? min(I + 1, C.nx - 1) : max(I - 1, 0);
        const int Jy = !lin ? J : (j & 1) ? min(J + 1, C.ny - 1) : max(J - 1, 0);
        sz[k] = L.zb[(size_t)j * L.nbx + I];
        sc0[k] = C.zo[C.idx(I, J)];
        scx[k] = C.zo[C.idx(Ix, J)];
        scy[k] = C.zo[C.idx(I, Jy)];
    }
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, i0 = X0 + 2 * (u % (TX / 2)), j0 = Y0 + 2 * (u / (TX / 2));
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int c = mg_at(L, i0 + (s & 1), j0 + (s >> 1));
            a[k][s] = L.a[c];
            bb[k][s] = b[c];
            dd[k][s] = L.dinv[c];
        }
    }
#pragma unroll
    for (int k = 0; k < T::NR; k++) {
        const int r = (int)threadIdx.x + k * NT;
        int fx, fy;
        mg_halo<TX, TY>(r, 0, fx, fy);
        const int c = r < TX + TY ? mg_at(L, X0 + fx, Y0 + fy) : 0;
        ha[k] = L.a[c];
        hb[k] = b[c];
        hd[k] = L.dinv[c];
    }
    if (done) return;                     // tested after the loads are issued: its own load overlaps theirs
#pragma unroll
    for (int k = 0; k < T::NH; k++) {
        const int t = (int)threadIdx.x + k * NT, ly = t / T::HX, m = t - ly * T::HX;
        const int lx = 2 * m + 1 - (ly & 1);
        const bool in = mg_inside(L, X0 - 2 + lx, Y0 - 2 + ly);
        if (ly < T::SY) w[ly][lx] = in ? sz[k] + mg_lin(L.w0, L.w1, sc0[k], scx[k], scy[k]) : 0.0f;
    }
    __syncthreads();
    auto relax = [&](const float4 &ak, TB bk, float d, int lx, int ly) {
        return mg_relax(ak, w[ly + 1][lx], w[ly][lx + 1], w[ly - 1][lx], w[ly][lx - 1], (float)bk, d);
    };
    float z0[T::NB], z3[T::NB];
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, fx = 2 * (u % (TX / 2)), fy = 2 * (u / (TX / 2));
        z0[k] = relax(a[k][0], bb[k][0], dd[k][0], fx + 2, fy + 2);
        z3[k] = relax(a[k][3], bb[k][3], dd[k][3], fx + 3, fy + 3);
        w[fy + 2][fx + 2] = z0[k];
        w[fy + 3][fx + 3] = z3[k];
    }
#pragma unroll
    for (int k = 0; k < T::NR; k++) {
        const int r = (int)threadIdx.x + k * NT;
        int fx, fy;
        mg_halo<TX, TY>(r, 0, fx, fy);
        if (r < TX + TY) w[fy + 2][fx + 2] = relax(ha[k], hb[k], hd[k], fx + 2, fy + 2);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < T::NB; k++) {
        const int u = (int)threadIdx.x + k * NT, fx = 2 * (u % (TX / 2)), fy = 2 * (u / (TX / 2));
        const int i0 = X0 + fx, j0 = Y0 + fy;
        if (i0 >= L.nx || j0 >= L.ny) continue;
        const bool hi = i0 + 1 < L.nx, hj = j0 + 1 < L.ny;
        const float z1 = relax(a[k][1], bb[k][1], dd[k][1], fx + 3, fy + 2);
        const float z2 = relax(a[k][2], bb[k][2], dd[k][2], fx + 2, fy + 3);
        const int c = L.idx(i0, j0);
        L.zo[c] = z0[k];
        if (hi) L.zo[c + 1] = z1;
        if (hj) L.zo[c + L.nxp] = z2;
        if (hi && hj) L.zo[c + L.nxp + 1] = z3[k];
    }
}

// --- the levels that fit one workgroup --------------------------------------------
// One launch for the rest of the cycle.  A level that small costs two launches
// of 4-5 us whatever its size, each a round trip to memory; here its exchanges
// are LDS phases.  A thread owns a 2x2 block of each level and keeps its z in registers: of a cell's four
// neighbours two are in its block, so a phase reads four values from LDS and
// writes two.  The first level's coefficients stay in registers from one load
// at the start, the second's too while it has more than one wave of blocks;
// the deeper ones' (side by side in memory) are copied to LDS then.  Levels of at most 64 blocks run in
// the first wave alone, whose LDS accesses are ordered without a barrier (a
// barrier of 16 waves made those phases three times as long).  From 63 x 63
// cells down to 16 x 16: 7.5 us; from 50 x 25 to 4 x 2: 9 us, against 26 us for
// two launches a level.  Two blocks a thread (levels of up to 8192 cells) took
// 13-15 us, more than the two tile launches they replace (6.8 us).
struct MgBlk {
    float4 a[4];                    // children (0,0) red, (1,0), (0,1) black, (1,1) red
    float d[4], b[4], z[4];
    int c;                          // padded index of (0,0); -1: no block
    int I, J;                       // the block: its parent's cell on the next level
};
__device__ __forceinline__ void mg_blk_at(MgBlk &B, const TailLev &V, int blk) {
#pragma unroll
    for (int s = 0; s < 4; s++) { B.a[s] = make_float4(0.f, 0.f, 0.f, 0.f); B.d[s] = B.b[s] = B.z[s] = 0.0f; }
    B.J = blk / V.nbx;
    B.I = blk - B.J * V.nbx;
    B.c = blk < V.nblk ? (2 * B.J + 1) * V.nxp + (2 * B.I + 1) : -1;
}
// Coefficients of a block; A and D: the level's arrays (global memory or
// LDS).  The ring is zero in both, so children outside the grid get zeros.
__device__ __forceinline__ void mg_blk_coef(MgBlk &B, const TailLev &V, const float4 *A, const float *D) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int c = B.c < 0 ? 0 : B.c + (s & 1) + (s >> 1) * V.nxp;     // 0: a corner of the ring
        B.a[s] = A[c];
        B.d[s] = D[c];
    }
}
__device__ __forceinline__ void mg_blk_rhs(MgBlk &B, const TailLev &V, const float *b) {
    if (B.c < 0) return;
#pragma unroll
    for (int s = 0; s < 4; s++) B.b[s] = b[B.c + (s & 1) + (s >> 1) * V.nxp];
}
__device__ __forceinline__ void mg_blk_z(MgBlk &B, const TailLev &V, const float *z) {
    if (B.c < 0) return;
    B.z[1] = z[B.c + 1];
    B.z[2] = z[B.c + V.nxp];
}
// Down sweep of a block: q = b/ap; then the black z; then the red residuals.
__device__ __forceinline__ void mg_blk_q(MgBlk &B, const TailLev &V, float *z) {
    if (B.c < 0) return;
#pragma unroll
    for (int s = 0; s < 4; s++) B.z[s] = B.b[s] * B.d[s];
    z[B.c] = B.z[0];
    z[B.c + V.nxp + 1] = B.z[3];
}
// sum a_k z_k of the black children (1,0) and (0,1), of the red ones (0,0) and (1,1)
__device__ __forceinline__ float mg_blk_sum1(const MgBlk &B, const TailLev &V, const float *z) {
    return mg_sum(B.a[1], B.z[3], z[B.c + 2], z[B.c + 1 - V.nxp], B.z[0]);
}
__device__ __forceinline__ float mg_blk_sum2(const MgBlk &B, const TailLev &V, const float *z) {
    return mg_sum(B.a[2], z[B.c + 2 * V.nxp], B.z[3], B.z[0], z[B.c + V.nxp - 1]);
}
__device__ __forceinline__ float mg_blk_sum0(const MgBlk &B, const TailLev &V, const float *z) {
    return mg_sum(B.a[0], B.z[2], B.z[1], z[B.c - V.nxp], z[B.c - 1]);
}
__device__ __forceinline__ float mg_blk_sum3(const MgBlk &B, const TailLev &V, const float *z) {
    return mg_sum(B.a[3], z[B.c + 2 * V.nxp + 1], z[B.c + V.nxp + 2], B.z[1], B.z[2]);
}
__device__ __forceinline__ void mg_blk_black0(MgBlk &B, const TailLev &V, float *z) {
    if (B.c < 0) return;
    const float s1 = mg_blk_sum1(B, V, z), s2 = mg_blk_sum2(B, V, z);
    z[B.c + 1] = B.z[1] = B.z[1] + s1 * B.d[1];
    z[B.c + V.nxp] = B.z[2] = B.z[2] + s2 * B.d[2];
}
__device__ __forceinline__ void mg_blk_restrict(const MgBlk &B, const TailLev &V, const TailLev &W, const float *z,
                                                float *bc) {
    if (B.c < 0) return;
    bc[(B.J + 1) * W.nxp + B.I + 1] = mg_blk_sum0(B, V, z) + mg_blk_sum3(B, V, z);
}
// Up sweep: the black cells' coarse correction; red and black relaxation.
__device__ __forceinline__ void mg_blk_prolong(MgBlk &B, const TailLev &V, const TailLev &W, float *z,
                                               const float *zc, float w0, float w1) {
    if (B.c < 0) return;
    const int C = (B.J + 1) * W.nxp + B.I + 1;
    const float zm = zc[C];
    const float zE = zc[B.I + 1 < W.nx ? C + 1 : C], zW = zc[B.I > 0 ? C - 1 : C];
    const float zN = zc[B.J + 1 < W.ny ? C + W.nxp : C], zS = zc[B.J > 0 ? C - W.nxp : C];
    if (2 * B.I + 1 < V.nx) z[B.c + 1] = B.z[1] = B.z[1] + mg_lin(w0, w1, zm, zE, zS);
    if (2 * B.J + 1 < V.ny) z[B.c + V.nxp] = B.z[2] = B.z[2] + mg_lin(w0, w1, zm, zW, zN);
}
__device__ __forceinline__ void mg_blk_red(MgBlk &B, const TailLev &V, float *z) {
    if (B.c < 0) return;
    const float s0 = mg_blk_sum0(B, V, z), s3 = mg_blk_sum3(B, V, z);
    z[B.c] = B.z[0] = (B.b[0] + s0) * B.d[0];
    z[B.c + V.nxp + 1] = B.z[3] = (B.b[3] + s3) * B.d[3];
}
__device__ __forceinline__ void mg_blk_black(MgBlk &B, const TailLev &V, float *z) {
    if (B.c < 0) return;
    const float s1 = mg_blk_sum1(B, V, z), s2 = mg_blk_sum2(B, V, z);
    z[B.c + 1] = B.z[1] = (B.b[1] + s1) * B.d[1];
    z[B.c + V.nxp] = B.z[2] = (B.b[2] + s2) * B.d[2];
}
// Orders the LDS accesses of one wave's phases.
__device__ __forceinline__ void mg_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The down sweep of a level, the up sweep, and a relaxation sweep; sync
// separates the phases.
template <class Sync>
__device__ __forceinline__ void mg_tail_down(MgBlk &B, const TailLev &V, const TailLev &W, float *S, Sync sync) {
    mg_blk_q(B, V, S + V.oz);
    sync();
    mg_blk_black0(B, V, S + V.oz);
    sync();
    mg_blk_restrict(B, V, W, S + V.oz, S + W.ob);
    sync();
}
template <class Sync>
__device__ __forceinline__ void mg_tail_sweep(MgBlk &B, const TailLev &V, float *S, Sync sync) {
    mg_blk_red(B, V, S + V.oz);
    sync();
    mg_blk_black(B, V, S + V.oz);
    sync();
}
template <class Sync>
__device__ __forceinline__ void mg_tail_up(MgBlk &B, const MgTail &T, int l, float *S, Sync sync) {
    const TailLev &V = T.L[l], &W = T.L[l + 1];
    mg_blk_prolong(B, V, W, S + V.oz, S + W.oz, T.w0, T.w1);
    sync();
    mg_tail_sweep(B, V, S, sync);
}
// Block t of a level whose coefficients are in LDS (its z of the black cells
// too when going up).
__device__ __forceinline__ void mg_tail_load(MgBlk &B, const TailLev &V, const float *S, int t, bool up) {
    mg_blk_at(B, V, t);
    mg_blk_coef(B, V, reinterpret_cast<const float4 *>(S + V.oa), S + V.od);
    mg_blk_rhs(B, V, S + V.ob);
    if (up) mg_blk_z(B, V, S + V.oz);
}

template <int NT, class TB>
__global__ void __launch_bounds__(NT) k_mg_tail(MgTail T, const TB *b, float *zo, const KryScal *sc) {
    const bool done = sc->done;
    extern __shared__ float4 lds4[];
    float *S = reinterpret_cast<float *>(lds4);
    const int t = threadIdx.x;
    const TailLev &V0 = T.L[0], &V1 = T.L[1];
    MgBlk top, sec, cur;
    TB tb[4];
    mg_blk_at(top, V0, t);
    mg_blk_coef(top, V0, V0.a, V0.dinv);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const bool in = top.c >= 0 && 2 * top.I + (s & 1) < V0.nx && 2 * top.J + (s >> 1) < V0.ny;
        tb[s] = b[in ? top.c + (s & 1) + (s >> 1) * V0.nxp : 0];
    }
    const bool reg1 = T.lds1 == 2;        // the second level's coefficients in registers
    if (reg1) {
        mg_blk_at(sec, V1, t);
        mg_blk_coef(sec, V1, V1.a, V1.dinv);
    }
    float4 la[2];
    float ld[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int q = t + k * NT < T.nlds ? t + k * NT : 0;
        la[k] = T.ga[q];
        ld[k] = T.gd[q];
    }
    if (done) return;                     // tested after the loads are issued: its own load overlaps theirs
#pragma unroll
    for (int s = 0; s < 4; s++) top.b[s] = (float)tb[s];
    float4 *A = reinterpret_cast<float4 *>(S + T.L[T.lds1].oa);
    float *D = S + T.L[T.lds1].od;
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (t + k * NT < T.nlds) {
            A[t + k * NT] = la[k];
            D[t + k * NT] = ld[k];
        }
    for (int q = t + 2 * NT; q < T.nlds; q += NT) {
        A[q] = T.ga[q];
        D[q] = T.gd[q];
    }
    for (int q = T.zero0 + t; q < T.zero1; q += NT) S[q] = 0.0f;
    __syncthreads();
    const auto block_sync = [] { __syncthreads(); };
    const auto wave_sync = [] { mg_wave_sync(); };
    const int last = T.n - 1;
    if (last > 0) mg_tail_down(top, V0, V1, S, block_sync);
    if (reg1) {
        mg_blk_rhs(sec, V1, S + V1.ob);
        if (last > 1) mg_tail_down(sec, V1, T.L[2], S, block_sync);
    }
    for (int l = T.lds1; l < T.deep && l < last; l++) {
        mg_tail_load(cur, T.L[l], S, t, false);
        mg_tail_down(cur, T.L[l], T.L[l + 1], S, block_sync);
    }
    if (T.deep <= last) {
        // T.L[deep] .. the last level in the first wave
        if (t < 64) {
            for (int l = T.deep; l < last; l++) {
                mg_tail_load(cur, T.L[l], S, t, false);
                mg_tail_down(cur, T.L[l], T.L[l + 1], S, wave_sync);
            }
            mg_tail_load(cur, T.L[last], S, t, false);
            for (int sw = 0; sw < T.sweeps; sw++) mg_tail_sweep(cur, T.L[last], S, wave_sync);
            for (int l = last - 1; l >= T.deep; l--) {
                mg_tail_load(cur, T.L[l], S, t, true);
                mg_tail_up(cur, T, l, S, wave_sync);
            }
        }
        __syncthreads();
    } else if (last >= T.lds1) {
        mg_tail_load(cur, T.L[last], S, t, false);
        for (int sw = 0; sw < T.sweeps; sw++) mg_tail_sweep(cur, T.L[last], S, block_sync);
    } else if (reg1 && last == 1) {
        for (int sw = 0; sw < T.sweeps; sw++) mg_tail_sweep(sec, V1, S, block_sync);
    } else {
        for (int sw = 0; sw < T.sweeps; sw++) mg_tail_sweep(top, V0, S, block_sync);
    }
    for (int l = min(T.deep, last) - 1; l >= T.lds1; l--) {
        mg_tail_load(cur, T.L[l], S, t, true);
        mg_tail_up(cur, T, l, S, block_sync);
    }
    if (reg1 && last > 1) mg_tail_up(sec, T, 1, S, block_sync);
    if (last > 0) mg_tail_up(top, T, 0, S, block_sync);
    if (top.c < 0) return;
    const bool hi = 2 * top.I + 1 < V0.nx, hj = 2 * top.J + 1 < V0.ny;
    zo[top.c] = top.z[0];
    if (hi) zo[top.c + 1] = top.z[1];
    if (hj) zo[top.c + V0.nxp] = top.z[2];
    if (hi && hj) zo[top.c + V0.nxp + 1] = top.z[3];
}

}  // namespace cms
