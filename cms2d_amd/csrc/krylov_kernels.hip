// krylov_kernels.hip -- solve() prologue and Jacobi-preconditioned BiCGStab
// sweeps (restating solvers.f90:205-304 and pbicgstab.f90:21-96; krylov.h
// describes the recurrence and the atomic-free reductions).
//
// Iteration `it` is five launches on the fixed grid:
//   k_bicg_p(it)     finish iteration it-1 from its r.r and r0.r partials
//                    (stop test, restart, beta); p = r + beta (p - omega v)
//   k_bicg_spmv1(it) v = A M^-1 p, partials r0.v
//   k_bicg_s(it)     alpha = rho / r0.v;  x += alpha M^-1 p;  s = r - alpha v
//   k_bicg_spmv2(it) t = A M^-1 s, partials t.s and t.t
//   k_bicg_r(it)     omega = t.s / t.t;  x += omega M^-1 s;  r = s - omega t,
//                    partials r.r and r0.r
#include "flow_state.h"

namespace cms {

#ifndef SMALL
#define SMALL F4(1.0e-15)
#endif

// The five sweeps.  On a small grid a block makes one pass and a launch lasts
// as long as its longest chain of loads, so each kernel issues the loads of its
// first cell, of the stopping flags and of the scalars before it sums the
// partials and before it tests a flag; only the stores wait for those (in
// turn, flag, partials, scalars and operands took 1.5-2 us more per launch).

// The start of iteration it (or of the solve, it == 0): which systems go on,
// their beta and omega, and whether r0 restarts; block 0 publishes the scalars.
template <int NS>
struct KryStart {
    int sdone[NS], siter[NS];
    double sthr[NS], srho[NS], sr0n[NS], salp[NS], somg[NS];
    bool act[NS];
    int rst[NS];
    double beta[NS], om[NS];
    // the scalars of system q as iteration it - 1 left them (slot pq)
    template <class Sys>
    __device__ __forceinline__ void scalars(const Sys &K, int q, int pq) {
        const KryScal &sc = K.sc[q];
        sdone[q] = sc.done; siter[q] = sc.iters[pq]; sthr[q] = sc.thr; srho[q] = sc.rho[pq];
        sr0n[q] = sc.r0n[pq]; salp[q] = sc.alpha[pq]; somg[q] = sc.omega[pq];
    }
    // tot: r.r and r0.r of each system (r.r and res.res when it == 0), n cells;
    // false: every system has stopped
    template <class Sys>
    __device__ __forceinline__ bool finish(const Sys &K, const double (&tot)[2 * NS], int it, int kmax, double rtol,
                                           double atol, int n, bool load) {
        const int pq = (it - 1) & 1, cq = it & 1;
        bool any = false;
#pragma unroll
        for (int q = 0; q < NS; q++) {
            KryScal &sc = K.sc[q];
            act[q] = false; rst[q] = 0; beta[q] = 0.0; om[q] = 1.0;
            if (load) scalars(K, q, pq);
            if (uni(sdone[q])) continue;
            const double rr = uni(tot[2 * q]), nr = uni(sqrt(rr));
            if (it == 0) {
                const double thr = fmax(rtol * nr, atol * sqrt((double)n));
                act[q] = !(nr <= thr);
                if (lead()) {
                    sc.rmom = sqrt(tot[2 * q + 1] / (double)(float)n);   // sqrt(adak/real(ncells))
                    sc.thr = thr;
                    sc.rho[0] = rr;
                    sc.r0n[0] = nr;
                    sc.iters[0] = 0;
                    sc.rnorm = nr;
                    if (!act[q]) { sc.done = 1; sc.final_iters = 0; }
                }
            } else {
                const double r0r = uni(tot[2 * q + 1]);
                const int iters = uni(siter[q]) + 1;
                const double rho_p = uni(srho[q]), r0n_p = uni(sr0n[q]), al = uni(salp[q]), omp = uni(somg[q]);
                double rho = rho_p, r0n = r0n_p;
                if (omp == 0.0 || nr <= uni(sthr[q]) || iters >= kmax) {
                    act[q] = false;
                } else if (fabs(r0r) <= 1e-12 * nr * r0n_p) {
                    rst[q] = 1; rho = rr; r0n = nr; beta[q] = 0.0; act[q] = true;
                } else {
                    beta[q] = uni((r0r / rho_p) * (al / omp)); rho = r0r; act[q] = true;
                }
                om[q] = omp;
                if (lead()) {
                    sc.rnorm = nr;
                    sc.iters[cq] = iters;
                    if (act[q]) { sc.rho[cq] = rho; sc.r0n[cq] = r0n; }
                    else { sc.done = 1; sc.final_iters = iters; }
                }
            }
            any = any || act[q];
        }
        return any;
    }
};

// Finishes iteration it-1 (or starts the solve when it == 0) and, unless
// fin_only, updates p.  Launched with fin_only on one block at the end of a
// batch so the host can read the state; the next batch repeats the same
// finish (same inputs, same result) before its first p update.
template <class Op, int NS, class T = double>
__global__ void __launch_bounds__(KBLOCK, NS == 2 ? 8 : 1)
k_bicg_p(Op A, KrySys<NS, T> K, int it, int nb, int kmax, double rtol, double atol, int fin_only) {
    auto w = A.walk();
    Idx x;
    T r[NS], p[NS], v[NS];
    auto load = [&]() {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            r[q] = K.r[q][x.c];
            p[q] = v[q] = T(0);
        }
        // the first iteration starts from p = r (p and v of an earlier solve are not read)
        if (it > 0)
#pragma unroll
            for (int q = 0; q < NS; q++) {
                p[q] = K.p[q][x.c];
                v[q] = K.v[q][x.c];
            }
    };
    // (two systems' operands and scalars together exceed the registers of eight
    // waves a SIMD: there they are loaded after the sums)
    constexpr bool PRE = NS == 1;
    bool ok = !fin_only && w.first(x);
    if (PRE && ok) load();
    const int pq = (it - 1) & 1;
    KryStart<NS> f;
    if (PRE) f.scalars(K, 0, pq);
    double tot[2 * NS];
    const double *src[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { src[2 * q] = K.red.pr[q]; src[2 * q + 1] = K.red.pr[q] + nb; }
    sum_partials<2 * NS>(src, nb, tot);
    if (!f.finish(K, tot, it, kmax, rtol, atol, A.n(), !PRE)) return;
    if (!PRE && ok) load();
    while (ok) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!f.act[q]) continue;
            if (f.rst[q]) K.r0[q][x.c] = r[q];
            K.p[q][x.c] = it == 0 ? r[q] : r[q] + (T)f.beta[q] * (p[q] - (T)f.om[q] * v[q]);
        }
        ok = w.next(x);
        if (ok) load();
    }
}

// MODE 1: v = A M^-1 p, partials r0.v.  MODE 2: t = A M^-1 s (s held in r),
// partials t.s and t.t.  PREC 1: M^-1 p and M^-1 s are the explicit zp, zs.
template <class Op, int NS, int MODE, int PREC = 0, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_spmv(Op A, KrySys<NS, T> K) {
    static_assert(PREC == 0 || NS == 1, "explicit preconditioner: one system");
    constexpr int NV = MODE == 1 ? NS : 2 * NS;
    double red[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) red[q] = 0.0;
    bool act[NS];
    bool any = false;
    auto w = A.walk();
    Idx x;
    T y[NS], m[NS];                       // A z and the vector of its product r0 or s
    const T *xv[NS], *dinv[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) {
        xv[q] = MODE == 1 ? K.p[q] : K.r[q];
        dinv[q] = K.dinv_w[q];
    }
    auto row = [&]() {
        if constexpr (PREC == 1) y[0] = A.apply_z(MODE == 1 ? K.zp : K.zs, K.ap_w[0], x);
        else A.apply_n(xv, dinv, x, y);
#pragma unroll
        for (int q = 0; q < NS; q++) m[q] = MODE == 1 ? K.r0[q][x.c] : xv[q][x.c];
    };
    int done[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) done[q] = K.sc[q].done;
    bool ok = w.first(x);
    if (ok) row();
#pragma unroll
    for (int q = 0; q < NS; q++) {
        act[q] = !uni(done[q]);
        any = any || act[q];
    }
    if (!any) return;
    while (ok) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!act[q]) continue;
            const double yd = y[q];
            if (MODE == 1) {
                K.v[q][x.c] = y[q];
                red[q] += (double)m[q] * yd;
            } else {
                K.t[q][x.c] = y[q];
                red[2 * q] += yd * (double)m[q];
                red[2 * q + 1] += yd * yd;
            }
        }
        ok = w.next(x);
        if (ok) row();
    }
    double *dst[NV];
#pragma unroll
    for (int q = 0; q < NS; q++) {
        if (MODE == 1) dst[q] = K.red.pv[q];
        else { dst[2 * q] = K.red.pt[q]; dst[2 * q + 1] = K.red.pt[q] + gridDim.x; }
    }
    put_partials<NV>(red, dst);
}

// alpha = rho / r0.v ; x += alpha M^-1 p ; s = r - alpha v (s overwrites r).
// PREC 1 defers the x update to k_bicg_r.
template <class Op, int NS, int PREC = 0, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_s(Op A, KrySys<NS, T> K, int it, int nb) {
    auto w = A.walk();
    Idx x;
    T r[NS], v[NS], p[NS], d[NS], xs[NS];
    auto load = [&](int q) {
        r[q] = K.r[q][x.c];
        v[q] = K.v[q][x.c];
        if constexpr (PREC == 0) { p[q] = K.p[q][x.c]; d[q] = K.dinv_w[q][x.c]; xs[q] = K.x[q][x.c]; }
    };
    bool ok = w.first(x);
    if (ok)
#pragma unroll
        for (int q = 0; q < NS; q++) load(q);
    const int cq = it & 1;
    struct { int done, iters; double rho; } pre[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) pre[q] = {K.sc[q].done, K.sc[q].iters[cq], K.sc[q].rho[cq]};
    double tot[NS];
    const double *src[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) src[q] = K.red.pv[q];
    sum_partials<NS>(src, nb, tot);
    bool act[NS];
    double al[NS];
    bool any = false;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        KryScal &sc = K.sc[q];
        act[q] = !uni(pre[q].done);
        al[q] = 0.0;
        if (!act[q]) continue;
        if (uni(tot[q]) == 0.0) {                       // r0.v = 0: stop before the update
            act[q] = false;
            if (lead()) { sc.done = 1; sc.final_iters = pre[q].iters; }
            continue;
        }
        al[q] = uni(pre[q].rho / tot[q]);
        if (lead()) sc.alpha[cq] = al[q];
        any = true;
    }
    if (!any) return;
    while (ok) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!act[q]) continue;
            if constexpr (PREC == 0) K.x[q][x.c] = xs[q] + al[q] * (p[q] * d[q]);
            K.r[q][x.c] = r[q] - (T)al[q] * v[q];
        }
        ok = w.next(x);
        if (ok)
#pragma unroll
            for (int q = 0; q < NS; q++)
                if (act[q]) load(q);
    }
}

// omega = t.s / t.t ; x += omega M^-1 s ; r = s - omega t ; partials r.r, r0.r
// PREC 1: x += alpha zp + omega zs.
template <class Op, int NS, int PREC = 0, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_r(Op A, KrySys<NS, T> K, int it, int nb) {
    auto w = A.walk();
    Idx x;
    T sv[NS], t[NS], d[NS], xs[NS], r0[NS];
    float zp = 0.0f, zs = 0.0f;
    auto load = [&](int q) {
        sv[q] = K.r[q][x.c];
        t[q] = K.t[q][x.c];
        xs[q] = K.x[q][x.c];
        r0[q] = K.r0[q][x.c];
        if constexpr (PREC == 1) { zp = K.zp[x.c]; zs = K.zs[x.c]; }
        else d[q] = K.dinv_w[q][x.c];
    };
    bool ok = w.first(x);
    if (ok)
#pragma unroll
        for (int q = 0; q < NS; q++) load(q);
    const int cq = it & 1;
    struct { int done; double alpha; } pre[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) pre[q] = {K.sc[q].done, K.sc[q].alpha[cq]};
    double tot[2 * NS];
    const double *src[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { src[2 * q] = K.red.pt[q]; src[2 * q + 1] = K.red.pt[q] + nb; }
    sum_partials<2 * NS>(src, nb, tot);
    bool act[NS];
    double om[NS], al[NS];
    bool any = false;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        act[q] = !uni(pre[q].done);
        const double ts = tot[2 * q], tt = tot[2 * q + 1];
        om[q] = uni(tt > 0.0 ? ts / tt : 0.0);
        al[q] = uni(pre[q].alpha);
        if (act[q] && lead()) K.sc[q].omega[cq] = om[q];
        any = any || act[q];
    }
    if (!any) return;
    double red[2 * NS];
#pragma unroll
    for (int q = 0; q < 2 * NS; q++) red[q] = 0.0;
    while (ok) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!act[q]) continue;
            if constexpr (PREC == 1) K.x[q][x.c] = xs[q] + ((T)al[q] * (T)zp + (T)om[q] * (T)zs);
            else K.x[q][x.c] = xs[q] + om[q] * (sv[q] * d[q]);
            const T r = sv[q] - (T)om[q] * t[q];
            K.r[q][x.c] = r;
            red[2 * q] += (double)r * (double)r;
            red[2 * q + 1] += (double)r0[q] * (double)r;
        }
        ok = w.next(x);
        if (ok)
#pragma unroll
            for (int q = 0; q < NS; q++)
                if (act[q]) load(q);
    }
    double *dst[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { dst[2 * q] = K.red.pr[q]; dst[2 * q + 1] = K.red.pr[q] + gridDim.x; }
    put_partials<2 * NS>(red, dst);
}

// The Jacobi iteration in three launches (systems of up to KRY_FUSED cells,
// where a launch costs more than its loads): p and s are formed where they are
// read, at a cell and at its neighbours, instead of in sweeps of their own
// (f1: k_bicg_p and v = A M^-1 p; f2: alpha and t = A M^-1 s; f3: both updates of x
// and r).  A neighbour's p needs r, p and v of the launches before, so p
// goes to the buffer that it was not read from, and v to the one that held t
// (K.p and K.p2, K.v and K.t in turn by the parity of it; t takes the place of
// the v that f1 read).  The values are those of the five sweeps.
template <int NS, class T>
struct KryBuf {
    T *pin[NS], *pout[NS], *vin[NS], *vout[NS];
    __device__ __forceinline__ KryBuf(const KrySys<NS, T> &K, int it) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            const bool o = it & 1;
            pin[q] = o ? K.p[q] : K.p2[q];
            pout[q] = o ? K.p2[q] : K.p[q];
            vin[q] = o ? K.v[q] : K.t[q];
            vout[q] = o ? K.t[q] : K.v[q];
        }
    }
};
template <class Op, int NS, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_f1(Op A, KrySys<NS, T> K, int it, int nb, int kmax, double rtol,
                                                   double atol) {
    const KryBuf<NS, T> B(K, it);
    auto w = A.walk();
    Idx x;
    bool ok = w.first(x);
    double tot[2 * NS];
    const double *src[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { src[2 * q] = K.red.pr[q]; src[2 * q + 1] = K.red.pr[q] + nb; }
    sum_partials<2 * NS>(src, nb, tot);
    KryStart<NS> f;
    if (!f.finish(K, tot, it, kmax, rtol, atol, A.n(), true)) return;
    double red[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) red[q] = 0.0;
    for (; ok; ok = w.next(x)) {
        T sum[NS];
        auto pnew = [&](int q, int c) {
            const T r = K.r[q][c];
            return it == 0 ? r : r + (T)f.beta[q] * (B.pin[q][c] - (T)f.om[q] * B.vin[q][c]);
        };
        A.template sums<NS, T>(x, [&](int q, int c) { return f.act[q] ? pnew(q, c) * K.dinv_w[q][c] : T(0); }, sum);
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!f.act[q]) continue;
            const int c = x.c;
            const T p = pnew(q, c), y = p - sum[q];
            T r0 = K.r0[q][c];
            if (f.rst[q]) K.r0[q][c] = r0 = K.r[q][c];
            B.pout[q][c] = p;
            B.vout[q][c] = y;
            red[q] += (double)r0 * (double)y;
        }
    }
    double *dst[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) dst[q] = K.red.pv[q];
    put_partials<NS>(red, dst);
}
template <class Op, int NS, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_f2(Op A, KrySys<NS, T> K, int it, int nb) {
    const KryBuf<NS, T> B(K, it);
    auto w = A.walk();
    Idx x;
    bool ok = w.first(x);
    const int cq = it & 1;
    int sdone[NS], siter[NS];
    double srho[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { sdone[q] = K.sc[q].done; siter[q] = K.sc[q].iters[cq]; srho[q] = K.sc[q].rho[cq]; }
    double tot[NS];
    const double *src[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) src[q] = K.red.pv[q];
    sum_partials<NS>(src, nb, tot);
    bool act[NS];
    double al[NS];
    bool any = false;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        act[q] = !uni(sdone[q]);
        al[q] = 0.0;
        if (!act[q]) continue;
        if (uni(tot[q]) == 0.0) {                  // r0.v = 0: stop before the update
            act[q] = false;
            if (lead()) { K.sc[q].done = 1; K.sc[q].final_iters = siter[q]; }
            continue;
        }
        al[q] = uni(srho[q] / tot[q]);
        if (lead()) K.sc[q].alpha[cq] = al[q];
        any = true;
    }
    if (!any) return;
    double red[2 * NS];
#pragma unroll
    for (int q = 0; q < 2 * NS; q++) red[q] = 0.0;
    for (; ok; ok = w.next(x)) {
        T sum[NS];
        auto snew = [&](int q, int c) { return K.r[q][c] - (T)al[q] * B.vout[q][c]; };
        A.template sums<NS, T>(x, [&](int q, int c) { return act[q] ? snew(q, c) * K.dinv_w[q][c] : T(0); }, sum);
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!act[q]) continue;
            const T s = snew(q, x.c), y = s - sum[q];
            const double yd = y;
            B.vin[q][x.c] = y;
            red[2 * q] += yd * (double)s;
            red[2 * q + 1] += yd * yd;
        }
    }
    double *dst[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { dst[2 * q] = K.red.pt[q]; dst[2 * q + 1] = K.red.pt[q] + gridDim.x; }
    put_partials<2 * NS>(red, dst);
}
template <class Op, int NS, class T = double>
__global__ void __launch_bounds__(KBLOCK) k_bicg_f3(Op A, KrySys<NS, T> K, int it, int nb) {
    const KryBuf<NS, T> B(K, it);
    auto w = A.walk();
    Idx x;
    T r[NS], v[NS], t[NS], d[NS], xs[NS], p[NS], r0[NS];
    auto load = [&](int q) {
        r[q] = K.r[q][x.c];
        v[q] = B.vout[q][x.c];
        t[q] = B.vin[q][x.c];
        d[q] = K.dinv_w[q][x.c];
        xs[q] = K.x[q][x.c];
        p[q] = B.pout[q][x.c];
        r0[q] = K.r0[q][x.c];
    };
    bool ok = w.first(x);
    constexpr bool PRE = NS == 1;         // (k_bicg_p)
    if (PRE && ok) load(0);
    const int cq = it & 1;
    int sdone[NS];
    double salp[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { sdone[q] = K.sc[q].done; salp[q] = K.sc[q].alpha[cq]; }
    double tot[2 * NS];
    const double *src[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { src[2 * q] = K.red.pt[q]; src[2 * q + 1] = K.red.pt[q] + nb; }
    sum_partials<2 * NS>(src, nb, tot);
    bool act[NS];
    double om[NS], al[NS];
    bool any = false;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        act[q] = !uni(sdone[q]);
        const double ts = tot[2 * q], tt = tot[2 * q + 1];
        om[q] = uni(tt > 0.0 ? ts / tt : 0.0);
        al[q] = uni(salp[q]);
        if (act[q] && lead()) K.sc[q].omega[cq] = om[q];
        any = any || act[q];
    }
    if (!any) return;
    double red[2 * NS];
#pragma unroll
    for (int q = 0; q < 2 * NS; q++) red[q] = 0.0;
    if (!PRE && ok)
#pragma unroll
        for (int q = 0; q < NS; q++) load(q);
    while (ok) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            if (!act[q]) continue;
            const T s = r[q] - (T)al[q] * v[q];
            const T x1 = xs[q] + al[q] * (p[q] * d[q]);
            K.x[q][x.c] = x1 + om[q] * (s * d[q]);
            const T rn = s - (T)om[q] * t[q];
            K.r[q][x.c] = rn;
            red[2 * q] += (double)rn * (double)rn;
            red[2 * q + 1] += (double)r0[q] * (double)rn;
        }
        ok = w.next(x);
        if (ok)
#pragma unroll
            for (int q = 0; q < NS; q++)
                if (act[q]) load(q);
    }
    double *dst[2 * NS];
#pragma unroll
    for (int q = 0; q < NS; q++) { dst[2 * q] = K.red.pr[q]; dst[2 * q + 1] = K.red.pr[q] + gridDim.x; }
    put_partials<2 * NS>(red, dst);
}

// Clears n 32-bit words with vector stores (used instead of a memset node).
__global__ void k_zero_words(unsigned int *p, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0u;
}

// solve() prologue on the reference's general cell list (solvers.f90:232-240)
// and the BiCGStab start, for the drop-in cms2d_solve.
// bias: the reference's small number added to the starting residual
// (pbicgstab.f90), 0 for the transposed solve of the adjoint, which must stay
// linear in its right-hand side.
__global__ void __launch_bounds__(KBLOCK) k_ell_prologue(EllOp A, const int *iwet, double *ss, const double *sp,
                                                        double *res, const double *phi, double relax,
                                                        KrySys<1> K, double bias) {
    double red[2] = {0.0, 0.0};
    const Chunk ch = block_chunk(A.ncells);
    const double rinv = 1.0 / relax, relaxm = 1.0 - relax;
    for (int c = ch.begin + threadIdx.x; c < ch.end; c += KBLOCK) {
        double asum = 0.0, anb = 0.0;
#pragma unroll
        for (int k = 0; k < ELL_MAX_FACES; k++) {
            if (k >= A.nf) break;
            const int nbc = A.c2c[A.nf * c + k];
            if (nbc < 0) continue;
            asum += A.a[A.nf * c + k];
            anb += A.a[A.nf * c + k] * phi[nbc];
        }
        double ap = (asum - sp[c]) * rinv;
        double ph = phi[c];
        double ssv = ss[c] + relaxm * ph * ap;
        ss[c] = ssv;
        double rs = iwet[c] * (anb + ssv - ap * ph) / ap;
        res[c] = rs;
        double r = anb + ssv - ap * ph + bias;
        K.dinv_w[0][c] = 1.0 / ap;
        K.r[0][c] = r; K.r0[0][c] = r;
        red[0] += r * r;
        red[1] += rs * rs;
    }
    double *const dst[2] = {K.red.pr[0], K.red.pr[0] + gridDim.x};
    put_partials<2>(red, dst);
    kry_reset(K.sc[0]);
}

}  // namespace cms

namespace cms {

// --- FP32 Krylov inside FP64 iterative refinement ----------------------------
// Outer sweep: d = inner FP32 BiCGStab solve of A d = r (FP32 matrix and
// vectors, multigrid preconditioner); x += d and r -= A d in FP64; stop when
// the FP64 ||r|| meets the FP64 solve's own threshold.

// Inner start from the FP64 residual: r = r0 = (float) r64, x = 0 (p starts from r).
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_ref_start(Op A, KrySys<1, float> Ki, const double *r64) {
    double red[2] = {0.0, 0.0};
    A.each([&](const Idx &x_) {
        const int c = x_.c;
        const float r = (float)r64[c];
        Ki.r[0][c] = r; Ki.r0[0][c] = r; Ki.x[0][c] = 0.0f;
        red[0] += (double)r * (double)r;
    });
    red[1] = red[0];
    double *const dst[2] = {Ki.red.pr[0], Ki.red.pr[0] + gridDim.x};
    put_partials<2>(red, dst);
    kry_reset(Ki.sc[0]);
}

// x += d, r -= A d (FP64 operator on the FP32 correction), partials ||r||^2.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_ref_update(Op A, KrySys<1, double> K, const float *d) {
    double red[2] = {0.0, 0.0};
    A.each([&](const Idx &x) {
        const int c = x.c;
        K.x[0][c] = K.x[0][c] + (double)d[c];
        const double r = K.r[0][c] - A.apply_z(d, K.ap_w[0], x);
        K.r[0][c] = r;
        red[0] += r * r;
    });
    double *const dst[2] = {K.red.pr[0], K.red.pr[0] + gridDim.x};
    put_partials<2>(red, dst);
}

// The u and v solves of the FP32 form (two systems, Jacobi): FP32 copies of
// the shared coefficients and of each system's diagonal.
__global__ void __launch_bounds__(KBLOCK) k_uv_to32(StencilOp A, KrySys<2, double> K, float4 *a,
                                                   KrySys<2, float> Ki) {
    A.each([&](const Idx &x) {
        const int c = x.c;
        a[c] = make_float4((float)A.aN[c], (float)A.aE[c], (float)A.aS[c], (float)A.aW[c]);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            Ki.ap_w[q][c] = (float)K.ap_w[q][c];
            Ki.dinv_w[q][c] = (float)K.dinv_w[q][c];
        }
    });
}
// Start of an inner FP32 sweep of the two systems: r = FP64 residual (0 for
// a system whose FP64 solve has stopped), x = 0.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_ref_start2(Op A, KrySys<2, float> Ki, KrySys<2, double> K) {
    double red[4] = {0.0, 0.0, 0.0, 0.0};
    bool live[2];
#pragma unroll
    for (int q = 0; q < 2; q++) live[q] = !K.sc[q].done;
    A.each([&](const Idx &x_) {
        const int c = x_.c;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const float r = live[q] ? (float)K.r[q][c] : 0.0f;
            Ki.r[q][c] = r; Ki.r0[q][c] = r; Ki.x[q][c] = 0.0f;
            red[2 * q] += (double)r * (double)r;
        }
    });
    red[1] = red[0];
    red[3] = red[2];
    double *const dst[4] = {Ki.red.pr[0], Ki.red.pr[0] + gridDim.x, Ki.red.pr[1], Ki.red.pr[1] + gridDim.x};
    put_partials<4>(red, dst);
    kry_reset(Ki.sc[0]);
    kry_reset(Ki.sc[1]);
}
// x += d, r -= A d for each running system (FP64 operator on the FP32
// correction), partials ||r||^2.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_ref_update2(Op A, KrySys<2, double> K, KrySys<2, float> Ki) {
    double red[2] = {0.0, 0.0};
    bool live[2];
#pragma unroll
    for (int q = 0; q < 2; q++) live[q] = !K.sc[q].done;
    A.each([&](const Idx &x) {
        const int c = x.c;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (!live[q]) continue;
            const float *d = Ki.x[q];
            K.x[q][c] = K.x[q][c] + (double)d[c];
            const double r = K.r[q][c] - A.apply_z(d, K.ap_w[q], x);
            K.r[q][c] = r;
            red[q] += r * r;
        }
    });
    double *const dst[2] = {K.red.pr[0], K.red.pr[1]};
    put_partials<2>(red, dst);
}
// One block: the FP64 stop tests of the two systems after a sweep.
__global__ void __launch_bounds__(KBLOCK) k_ref_check2(KrySys<2, double> K, int nb) {
    double tot[2];
    const double *src[2] = {K.red.pr[0], K.red.pr[1]};
    sum_partials<2>(src, nb, tot);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (K.sc[q].done) continue;
            const double nr = sqrt(tot[q]);
            K.sc[q].rnorm = nr;
            if (nr <= K.sc[q].thr) K.sc[q].done = 1;
        }
}

// One block: the FP64 stop test of the outer sweep.
__global__ void __launch_bounds__(KBLOCK) k_ref_check(KrySys<1, double> K, int nb) {
    double tot[1];
    const double *src[1] = {K.red.pr[0]};
    sum_partials<1>(src, nb, tot);
    if (threadIdx.x == 0) {
        const double nr = sqrt(tot[0]);
        K.sc[0].rnorm = nr;
        if (nr <= K.sc[0].thr) K.sc[0].done = 1;
    }
}

}  // namespace cms

namespace cms {

// --- GMRES(m) -----------------------------------------------------------------

// Start of a cycle (one block): beta = ||r|| from partials pr0 (pr1: res.res
// of the solve prologue on the first cycle, for rmom).
__global__ void __launch_bounds__(KBLOCK) k_gm_begin(GmSys G, const double *pr0, const double *pr1, int nb,
                                                     int first, int n, double rtol, double atol) {
    double tot[2];
    const double *src[2] = {pr0, pr1 ? pr1 : pr0};
    sum_partials<2>(src, nb, tot);
    if (threadIdx.x != 0) return;
    GmScal &s = *G.sc;
    const double beta = sqrt(tot[0]);
    if (first) {
        s.ks.thr = fmax(rtol * beta, atol * sqrt((double)n));
        s.ks.rmom = sqrt(tot[1] / (double)(float)n);
        s.iters = 0;
    }
    s.beta = beta;
    s.g[0] = beta;
    s.j = 0;
    s.cycle_end = 0;
    s.ks.rnorm = beta;
    s.ks.done = beta <= s.ks.thr ? 1 : 0;
    s.ks.final_iters = s.iters;
    s.ks_final.done = 0;
}

template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_v0(Op A, GmSys G) {
    if (G.sc->ks.done) return;
    const double bi = 1.0 / G.sc->beta;
    A.each([&](const Idx &x_) {
        const int c = x_.c;
        G.V[0][c] = G.r[c] * bi;
    });
}

// w = A z into V[j+1]; partial sums of (w, V[i]), i <= j, in slot i.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_spmv_dot(Op A, GmSys G, int j) {
    if (G.sc->ks.done) return;
    double acc[GM_M + 1];
#pragma unroll
    for (int i = 0; i <= GM_M; i++) acc[i] = 0.0;
    A.each([&](const Idx &x) {
        const double w = A.apply_z(G.z, G.ap, x);
        G.V[j + 1][x.c] = w;
#pragma unroll
        for (int i = 0; i <= GM_M; i++)
            if (i <= j) acc[i] += w * G.V[i][x.c];
    });
#pragma unroll
    for (int i = 0; i <= GM_M; i++) {
        if (i <= j) {                   // j is uniform: every thread takes the same branches
            double v[1] = {acc[i]};
            double *const dst[1] = {G.part + (size_t)i * gridDim.x};
            put_partials<1>(v, dst);
        }
    }
}

// One block: column j of H from the partials.
__global__ void __launch_bounds__(KBLOCK) k_gm_hred(GmSys G, int j, int nb) {
    if (G.sc->ks.done) return;
    for (int i = 0; i <= j; i++) {
        double tot[1];
        const double *src[1] = {G.part + (size_t)i * nb};
        sum_partials<1>(src, nb, tot);
        if (threadIdx.x == 0) G.sc->H[(GM_M + 1) * j + i] = tot[0];
    }
}

// w -= sum_i H[i,j] V[i]; partial ||w||^2 in slot GM_M + 1.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_orth(Op A, GmSys G, int j) {
    if (G.sc->ks.done) return;
    double h[GM_M + 1];
#pragma unroll
    for (int i = 0; i <= GM_M; i++) h[i] = i <= j ? G.sc->H[(GM_M + 1) * j + i] : 0.0;
    double acc[1] = {0.0};
    A.each([&](const Idx &x_) {
        const int c = x_.c;
        double w = G.V[j + 1][c];
#pragma unroll
        for (int i = 0; i <= GM_M; i++)
            if (i <= j) w -= h[i] * G.V[i][c];
        G.V[j + 1][c] = w;
        acc[0] += w * w;
    });
    double *const dst[1] = {G.part + (size_t)(GM_M + 1) * gridDim.x};
    put_partials<1>(acc, dst);
}

// One block: H[j+1,j] = ||w||, Givens rotations, residual estimate, stop test.
__global__ void __launch_bounds__(KBLOCK) k_gm_finish(GmSys G, int j, int nb) {
    if (G.sc->ks.done) return;
    double tot[1];
    const double *src[1] = {G.part + (size_t)(GM_M + 1) * nb};
    sum_partials<1>(src, nb, tot);
    if (threadIdx.x != 0) return;
    GmScal &s = *G.sc;
    double *Hc = s.H + (GM_M + 1) * j;
    const double nw = sqrt(tot[0]);
    Hc[j + 1] = nw;
    for (int i = 0; i < j; i++) {
        const double a = Hc[i], b = Hc[i + 1];
        Hc[i] = s.cs[i] * a + s.sn[i] * b;
        Hc[i + 1] = -s.sn[i] * a + s.cs[i] * b;
    }
    const double a = Hc[j], b = Hc[j + 1], rho = hypot(a, b);
    const double c = rho > 0.0 ? a / rho : 1.0, sn = rho > 0.0 ? b / rho : 0.0;
    Hc[j] = rho;
    Hc[j + 1] = 0.0;
    s.cs[j] = c;
    s.sn[j] = sn;
    s.g[j + 1] = -sn * s.g[j];
    s.g[j] = c * s.g[j];
    s.iters += 1;
    s.j = j + 1;
    s.hinv = nw > 0.0 ? 1.0 / nw : 0.0;
    const double res = fabs(s.g[j + 1]);
    s.ks.rnorm = res;
    if (res <= s.ks.thr || j + 1 == GM_M || nw == 0.0) {
        s.ks.done = 1;
        s.cycle_end = 1;
        s.ks.final_iters = s.iters;
    }
}

template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_scale(Op A, GmSys G, int j) {
    if (G.sc->ks.done) return;
    const double hi = G.sc->hinv;
    A.each([&](const Idx &x_) {
        const int c = x_.c;
        G.V[j + 1][c] *= hi;
    });
}

// One block: y = R^-1 g over the cycle's k steps.
__global__ void k_gm_solve(GmSys G) {
    if (threadIdx.x != 0) return;
    GmScal &s = *G.sc;
    const int k = s.j;
    for (int i = k - 1; i >= 0; i--) {
        double v = s.g[i];
        for (int l = i + 1; l < k; l++) v -= s.H[(GM_M + 1) * l + i] * s.y[l];
        const double d = s.H[(GM_M + 1) * i + i];
        s.y[i] = d != 0.0 ? v / d : 0.0;
    }
}

// u = sum_{i<k} y_i V[i] into V[k].
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_combine(Op A, GmSys G, int k) {
    double y[GM_M];
#pragma unroll
    for (int i = 0; i < GM_M; i++) y[i] = i < k ? G.sc->y[i] : 0.0;
    A.each([&](const Idx &x_) {
        const int c = x_.c;
        double u = 0.0;
#pragma unroll
        for (int i = 0; i < GM_M; i++)
            if (i < k) u += y[i] * G.V[i][c];
        G.V[k][c] = u;
    });
}

// x += z, r -= A z (z = M^-1 V y); partials r.r in slot 0.
template <class Op>
__global__ void __launch_bounds__(KBLOCK) k_gm_update(Op A, GmSys G) {
    double acc[1] = {0.0};
    A.each([&](const Idx &x) {
        const int c = x.c;
        G.x[c] = G.x[c] + (double)G.z[c];
        const double r = G.r[c] - A.apply_z(G.z, G.ap, x);
        G.r[c] = r;
        acc[0] += r * r;
    });
    double *const dst[1] = {G.part};
    put_partials<1>(acc, dst);
}

}  // namespace cms
