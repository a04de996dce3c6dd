// MMA (Svanberg) and CONLIN for one constraint on the device: the O(n) passes of
// MMA<T>::UpdateVariables (src/Optimize/Solver/MMA.h:116-419) as kernels
// with fixed-order workgroup partials; the O(1) scalar algebra of the
// primal-dual interior-point iteration (the (m+1)^2 = 2x2 Newton system
// solved by solvels, MMA.h:464-509) runs on the host between launches.
// Included by pf_capi.hip (same translation unit, no FP contraction).
#pragma once

namespace pf {

// Asymptotes (MMA.h:118-142), move limits (145-150), p0, q0, p, q and the
// b-sum terms (153-175).  xmin/xmax are uniform.
__global__ void __launch_bounds__(256) k_mma_prep(long n, int early, const double* __restrict__ xk,
                                                  const double* __restrict__ xkm1, const double* __restrict__ xkm2,
                                                  double* __restrict__ L, double* __restrict__ U, double xmin,
                                                  double xmax, double asyinit, double asydecr, double asyincr,
                                                  double albefa, double move, double raa0,
                                                  const double* __restrict__ dfdx, const double* __restrict__ dgdx,
                                                  double* __restrict__ alpha, double* __restrict__ beta,
                                                  double* __restrict__ p0, double* __restrict__ q0,
                                                  double* __restrict__ p, double* __restrict__ q,
                                                  double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[1] = {0.0};
    const double dx = xmax - xmin;
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        double x = xk[j], l, u;
        if (early) {
            l = x - asyinit * dx;
            u = x + asyinit * dx;
        } else {
            double tmp = (x - xkm1[j]) * (xkm1[j] - xkm2[j]);
            double lo = L[j], up = U[j], x1 = xkm1[j];
            if (tmp < 0.0) {
                l = x - asydecr * (x1 - lo);
                u = x + asydecr * (up - x1);
            } else if (tmp > 0.0) {
                l = x - asyincr * (x1 - lo);
                u = x + asyincr * (up - x1);
            } else {
                l = x - (x1 - lo);
                u = x + (up - x1);
            }
        }
        // std::min(std::max(a, b), c)
        double a1 = x - 10.0 * dx, c1 = x - 0.01 * dx;
        double m1 = (a1 < l) ? l : a1;
        l = (c1 < m1) ? c1 : m1;
        double a2 = x + 0.01 * dx, c2 = x + 10.0 * dx;
        double m2 = (a2 < u) ? u : a2;
        u = (c2 < m2) ? c2 : m2;
        L[j] = l;
        U[j] = u;
        // std::max({xmin, L + albefa (x - L), x - move dx}) / std::min({...})
        double al = xmin, t1 = l + albefa * (x - l), t2 = x - move * dx;
        if (al < t1) al = t1;
        if (al < t2) al = t2;
        double be = xmax, s1 = u - albefa * (u - x), s2 = x + move * dx;
        if (s1 < be) be = s1;
        if (s2 < be) be = s2;
        alpha[j] = al;
        beta[j] = be;
        double ux = u - x, xl = x - l;
        double df = dfdx[j];
        double dp = (df < 0.0) ? 0.0 : df, dm = (-df < 0.0) ? 0.0 : -df;  // std::max(v, T())
        p0[j] = (ux * ux) * (1.001 * dp + 0.001 * dm + raa0 / dx);
        q0[j] = (xl * xl) * (0.001 * dp + 1.001 * dm + raa0 / dx);
        double dg = dgdx[j];
        double gp = (dg < 0.0) ? 0.0 : dg, gm = (-dg < 0.0) ? 0.0 : -dg;
        double pj = (ux * ux) * (1.001 * gp + 0.001 * gm + raa0 / dx);
        double qj = (xl * xl) * (0.001 * gp + 1.001 * gm + raa0 / dx);
        p[j] = pj;
        q[j] = qj;
        acc[0] += pj / ux + qj / xl;
    }
    store_partials<1>(acc, lds, part);
}

// Interior-point start (MMA.h:192-196).
__global__ void k_mma_start(long n, const double* __restrict__ alpha, const double* __restrict__ beta,
                            double* __restrict__ x, double* __restrict__ gsi, double* __restrict__ ita) {
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        double xv = 0.5 * (alpha[j] + beta[j]);
        double g = 1.0 / (xv - alpha[j]), t = 1.0 / (beta[j] - xv);
        x[j] = xv;
        gsi[j] = (1.0 < g) ? g : 1.0;
        ita[j] = (1.0 < t) ? t : 1.0;
    }
}

// KKT residual terms of equations (5.9a,e,f) at one point (MMA.h:439-443).
__device__ inline double mma_kkt_terms(double x, double gs, double it, double lam, double eps, double al, double be,
                                       double l, double u, double p0, double q0, double p, double q, double& gsum) {
    double pl = p0 + lam * p, ql = q0 + lam * q;
    double ux = u - x, xl = x - l;
    gsum = p / ux + q / xl;
    double a = pl / (ux * ux) - ql / (xl * xl) - gs + it;
    double e = gs * (x - al) - eps;
    double f = it * (be - x) - eps;
    double s = 0.0;
    s += a * a;
    s += e * e;
    s += f * f;
    return s;
}

// Newton coefficients (MMA.h:201-222) and the n-sums of the 2x2 system
// (MMA.h:260-278): partials of sum(p/(U-x) + q/(x-L)), sum(G^2/Dx),
// sum(G dlx/Dx) and the KKT norm terms at the current point.
__global__ void __launch_bounds__(256) k_mma_newton_a(long n, double lam, double eps, const double* __restrict__ x,
                                                      const double* __restrict__ gsi, const double* __restrict__ ita,
                                                      const double* __restrict__ alpha, const double* __restrict__ beta,
                                                      const double* __restrict__ L, const double* __restrict__ U,
                                                      const double* __restrict__ p0, const double* __restrict__ q0,
                                                      const double* __restrict__ p, const double* __restrict__ q,
                                                      double* __restrict__ G, double* __restrict__ Dx,
                                                      double* __restrict__ dlx, double* __restrict__ part) {
    __shared__ double lds[64];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        double xv = x[j], l = L[j], u = U[j], al = alpha[j], be = beta[j];
        double pl = p0[j] + lam * p[j], ql = q0[j] + lam * q[j];
        double ux = u - xv, xl = xv - l;
        double ux2 = ux * ux, xl2 = xl * xl;
        double g = p[j] / ux2 - q[j] / xl2;
        double d = 2.0 * pl / cube_rn(ux) + 2.0 * ql / cube_rn(xl) + gsi[j] / (xv - al) + ita[j] / (be - xv);
        double dl = pl / ux2 - ql / xl2 - eps / (xv - al) + eps / (be - xv);
        G[j] = g;
        Dx[j] = d;
        dlx[j] = dl;
        double gs;
        double kt = mma_kkt_terms(xv, gsi[j], ita[j], lam, eps, al, be, l, u, p0[j], q0[j], p[j], q[j], gs);
        acc[0] += gs;
        acc[1] += g * g / d;
        acc[2] += g * dl / d;
        acc[3] += kt;
    }
    store_partials<4>(acc, lds, part);
}

// Newton direction of the primal variables (MMA.h:283-290, 303-306) and the
// step bound over j (MMA.h:347-352): partial maxima.
__global__ void __launch_bounds__(256) k_mma_newton_b(long n, double dlam, double eps, const double* __restrict__ x,
                                                      const double* __restrict__ gsi, const double* __restrict__ ita,
                                                      const double* __restrict__ alpha, const double* __restrict__ beta,
                                                      const double* __restrict__ G, const double* __restrict__ Dx,
                                                      const double* __restrict__ dlx, double* __restrict__ dx,
                                                      double* __restrict__ dgsi, double* __restrict__ dita,
                                                      double* __restrict__ part) {
    __shared__ double lds[16];
    double mx = 0.0;  // txmax starts at T()
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        double xv = x[j], al = alpha[j], be = beta[j], d = Dx[j];
        double v = -dlx[j] / d;
        v -= G[j] * dlam / d;
        double gs = gsi[j], it = ita[j];
        double dg = -gs * v / (xv - al) - gs + eps / (xv - al);
        double di = it * v / (be - xv) - it + eps / (be - xv);
        dx[j] = v;
        dgsi[j] = dg;
        dita[j] = di;
        double t = -1.01 * v / (xv - al);
        double t2 = 1.01 * v / (be - xv);
        double t3 = -1.01 * dg / gs;
        double t4 = -1.01 * di / it;
        if (t < t2) t = t2;
        if (t < t3) t = t3;
        if (t < t4) t = t4;
        if (mx < t) mx = t;
    }
    // block max (order-free)
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        double o = __shfl_xor(mx, off, 64);
        mx = (mx < o) ? o : mx;
    }
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = lds[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = (m < lds[w]) ? lds[w] : m;
        part[blockIdx.x] = m;
    }
}

// Trial point of the line search (MMA.h:372-385): writes x + tau dx etc. and
// the partial KKT sums at that point.
__global__ void __launch_bounds__(256) k_mma_trial(long n, double tau, double lam, double eps,
                                                   const double* __restrict__ x, const double* __restrict__ gsi,
                                                   const double* __restrict__ ita, const double* __restrict__ dx,
                                                   const double* __restrict__ dgsi, const double* __restrict__ dita,
                                                   const double* __restrict__ alpha, const double* __restrict__ beta,
                                                   const double* __restrict__ L, const double* __restrict__ U,
                                                   const double* __restrict__ p0, const double* __restrict__ q0,
                                                   const double* __restrict__ p, const double* __restrict__ q,
                                                   double* __restrict__ xp, double* __restrict__ gp,
                                                   double* __restrict__ ip, double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[2] = {0.0, 0.0};
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        double xv = x[j] + tau * dx[j];
        double gv = gsi[j] + tau * dgsi[j];
        double iv = ita[j] + tau * dita[j];
        xp[j] = xv;
        gp[j] = gv;
        ip[j] = iv;
        double gs;
        acc[0] += mma_kkt_terms(xv, gv, iv, lam, eps, alpha[j], beta[j], L[j], U[j], p0[j], q0[j], p[j], q[j], gs);
        acc[1] += gs;
    }
    store_partials<2>(acc, lds, part);
}

// ------------------------------------------------------------- CONLIN ----
// CONLIN<T> (src/Optimize/Solver/CONLIN.h:90-365) shares the interior-point
// driver; only the approximation differs: p x + q / x with p, q the positive
// and negative parts of the derivative (q scaled by x_k^2), move limits
// without asymptotes.

// Move limits (CONLIN.h:92-96), p0, q0 (99-105), p, q and the b-sum terms
// (108-120).
__global__ void __launch_bounds__(256) k_conlin_prep(long n, const double* __restrict__ xk, double xmin, double xmax,
                                                     double move, const double* __restrict__ dfdx,
                                                     const double* __restrict__ dgdx, double* __restrict__ alpha,
                                                     double* __restrict__ beta, double* __restrict__ p0,
                                                     double* __restrict__ q0, double* __restrict__ p,
                                                     double* __restrict__ q, double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[1] = {0.0};
    const double dx = xmax - xmin;
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        const double x = xk[j];
        // std::max({xmin, x - move dx}), std::min({xmax, x + move dx})
        double al = xmin, t1 = x - move * dx;
        if (al < t1) al = t1;
        double be = xmax, t2 = x + move * dx;
        if (t2 < be) be = t2;
        alpha[j] = al;
        beta[j] = be;
        const double x2 = x * x;  // pow(x, 2.0)
        const double df = dfdx[j], dg = dgdx[j];
        p0[j] = (df < 0.0) ? 0.0 : df;
        q0[j] = ((-df < 0.0) ? 0.0 : -df) * x2;
        const double pj = (dg < 0.0) ? 0.0 : dg;
        const double qj = ((-dg < 0.0) ? 0.0 : -dg) * x2;
        p[j] = pj;
        q[j] = qj;
        acc[0] += pj * x + qj / x;
    }
    store_partials<1>(acc, lds, part);
}

// KKT residual terms of equations (5.9a,e,f) (CONLIN.h:392-396).
__device__ inline double conlin_kkt_terms(double x, double gs, double it, double lam, double eps, double al,
                                          double be, double p0, double q0, double p, double q, double& gsum) {
    const double pl = p0 + lam * p, ql = q0 + lam * q;
    gsum = p * x + q / x;
    const double a = pl - ql / (x * x) - gs + it;
    const double e = gs * (x - al) - eps;
    const double f = it * (be - x) - eps;
    double s = 0.0;
    s += a * a;
    s += e * e;
    s += f * f;
    return s;
}

// Newton coefficients (CONLIN.h:143-170) and the n-sums of the 2x2 system,
// as k_mma_newton_a.
__global__ void __launch_bounds__(256) k_conlin_newton_a(long n, double lam, double eps, const double* __restrict__ x,
                                                         const double* __restrict__ gsi, const double* __restrict__ ita,
                                                         const double* __restrict__ alpha,
                                                         const double* __restrict__ beta, const double* __restrict__ p0,
                                                         const double* __restrict__ q0, const double* __restrict__ p,
                                                         const double* __restrict__ q, double* __restrict__ G,
                                                         double* __restrict__ Dx, double* __restrict__ dlx,
                                                         double* __restrict__ part) {
    __shared__ double lds[64];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        const double xv = x[j], al = alpha[j], be = beta[j];
        const double pl = p0[j] + lam * p[j], ql = q0[j] + lam * q[j];
        const double x2 = xv * xv;
        const double g = p[j] - q[j] / x2;
        const double d = 2.0 * ql / cube_rn(xv) + gsi[j] / (xv - al) + ita[j] / (be - xv);
        const double dl = pl - ql / x2 - eps / (xv - al) + eps / (be - xv);
        G[j] = g;
        Dx[j] = d;
        dlx[j] = dl;
        double gs;
        const double kt = conlin_kkt_terms(xv, gsi[j], ita[j], lam, eps, al, be, p0[j], q0[j], p[j], q[j], gs);
        acc[0] += gs;
        acc[1] += g * g / d;
        acc[2] += g * dl / d;
        acc[3] += kt;
    }
    store_partials<4>(acc, lds, part);
}

// Trial point of the line search (CONLIN.h:318-340), as k_mma_trial.
__global__ void __launch_bounds__(256) k_conlin_trial(long n, double tau, double lam, double eps,
                                                      const double* __restrict__ x, const double* __restrict__ gsi,
                                                      const double* __restrict__ ita, const double* __restrict__ dx,
                                                      const double* __restrict__ dgsi, const double* __restrict__ dita,
                                                      const double* __restrict__ alpha, const double* __restrict__ beta,
                                                      const double* __restrict__ p0, const double* __restrict__ q0,
                                                      const double* __restrict__ p, const double* __restrict__ q,
                                                      double* __restrict__ xp, double* __restrict__ gp,
                                                      double* __restrict__ ip, double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[2] = {0.0, 0.0};
    for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
        const double xv = x[j] + tau * dx[j];
        const double gv = gsi[j] + tau * dgsi[j];
        const double iv = ita[j] + tau * dita[j];
        xp[j] = xv;
        gp[j] = gv;
        ip[j] = iv;
        double gs;
        acc[0] += conlin_kkt_terms(xv, gv, iv, lam, eps, alpha[j], beta[j], p0[j], q0[j], p[j], q[j], gs);
        acc[1] += gs;
    }
    store_partials<2>(acc, lds, part);
}

// ------------------------------------------------- resident update -----
// The whole UpdateVariables in one cooperative launch: the approximation, the
// interior point and the Newton direction of S variables per thread stay in
// registers (17 values each; with four variables 41 of them, CONLIN 25, go to
// scratch), the scalar algebra runs in every thread on sums
// that all workgroups add in one order (res_publish, res_collect).  The
// launched form reads and writes 16 vectors per Newton step and returns to
// the host four times for its sums.  Measured through pf_mma_update (host
// vectors, 35 steps): 4.7 ms at 524,288 variables launched, 1.6 resident, of
// which 1 ms are the copies; 2.1 and 0.4 ms at 4,800.  What bounds it are the
// exchanges (about 2.5 us each, at least three per Newton step) and, with four
// variables per thread, the divisions between them.
struct MmaRes {
    long n;
    int early, max_newton;
    unsigned tag;
    double a0, a, c, d, xmin, xmax, raa0, albefa, move, asyinit, asydecr, asyincr, g;
    const double *xk, *xkm1, *xkm2, *L, *U, *dfdx, *dgdx;
    double *xo, *Lo, *Uo;  // the new x, L and U
    u64* slots;
    ResDev* R;  // v[0]: Newton steps, v[1]: 1 when max_newton was reached
};
constexpr int kMmaResThreads = 512;

// MMA<T>::solvels for the 2x2 system (MMA.h:464-509).
__host__ __device__ inline void mma_solve2(double A00, double A01, double A10, double A11, double b0, double b1,
                                           double& x0, double& x1) {
    if (fabs(A00) < fabs(A10)) {
        double s = b0; b0 = b1; b1 = s;
        s = A00; A00 = A10; A10 = s;
        s = A01; A01 = A11; A11 = s;
    }
    A11 -= A01 * A10 / A00;
    b1 -= b0 * A10 / A00;
    x1 = b1;
    x1 /= A11;
    x0 = b0;
    x0 -= x1 * A01;
    x0 /= A00;
}

template <int S, bool CONLIN>
__global__ void __launch_bounds__(kMmaResThreads) k_mma_resident(MmaRes M) {
    __shared__ ResLds lds;
    constexpr int NT = kMmaResThreads;
    if (threadIdx.x == 0) lds.bad = 0;
    __syncthreads();
    unsigned tag = M.tag;
    auto fail = [&]() {
        if (threadIdx.x == 0) M.R->stall = 1;
    };
    auto index = [&](int s) { return ((long)blockIdx.x * S + s) * NT + threadIdx.x; };
    double L[CONLIN ? 1 : S], U[CONLIN ? 1 : S], al[S], be[S], p0[S], q0[S], p[S], q[S], x[S], gsi[S], ita[S];
    double dx[S], dg[S], di[S];
    const double wd = M.xmax - M.xmin;
    double acc1[1] = {0.0};
#pragma unroll
    for (int s = 0; s < S; s++) {
        const long j = index(s);
        const bool on = j < M.n;
        const double xv = on ? M.xk[j] : 0.5, df = on ? M.dfdx[j] : 0.0, dgj = on ? M.dgdx[j] : 0.0;
        double bs;
        if constexpr (CONLIN) {  // k_conlin_prep
            double a = M.xmin, t1 = xv - M.move * wd;
            if (a < t1) a = t1;
            double b = M.xmax, t2 = xv + M.move * wd;
            if (t2 < b) b = t2;
            al[s] = a;
            be[s] = b;
            const double x2 = xv * xv;
            p0[s] = (df < 0.0) ? 0.0 : df;
            q0[s] = ((-df < 0.0) ? 0.0 : -df) * x2;
            p[s] = (dgj < 0.0) ? 0.0 : dgj;
            q[s] = ((-dgj < 0.0) ? 0.0 : -dgj) * x2;
            bs = p[s] * xv + q[s] / xv;
        } else {  // k_mma_prep
            double l, u;
            if (M.early || !on) {
                l = xv - M.asyinit * wd;
                u = xv + M.asyinit * wd;
            } else {
                const double x1 = M.xkm1[j], lo = M.L[j], up = M.U[j];
                const double tmp = (xv - x1) * (x1 - M.xkm2[j]);
                if (tmp < 0.0) {
                    l = xv - M.asydecr * (x1 - lo);
                    u = xv + M.asydecr * (up - x1);
                } else if (tmp > 0.0) {
                    l = xv - M.asyincr * (x1 - lo);
                    u = xv + M.asyincr * (up - x1);
                } else {
                    l = xv - (x1 - lo);
                    u = xv + (up - x1);
                }
            }
            const double a1 = xv - 10.0 * wd, c1 = xv - 0.01 * wd;
            const double m1 = (a1 < l) ? l : a1;
            l = (c1 < m1) ? c1 : m1;
            const double a2 = xv + 0.01 * wd, c2 = xv + 10.0 * wd;
            const double m2 = (a2 < u) ? u : a2;
            u = (c2 < m2) ? c2 : m2;
            L[s] = l;
            U[s] = u;
            double a = M.xmin, t1 = l + M.albefa * (xv - l), t2 = xv - M.move * wd;
            if (a < t1) a = t1;
            if (a < t2) a = t2;
            double b = M.xmax, s1 = u - M.albefa * (u - xv), s2 = xv + M.move * wd;
            if (s1 < b) b = s1;
            if (s2 < b) b = s2;
            al[s] = a;
            be[s] = b;
            const double ux = u - xv, xl = xv - l;
            const double dp = (df < 0.0) ? 0.0 : df, dm = (-df < 0.0) ? 0.0 : -df;
            p0[s] = (ux * ux) * (1.001 * dp + 0.001 * dm + M.raa0 / wd);
            q0[s] = (xl * xl) * (0.001 * dp + 1.001 * dm + M.raa0 / wd);
            const double gp = (dgj < 0.0) ? 0.0 : dgj, gm = (-dgj < 0.0) ? 0.0 : -dgj;
            p[s] = (ux * ux) * (1.001 * gp + 0.001 * gm + M.raa0 / wd);
            q[s] = (xl * xl) * (0.001 * gp + 1.001 * gm + M.raa0 / wd);
            bs = p[s] / ux + q[s] / xl;
        }
        if (on) acc1[0] += bs;
        // k_mma_start
        const double xs = 0.5 * (al[s] + be[s]);
        const double g = 1.0 / (xs - al[s]), t = 1.0 / (be[s] - xs);
        x[s] = xs;
        gsi[s] = (1.0 < g) ? g : 1.0;
        ita[s] = (1.0 < t) ? t : 1.0;
    }
    res_publish<1, NT>(acc1, lds, M.slots, tag);
    if (!res_collect<1, NT>(acc1, lds, M.slots, tag)) return fail();
    tag++;
    const double a = M.a, c = M.c, d = M.d, a0 = M.a0;
    const double b = -M.g + acc1[0];
    double eps = 1.0, y = 1.0, z = 1.0, zeta = 1.0, lam = 1.0, sv = 1.0;
    double mu = (1.0 < 0.5 * c) ? 0.5 * c : 1.0;
    auto kkt_terms = [&](int s, double xv, double gs, double it, double l, double& gsum) {
        if constexpr (CONLIN)
            return conlin_kkt_terms(xv, gs, it, l, eps, al[s], be[s], p0[s], q0[s], p[s], q[s], gsum);
        else
            return mma_kkt_terms(xv, gs, it, l, eps, al[s], be[s], L[s], U[s], p0[s], q0[s], p[s], q[s], gsum);
    };
    auto kkt = [&](double Ksum, double gsum, double yv, double zv, double lv, double mv, double zetav, double ssv) {
        double norm = Ksum;
        double t;
        t = c + d * yv - lv - mv; norm += t * t;
        t = gsum - a * zv - yv + ssv - b; norm += t * t;
        t = mv * yv - eps; norm += t * t;
        t = lv * ssv - eps; norm += t * t;
        t = a0 - zetav - (0.0 + lv * a); norm += t * t;
        t = zetav * zv - eps; norm += t * t;
        return sqrt(norm);
    };
    int l = 0;
    for (; eps > 1.0e-7; l++) {
        if (l >= M.max_newton) {
            if (threadIdx.x == 0 && blockIdx.x == 0) {
                M.R->v[0] = l;
                M.R->v[1] = 1.0;
            }
            return;
        }
        // Newton coefficients: G, Dx, dlx as in k_mma_newton_a / k_conlin_newton_a
        double G[S], Dx[S], dl[S];
        double Sm[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < S; s++) {
            const double xv = x[s], pl = p0[s] + lam * p[s], ql = q0[s] + lam * q[s];
            if constexpr (CONLIN) {
                const double x2 = xv * xv;
                G[s] = p[s] - q[s] / x2;
                Dx[s] = 2.0 * ql / cube_rn(xv) + gsi[s] / (xv - al[s]) + ita[s] / (be[s] - xv);
                dl[s] = pl - ql / x2 - eps / (xv - al[s]) + eps / (be[s] - xv);
            } else {
                const double ux = U[s] - xv, xl = xv - L[s];
                const double ux2 = ux * ux, xl2 = xl * xl;
                G[s] = p[s] / ux2 - q[s] / xl2;
                Dx[s] = 2.0 * pl / cube_rn(ux) + 2.0 * ql / cube_rn(xl) + gsi[s] / (xv - al[s]) +
                        ita[s] / (be[s] - xv);
                dl[s] = pl / ux2 - ql / xl2 - eps / (xv - al[s]) + eps / (be[s] - xv);
            }
            double gs;
            const double kt = kkt_terms(s, xv, gsi[s], ita[s], lam, gs);
            if (index(s) < M.n) {
                Sm[0] += gs;
                Sm[1] += G[s] * G[s] / Dx[s];
                Sm[2] += G[s] * dl[s] / Dx[s];
                Sm[3] += kt;
            }
        }
        res_publish<4, NT>(Sm, lds, M.slots, tag);
        if (!res_collect<4, NT>(Sm, lds, M.slots, tag)) return fail();
        tag++;
        const double Dy = d + mu / y;
        const double Dl = sv / lam;
        const double dly = c + d * y - lam - eps / y;
        const double dlz = a0 - eps / z - (0.0 + lam * a);
        double dll = -a * z - y - b + eps / lam;
        dll += Sm[0];
        const double Dlly = Dl + 1.0 / Dy;
        const double dlly = dll + dly / Dy;
        double A00 = 0.0 + Sm[1];
        A00 += Dlly;
        double dlam, dz;
        mma_solve2(A00, a, a, -zeta / z, dlly - Sm[2], dlz, dlam, dz);
        // the direction and the step bound, as in k_mma_newton_b
        double mx[1] = {0.0};
#pragma unroll
        for (int s = 0; s < S; s++) {
            const double xv = x[s];
            double v = -dl[s] / Dx[s];
            v -= G[s] * dlam / Dx[s];
            const double gs = gsi[s], it = ita[s];
            dx[s] = v;
            dg[s] = -gs * v / (xv - al[s]) - gs + eps / (xv - al[s]);
            di[s] = it * v / (be[s] - xv) - it + eps / (be[s] - xv);
            double t = -1.01 * v / (xv - al[s]);
            const double t2 = 1.01 * v / (be[s] - xv), t3 = -1.01 * dg[s] / gs, t4 = -1.01 * di[s] / it;
            if (t < t2) t = t2;
            if (t < t3) t = t3;
            if (t < t4) t = t4;
            if (index(s) < M.n && mx[0] < t) mx[0] = t;
        }
        res_publish<1, NT, true>(mx, lds, M.slots, tag);
        const double dy = dlam / Dy - dly / Dy;
        const double dmu = -mu * dy / y - mu + eps / y;
        const double ds = -sv * dlam / lam - sv + eps / lam;
        const double dzeta = -zeta * dz / z - zeta + eps / z;
        double tymax = 0.0;
        {
            double t = -1.01 * dy / y;
            const double t2 = -1.01 * dlam / lam, t3 = -1.01 * dmu / mu, t4 = -1.01 * ds / sv;
            if (t < t2) t = t2;
            if (t < t3) t = t3;
            if (t < t4) t = t4;
            if (tymax < t) tymax = t;
        }
        const double deltawl = kkt(Sm[3], Sm[0], y, z, lam, mu, zeta, sv);
        if (!res_collect<1, NT, true>(mx, lds, M.slots, tag)) return fail();
        tag++;
        double m5 = 1.0;
        const double tz = -1.01 * dz / z, tzeta = -1.01 * dzeta / zeta;
        if (m5 < mx[0]) m5 = mx[0];
        if (m5 < tymax) m5 = tymax;
        if (m5 < tz) m5 = tz;
        if (m5 < tzeta) m5 = tzeta;
        double tau = 1.0 / m5;
        double yp = y, lp = lam, mp = mu, sp = sv, zp = z, zetap = zeta, dw1 = 0.0, taken = tau;
        for (int ll = 0; ll < 50; ll++) {
            yp = y + tau * dy;
            lp = lam + tau * dlam;
            mp = mu + tau * dmu;
            sp = sv + tau * ds;
            zp = z + tau * dz;
            zetap = zeta + tau * dzeta;
            double T[2] = {0.0, 0.0};
#pragma unroll
            for (int s = 0; s < S; s++) {
                double gs;
                const double kt = kkt_terms(s, x[s] + tau * dx[s], gsi[s] + tau * dg[s], ita[s] + tau * di[s], lp, gs);
                if (index(s) < M.n) {
                    T[0] += kt;
                    T[1] += gs;
                }
            }
            res_publish<2, NT>(T, lds, M.slots, tag);
            if (!res_collect<2, NT>(T, lds, M.slots, tag)) return fail();
            tag++;
            taken = tau;
            dw1 = kkt(T[0], T[1], yp, zp, lp, mp, zetap, sp);
            if (dw1 < deltawl) break;
            tau *= 0.5;
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
            x[s] = x[s] + taken * dx[s];
            gsi[s] = gsi[s] + taken * dg[s];
            ita[s] = ita[s] + taken * di[s];
        }
        y = yp; z = zp; lam = lp; mu = mp; zeta = zetap; sv = sp;
        if (dw1 < 0.9 * eps) eps *= 0.1;
    }
#pragma unroll
    for (int s = 0; s < S; s++) {
        const long j = index(s);
        if (j >= M.n) continue;
        M.xo[j] = x[s];
        if constexpr (!CONLIN) {
            M.Lo[j] = L[s];
            M.Uo[j] = U[s];
        }
    }
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        M.R->v[0] = l;
        M.R->v[1] = 0.0;
    }
}

}  // namespace pf
