// Geometric multigrid V-cycle for the hex8 matrix-free operator (the 3D
// counterpart of pf_mg.hip; no counterpart in the reference).
//
// Level l+1 halves the three element counts; a coarse element's 24 x 24
// matrix is the Galerkin product sum_a P_a^T K_a P_a of its eight children's
// (trilinear P_a, the same weights for the three DOF directions; fixed DOFs
// removed at level 0 by zeroing their rows and columns).  Nodes (i, j, k) ->
// ((ny+1)(nz+1)) i + (nz+1) j + k; element-local node q at offsets
// (0,0,0), (1,0,0), (1,1,0), (0,1,0), then the same four at dk = 1
// (ShapeFunction8Cubic order).  Vectors are nodal, 3 entries per node.
// Smoothing is damped Jacobi in two passes per sweep (an elementwise update,
// then an operator application that gathers the updated vector), since a
// 3D node's operator row touches 27 nodes through 8 elements.
#pragma once

#include "pf_device.h"

namespace pf {

__device__ inline void mg3_lxyz(int q, int& x, int& y, int& z) {
    z = q >> 2;
    const int m = q & 3;
    x = (m == 1 || m == 2) ? 1 : 0;
    y = (m >= 2) ? 1 : 0;
}

// element-matrix sources (FP32): level 0 E_e K0, coarse levels one 24 x 24
// matrix per element
struct Mg3KeShared {
    const float* E;
    const float* K0;
    __device__ float operator()(long e, int r, int c) const { return E[e] * K0[r * 24 + c]; }
};
struct Mg3KeFull {
    const float* Ke;
    __device__ float operator()(long e, int r, int c) const { return Ke[e * 576 + r * 24 + c]; }
};

// (A x) at node (i, j, k) over its (up to) eight elements
template <class KE>
__device__ inline void mg3_node_apply(int nx, int ny, int nz, int i, int j, int k, const KE& ke,
                                      const float* __restrict__ x, float (&ax)[3]) {
#pragma clang fp contract(fast)  // preconditioner arithmetic: FMA allowed
    ax[0] = ax[1] = ax[2] = 0.f;
    const long pl = (long)(ny + 1) * (nz + 1);
    for (int ea = 0; ea < 2; ea++) {
        const int ei = i - 1 + ea;
        if (ei < 0 || ei >= nx) continue;
        for (int eb = 0; eb < 2; eb++) {
            const int ej = j - 1 + eb;
            if (ej < 0 || ej >= ny) continue;
            for (int ec = 0; ec < 2; ec++) {
                const int ek = k - 1 + ec;
                if (ek < 0 || ek >= nz) continue;
                const long e = ((long)ny * nz) * ei + (long)nz * ej + ek;
                const int di = i - ei, dj = j - ej, dk = k - ek;
                const int me = 4 * dk + (dj == 0 ? di : 3 - di);
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    int qx, qy, qz;
                    mg3_lxyz(q, qx, qy, qz);
                    const long m = pl * (ei + qx) + (long)(nz + 1) * (ej + qy) + (ek + qz);
                    const float u0 = x[3 * m], u1 = x[3 * m + 1], u2 = x[3 * m + 2];
#pragma unroll
                    for (int r = 0; r < 3; r++)
                        ax[r] += ke(e, 3 * me + r, 3 * q) * u0 + ke(e, 3 * me + r, 3 * q + 1) * u1 +
                                 ke(e, 3 * me + r, 3 * q + 2) * u2;
                }
            }
        }
    }
}

// x + omega D^-1 res (x null: 0; res null: r), masked, at DOF t
__device__ inline float mg3_update_val(long t, float omega, const float* __restrict__ x,
                                       const float* __restrict__ res, const float* __restrict__ r,
                                       const float* __restrict__ D, const uint8_t* __restrict__ fix) {
    const long n = t / 3;
    const int d = (int)(t - 3 * n);
    const float rs = res ? res[t] : r[t];
    float v = (x ? x[t] : 0.f) + omega * rs / D[t];
    if ((fix[n] >> d) & 1) v = 0.f;
    return v;
}

__device__ inline void mg3_update_at(long t, float omega, const float* __restrict__ x,
                                     const float* __restrict__ res, const float* __restrict__ r,
                                     const float* __restrict__ D, const uint8_t* __restrict__ fix,
                                     float* __restrict__ out) {
    out[t] = mg3_update_val(t, omega, x, res, r, D, fix);
}

__global__ void __launch_bounds__(256) k_mg3_update(long nv, float omega, const float* __restrict__ x,
                                                    const float* __restrict__ res, const float* __restrict__ r,
                                                    const float* __restrict__ D, const uint8_t* __restrict__ fix,
                                                    float* __restrict__ out, const int* __restrict__ done) {
    if (done && *done) return;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < nv; t += (long)gridDim.x * blockDim.x)
        mg3_update_at(t, omega, x, res, r, D, fix, out);
}

// x + P xc (trilinear prolongation of the coarse correction), masked, at
// node n: its three values
__device__ inline void mg3_prolong_node(long n, int nx, int ny, int nz, const float* __restrict__ x,
                                        const float* __restrict__ xc, const uint8_t* __restrict__ fix,
                                        float (&v)[3]) {
#pragma clang fp contract(fast)
    const long pl = (long)(ny + 1) * (nz + 1);
    const int cny = ny / 2, cnz = nz / 2;
    const long cpl = (long)(cny + 1) * (cnz + 1);
    const int i = (int)(n / pl);
    const long rem = n - (long)i * pl;
    const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
    const int I0 = i >> 1, J0 = j >> 1, K0c = k >> 1, oi = i & 1, oj = j & 1, ok = k & 1;
    float s[3] = {0.f, 0.f, 0.f};
    for (int a = 0; a <= oi; a++)
        for (int b = 0; b <= oj; b++)
            for (int c = 0; c <= ok; c++) {
                const float w = (oi ? 0.5f : 1.f) * (oj ? 0.5f : 1.f) * (ok ? 0.5f : 1.f);
                const long m = cpl * (I0 + a) + (long)(cnz + 1) * (J0 + b) + (K0c + c);
                s[0] += w * xc[3 * m];
                s[1] += w * xc[3 * m + 1];
                s[2] += w * xc[3 * m + 2];
            }
    const uint8_t f = fix[n];
    for (int d = 0; d < 3; d++) v[d] = ((f >> d) & 1) ? 0.f : x[3 * n + d] + s[d];
}

__device__ inline void mg3_prolong_at(long n, int nx, int ny, int nz, const float* __restrict__ x,
                                      const float* __restrict__ xc, const uint8_t* __restrict__ fix,
                                      float* __restrict__ out) {
    float v[3];
    mg3_prolong_node(n, nx, ny, nz, x, xc, fix, v);
    for (int d = 0; d < 3; d++) out[3 * n + d] = v[d];
}

__global__ void __launch_bounds__(256) k_mg3_prolong(int nx, int ny, int nz, const float* __restrict__ x,
                                                     const float* __restrict__ xc, const uint8_t* __restrict__ fix,
                                                     float* __restrict__ out, const int* __restrict__ done) {
    if (done && *done) return;
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x)
        mg3_prolong_at(n, nx, ny, nz, x, xc, fix, out);
}

// res = r - A x (masked) at node n; with x_out, x_out = x + omega D^-1 res
// instead
template <class KE>
__device__ inline void mg3_residual_at(long n, int nx, int ny, int nz, const KE& ke, const float* __restrict__ D,
                                       const uint8_t* __restrict__ fix, float omega, const float* __restrict__ r,
                                       const float* __restrict__ x, float* __restrict__ res,
                                       float* __restrict__ x_out) {
#pragma clang fp contract(fast)
    const long pl = (long)(ny + 1) * (nz + 1);
    const int i = (int)(n / pl);
    const long rem = n - (long)i * pl;
    const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
    float ax[3];
    mg3_node_apply(nx, ny, nz, i, j, k, ke, x, ax);
    const uint8_t f = fix[n];
    for (int d = 0; d < 3; d++) {
        float v = r[3 * n + d] - ax[d];
        if (x_out) v = x[3 * n + d] + omega * v / D[3 * n + d];
        if ((f >> d) & 1) v = 0.f;
        if (x_out)
            x_out[3 * n + d] = v;
        else
            res[3 * n + d] = v;
    }
}

// res = r - A x (masked); with x_out, x_out = x + omega D^-1 res instead
template <class KE>
__global__ void __launch_bounds__(256) k_mg3_residual(int nx, int ny, int nz, KE ke, const float* __restrict__ D,
                                                      const uint8_t* __restrict__ fix, float omega,
                                                      const float* __restrict__ r, const float* __restrict__ x,
                                                      float* __restrict__ res, float* __restrict__ x_out,
                                                      const int* __restrict__ done) {
#pragma clang fp contract(fast)
    if (done && *done) return;
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    // XCD-contiguous node ranges: the four node lines around an element line
    // (and so the nodes that read each element matrix) share an L2
    const BlockRange xr = xcd_block_range(nn);
    for (long n = xr.begin + threadIdx.x; n < xr.end; n += blockDim.x)
        mg3_residual_at(n, nx, ny, nz, ke, D, fix, omega, r, x, res, x_out);
}

// The same residual in two passes for the coarse levels of 1024+ elements,
// where the node form reads each 2.3 KB element matrix from the L2 once per
// node line around it (level 1 at 128 x 64 x 64: 26.6 + 6.0 us against about
// 61 in the node form; levels of 4096 and 1024 elements: about 9.6 against
// 22 and 16 us).  k_mg3_elem_apply: y_e = Ke x_e for every element, thread
// (e, q) forming rows 3q..3q+2 (288 contiguous bytes of the matrix, so the
// element's eight threads read it together, once); k_mg3_node_gather: a
// node's rows are the sum of its elements' y in mg3_node_apply's element
// order, then the residual, update and mask of k_mg3_residual.
constexpr long kMg3ElemMin = 1024;  // elements of a level that takes the two-pass form
// rows 3q..3q+2 of y_e = K_e x_e (xe: the element vector, 24 values) into ye
__device__ inline void mg3_elem_rows(const float* __restrict__ Ke, long e, int q, const float* __restrict__ xe,
                                     float* __restrict__ ye) {
#pragma clang fp contract(fast)
    const float4* K = reinterpret_cast<const float4*>(Ke + e * 576 + 72 * q);
    float acc[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 3; r++) {
        float row[24];
#pragma unroll
        for (int c4 = 0; c4 < 6; c4++) {
            const float4 v = K[6 * r + c4];
            row[4 * c4] = v.x;
            row[4 * c4 + 1] = v.y;
            row[4 * c4 + 2] = v.z;
            row[4 * c4 + 3] = v.w;
        }
#pragma unroll
        for (int p = 0; p < 8; p++)
            acc[r] += row[3 * p] * xe[3 * p] + row[3 * p + 1] * xe[3 * p + 1] + row[3 * p + 2] * xe[3 * p + 2];
    }
    float* y = ye + e * 24 + 3 * q;
    y[0] = acc[0];
    y[1] = acc[1];
    y[2] = acc[2];
}

// Where the two-pass residual's input vector xin comes from: x itself, or
// formed on the fly at each node it is read at (the sweep launches that
// would otherwise precede it, fused): the first pre-smoothing update
// omega D^-1 r, or the coarse correction's prolongation x + P xc.
enum { kMg3In = 0, kMg3InUpdate = 1, kMg3InProlong = 2 };

template <int MODE>
__device__ inline void mg3_xin_node(long m, int nx, int ny, int nz, float omega, const float* __restrict__ x,
                                    const float* __restrict__ xc, const float* __restrict__ r,
                                    const float* __restrict__ D, const uint8_t* __restrict__ fix, float (&u)[3]) {
    if constexpr (MODE == kMg3InUpdate) {
        for (int d = 0; d < 3; d++) u[d] = mg3_update_val(3 * m + d, omega, nullptr, nullptr, r, D, fix);
    } else if constexpr (MODE == kMg3InProlong) {
        mg3_prolong_node(m, nx, ny, nz, x, xc, fix, u);
    } else {
        for (int d = 0; d < 3; d++) u[d] = x[3 * m + d];
    }
}

template <int MODE>
__global__ void __launch_bounds__(256) k_mg3_elem_apply(int nx, int ny, int nz, const float* __restrict__ Ke,
                                                        const float* __restrict__ x, const float* __restrict__ xc,
                                                        const float* __restrict__ r, const float* __restrict__ D,
                                                        const uint8_t* __restrict__ fix, float omega,
                                                        float* __restrict__ ye, const int* __restrict__ done) {
#pragma clang fp contract(fast)
    if (done && *done) return;
    __shared__ float sxe[32 * 24];  // the element vectors of the workgroup's 32 elements
    const long ne = (long)nx * ny * nz;
    const long pl = (long)(ny + 1) * (nz + 1);
    const int le = threadIdx.x >> 3, q = threadIdx.x & 7;
    int qx, qy, qz;
    mg3_lxyz(q, qx, qy, qz);
    const BlockRange xr = xcd_block_range((ne + 31) / 32);  // groups of 32 elements
    for (long grp = xr.begin; grp < xr.end; grp++) {
        const long e = grp * 32 + le;
        const bool ok = e < ne;
        float u0 = 0.f, u1 = 0.f, u2 = 0.f;
        if (ok) {
            const int ei = (int)(e / ((long)ny * nz));
            const long rem = e - (long)ei * ny * nz;
            const int ej = (int)(rem / nz), ek = (int)(rem - (long)ej * nz);
            const long m = pl * (ei + qx) + (long)(nz + 1) * (ej + qy) + (ek + qz);
            float u[3];
            mg3_xin_node<MODE>(m, nx, ny, nz, omega, x, xc, r, D, fix, u);
            u0 = u[0];
            u1 = u[1];
            u2 = u[2];
        }
        float* xe = sxe + le * 24;
        xe[3 * q] = u0;
        xe[3 * q + 1] = u1;
        xe[3 * q + 2] = u2;
        __syncthreads();
        if (ok) mg3_elem_rows(Ke, e, q, xe, ye);
        __syncthreads();  // the next group overwrites sxe
    }
}

// a node's rows of A x gathered from its elements' y_e (mg3_node_apply's
// element order), then the residual, update and mask of mg3_residual_at
// (MODE kMg3InUpdate: x_out receives the update omega D^-1 r, res the
// residual)
template <int MODE = kMg3In>
__device__ inline void mg3_gather_at(long n, int nx, int ny, int nz, const float* __restrict__ ye,
                                     const float* __restrict__ D, const uint8_t* __restrict__ fix, float omega,
                                     const float* __restrict__ r, const float* __restrict__ x,
                                     const float* __restrict__ xc, float* __restrict__ res,
                                     float* __restrict__ x_out) {
    const long pl = (long)(ny + 1) * (nz + 1);
    const int i = (int)(n / pl);
    const long rem = n - (long)i * pl;
    const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
    float ax[3] = {0.f, 0.f, 0.f};
    for (int ea = 0; ea < 2; ea++) {
        const int ei = i - 1 + ea;
        if (ei < 0 || ei >= nx) continue;
        for (int eb = 0; eb < 2; eb++) {
            const int ej = j - 1 + eb;
            if (ej < 0 || ej >= ny) continue;
            for (int ec = 0; ec < 2; ec++) {
                const int ek = k - 1 + ec;
                if (ek < 0 || ek >= nz) continue;
                const long e = ((long)ny * nz) * ei + (long)nz * ej + ek;
                const int di = i - ei, dj = j - ej, dk = k - ek;
                const int me = 4 * dk + (dj == 0 ? di : 3 - di);
                const float* y = ye + e * 24 + 3 * me;
                ax[0] += y[0];
                ax[1] += y[1];
                ax[2] += y[2];
            }
        }
    }
    const uint8_t f = fix[n];
    if constexpr (MODE == kMg3InUpdate) {
        float u[3];
        mg3_xin_node<MODE>(n, nx, ny, nz, omega, x, xc, r, D, fix, u);
        for (int d = 0; d < 3; d++) {
            x_out[3 * n + d] = u[d];
            float v = r[3 * n + d] - ax[d];
            if ((f >> d) & 1) v = 0.f;
            res[3 * n + d] = v;
        }
    } else {
        float u[3];
        if (x_out) mg3_xin_node<MODE>(n, nx, ny, nz, omega, x, xc, r, D, fix, u);
        for (int d = 0; d < 3; d++) {
            float v = r[3 * n + d] - ax[d];
            if (x_out) v = u[d] + omega * v / D[3 * n + d];
            if ((f >> d) & 1) v = 0.f;
            if (x_out)
                x_out[3 * n + d] = v;
            else
                res[3 * n + d] = v;
        }
    }
}

template <int MODE>
__global__ void __launch_bounds__(256) k_mg3_node_gather(int nx, int ny, int nz, const float* __restrict__ ye,
                                                         const float* __restrict__ D, const uint8_t* __restrict__ fix,
                                                         float omega, const float* __restrict__ r,
                                                         const float* __restrict__ x, const float* __restrict__ xc,
                                                         float* __restrict__ res, float* __restrict__ x_out,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    const BlockRange xr = xcd_block_range(nn);
    for (long n = xr.begin + threadIdx.x; n < xr.end; n += blockDim.x)
        mg3_gather_at<MODE>(n, nx, ny, nz, ye, D, fix, omega, r, x, xc, res, x_out);
}

// r_c = P^T res at coarse node n = (I, J, K): the 27 fine nodes
// (2I + a, 2J + b, 2K + c), weights (1 - |a|/2)(1 - |b|/2)(1 - |c|/2), masked
__device__ inline void mg3_restrict_at(long n, int cnx, int cny, int cnz, const float* __restrict__ res,
                                       const uint8_t* __restrict__ cfix, float* __restrict__ rc) {
#pragma clang fp contract(fast)
    const int nx = 2 * cnx, ny = 2 * cny, nz = 2 * cnz;
    const long cpl = (long)(cny + 1) * (cnz + 1), pl = (long)(ny + 1) * (nz + 1);
    const int I = (int)(n / cpl);
    const long rem = n - (long)I * cpl;
    const int J = (int)(rem / (cnz + 1)), K = (int)(rem - (long)J * (cnz + 1));
    float s[3] = {0.f, 0.f, 0.f};
    for (int a = -1; a <= 1; a++)
        for (int b = -1; b <= 1; b++)
            for (int c = -1; c <= 1; c++) {
                const int i = 2 * I + a, j = 2 * J + b, k = 2 * K + c;
                if (i < 0 || i > nx || j < 0 || j > ny || k < 0 || k > nz) continue;
                const float w = (a ? 0.5f : 1.f) * (b ? 0.5f : 1.f) * (c ? 0.5f : 1.f);
                const long m = pl * i + (long)(nz + 1) * j + k;
                s[0] += w * res[3 * m];
                s[1] += w * res[3 * m + 1];
                s[2] += w * res[3 * m + 2];
            }
    const uint8_t f = cfix[n];
    for (int d = 0; d < 3; d++) rc[3 * n + d] = ((f >> d) & 1) ? 0.f : s[d];
}

__global__ void __launch_bounds__(256) k_mg3_restrict(int cnx, int cny, int cnz, const float* __restrict__ res,
                                                      const uint8_t* __restrict__ cfix, float* __restrict__ rc,
                                                      const int* __restrict__ done) {
    if (done && *done) return;
    const long cnn = (long)(cnx + 1) * (cny + 1) * (cnz + 1);
    const BlockRange xr = xcd_block_range(cnn);  // the 27 fine nodes through one L2
    for (long n = xr.begin + threadIdx.x; n < xr.end; n += blockDim.x) mg3_restrict_at(n, cnx, cny, cnz, res, cfix, rc);
}

// Galerkin coarse element matrices of levels 2 and up from the level above's,
// one thread per (coarse element, row): row 3q + d of Kc is
// sum_a sum_k w_a[k][q] (row 3k + d of K_a) P_a (level 1: k_mg3_coarsen0).
__global__ void __launch_bounds__(256) k_mg3_coarsen(int cnx, int cny, int cnz, const double* __restrict__ Kf,
                                                     double* __restrict__ Kc, float* __restrict__ Kc32) {
    const long nce = (long)cnx * cny * cnz;
    const int ny = 2 * cny, nz = 2 * cnz;
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t >= nce * 24) return;
    const long ce = t / 24;
    const int row = (int)(t - ce * 24), q = row / 3, d = row - 3 * (row / 3);
    const long cpl = (long)cny * cnz;
    const int CI = (int)(ce / cpl);
    const long rem = ce - (long)CI * cpl;
    const int CJ = (int)(rem / cnz), CK = (int)(rem - (long)CJ * cnz);
    // No array is indexed by a runtime value (that put them in scratch): the
    // trilinear weights are evaluated where they are used, and the loops over
    // the output columns are unrolled.
    double out[24];
#pragma unroll
    for (int c = 0; c < 24; c++) out[c] = 0.0;
    int qx, qy, qz;
    mg3_lxyz(q, qx, qy, qz);
    // weight of coarse node (bx, by, bz) at the child node at (x, y, z) of the coarse element
    auto tri = [](int bx, int by, int bz, double x, double y, double z) {
        return (bx ? x : 1 - x) * (by ? y : 1 - y) * (bz ? z : 1 - z);
    };
    // the children loop is unrolled so that the trilinear weights of the
    // columns (w2) are constants: the products with a zero weight (58% of
    // them) drop out at compile time
#pragma unroll
    for (int ch = 0; ch < 8; ch++) {
        int a0, a1, a2;
        mg3_lxyz(ch, a0, a1, a2);
        const int fi = 2 * CI + a0, fj = 2 * CJ + a1, fk = 2 * CK + a2;
        const long fe = ((long)ny * nz) * fi + (long)nz * fj + fk;
#pragma unroll 1
        for (int k = 0; k < 8; k++) {
            int lx, ly, lz;
            mg3_lxyz(k, lx, ly, lz);
            const double wq = tri(qx, qy, qz, 0.5 * (a0 + lx), 0.5 * (a1 + ly), 0.5 * (a2 + lz));
            if (wq == 0.0) continue;
            const int rr = 3 * k + d;
#pragma unroll
            for (int k2 = 0; k2 < 8; k2++) {
                int mx, my, mz;
                mg3_lxyz(k2, mx, my, mz);
                const double x2 = 0.5 * (a0 + mx), y2 = 0.5 * (a1 + my), z2 = 0.5 * (a2 + mz);
                double w2[8];
#pragma unroll
                for (int q2 = 0; q2 < 8; q2++) {
                    int bx, by, bz;
                    mg3_lxyz(q2, bx, by, bz);
                    w2[q2] = tri(bx, by, bz, x2, y2, z2);
                }
#pragma unroll
                for (int d2 = 0; d2 < 3; d2++) {
                    const double wk = wq * Kf[fe * 576 + rr * 24 + 3 * k2 + d2];
#pragma unroll
                    for (int q2 = 0; q2 < 8; q2++)
                        if (w2[q2] != 0.0) out[3 * q2 + d2] += wk * w2[q2];
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 24; c++) {
        Kc[ce * 576 + row * 24 + c] = out[c];
        Kc32[ce * 576 + row * 24 + c] = (float)out[c];
    }
}

// Weight of coarse corner q at corner k of child ch (all in reference order).
__device__ inline double mg3_child_weight(int q, int ch, int k) {
    int qx, qy, qz, ax, ay, az, kx, ky, kz;
    mg3_lxyz(q, qx, qy, qz);
    mg3_lxyz(ch, ax, ay, az);
    mg3_lxyz(k, kx, ky, kz);
    const double x = 0.5 * (ax + kx), y = 0.5 * (ay + ky), z = 0.5 * (az + kz);
    return (qx ? x : 1 - x) * (qy ? y : 1 - y) * (qz ? z : 1 - z);
}

// M[ch] = P_ch^T K0 P_ch: what child ch adds to a coarse element's matrix per
// unit modulus where none of its nodes is fixed.  One thread per entry.
__global__ void __launch_bounds__(256) k_mg3_child_matrices(const double* __restrict__ K0, double* __restrict__ M) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= 8 * 576) return;
    const int ch = t / 576, row = (t % 576) / 24, col = t % 24;
    double s = 0.0;
    for (int k = 0; k < 8; k++) {
        const double w = mg3_child_weight(row / 3, ch, k);
        if (w == 0.0) continue;
        for (int k2 = 0; k2 < 8; k2++)
            s += w * K0[(3 * k + row % 3) * 24 + 3 * k2 + col % 3] * mg3_child_weight(col / 3, ch, k2);
    }
    M[t] = s;
}

// Level 1 from the moduli: Kc = sum_ch E_ch M[ch], three entries per thread
// with their eight children's values in registers, entries contiguous over the
// lanes.  128x64x64: 307 us (453 MB written, 1.5 TB/s: the loads of the moduli
// and fixity bits of one element at a time bound it), against 2.25 ms with the
// products with K0 formed again in every element.  An element with a fixed node
// in it takes those products, masked.
constexpr int kMg3C0Threads = 192;
__global__ void __launch_bounds__(kMg3C0Threads) k_mg3_coarsen0(int cnx, int cny, int cnz, const double* __restrict__ E,
                                                                const double* __restrict__ K0,
                                                                const double* __restrict__ M,
                                                                const uint8_t* __restrict__ fix,
                                                                double* __restrict__ Kc, float* __restrict__ Kc32) {
    const long nce = (long)cnx * cny * cnz;
    const int ny = 2 * cny, nz = 2 * cnz, t = threadIdx.x, lane = t & 63;
    const long pl = (long)(ny + 1) * (nz + 1), epl = (long)ny * nz;
    double m[3][8];
#pragma unroll
    for (int s = 0; s < 3; s++)
#pragma unroll
        for (int ch = 0; ch < 8; ch++) m[s][ch] = M[ch * 576 + t + kMg3C0Threads * s];
    for (long ce = blockIdx.x; ce < nce; ce += gridDim.x) {
        const int CI = (int)(ce / ((long)cny * cnz));
        const int rem = (int)(ce - (long)CI * cny * cnz), CJ = rem / cnz, CK = rem - CJ * cnz;
        const long n0 = pl * (2 * CI) + (long)(nz + 1) * (2 * CJ) + 2 * CK;
        const long f0 = epl * (2 * CI) + (long)nz * (2 * CJ) + 2 * CK;
        int fx = 0;  // lanes 0 .. 26: the element's fine nodes
        if (lane < 27) fx = fix[n0 + pl * (lane / 9) + (long)(nz + 1) * (lane / 3 % 3) + lane % 3];
        double e[8];
#pragma unroll
        for (int ch = 0; ch < 8; ch++) {
            int a0, a1, a2;
            mg3_lxyz(ch, a0, a1, a2);
            e[ch] = E[f0 + epl * a0 + (long)nz * a1 + a2];
        }
        const bool fixed = __ballot(fx != 0) != 0;  // the same in every wave
        double out[3];
#pragma unroll
        for (int s = 0; s < 3; s++) {
            out[s] = 0.0;
#pragma unroll
            for (int ch = 0; ch < 8; ch++) out[s] += e[ch] * m[s][ch];
        }
        if (fixed) {
#pragma unroll 1
            for (int s = 0; s < 3; s++) {
                const int q = t + kMg3C0Threads * s, row = q / 24, col = q % 24;
                double sum = 0.0;
#pragma unroll 1
                for (int ch = 0; ch < 8; ch++) {
                    int a0, a1, a2;
                    mg3_lxyz(ch, a0, a1, a2);
                    const double ec = E[f0 + epl * a0 + (long)nz * a1 + a2];
#pragma unroll 1
                    for (int k = 0; k < 8; k++) {
                        int x, y, z;
                        mg3_lxyz(k, x, y, z);
                        const double w = mg3_child_weight(row / 3, ch, k);
                        if (w == 0.0 ||
                            ((fix[n0 + pl * (a0 + x) + (long)(nz + 1) * (a1 + y) + a2 + z] >> (row % 3)) & 1))
                            continue;
#pragma unroll 1
                        for (int k2 = 0; k2 < 8; k2++) {
                            mg3_lxyz(k2, x, y, z);
                            if ((fix[n0 + pl * (a0 + x) + (long)(nz + 1) * (a1 + y) + a2 + z] >> (col % 3)) & 1) continue;
                            sum += ec * w * K0[(3 * k + row % 3) * 24 + 3 * k2 + col % 3] *
                                   mg3_child_weight(col / 3, ch, k2);
                        }
                    }
                }
                if (s == 0) out[0] = sum;
                else if (s == 1) out[1] = sum;
                else out[2] = sum;
            }
        }
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const long o = ce * 576 + t + kMg3C0Threads * s;
            Kc[o] = out[s];
            Kc32[o] = (float)out[s];
        }
    }
}

// diagonal and fixity of a coarse level (a DOF without stiffness is fixed)
__global__ void __launch_bounds__(256) k_mg3_diag_full(int nx, int ny, int nz, const double* __restrict__ Ke,
                                                       float* __restrict__ D, uint8_t* __restrict__ fix) {
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    const long pl = (long)(ny + 1) * (nz + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        const int i = (int)(n / pl);
        const long rem = n - (long)i * pl;
        const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
        double dg[3] = {0.0, 0.0, 0.0};
        for (int ea = 0; ea < 2; ea++)
            for (int eb = 0; eb < 2; eb++)
                for (int ec = 0; ec < 2; ec++) {
                    const int ei = i - 1 + ea, ej = j - 1 + eb, ek = k - 1 + ec;
                    if (ei < 0 || ei >= nx || ej < 0 || ej >= ny || ek < 0 || ek >= nz) continue;
                    const long e = ((long)ny * nz) * ei + (long)nz * ej + ek;
                    const int di = i - ei, dj = j - ej, dk = k - ek;
                    const int me = 4 * dk + (dj == 0 ? di : 3 - di);
                    for (int d = 0; d < 3; d++) dg[d] += Ke[e * 576 + (3 * me + d) * 24 + 3 * me + d];
                }
        uint8_t f = 0;
        for (int d = 0; d < 3; d++) {
            if (!(dg[d] > 0.0)) f |= (uint8_t)(1u << d);
            D[3 * n + d] = ((f >> d) & 1) ? 1.f : (float)dg[d];
        }
        fix[n] = f;
    }
}

// level-0 diagonal in FP32 from E and K0 (fixed DOFs: 1)
__global__ void __launch_bounds__(256) k_mg3_diag0(int nx, int ny, int nz, const double* __restrict__ E,
                                                   const double* __restrict__ K0, const uint8_t* __restrict__ fix,
                                                   float* __restrict__ D) {
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    const long pl = (long)(ny + 1) * (nz + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        const int i = (int)(n / pl);
        const long rem = n - (long)i * pl;
        const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
        double dg[3] = {0.0, 0.0, 0.0};
        for (int ea = 0; ea < 2; ea++)
            for (int eb = 0; eb < 2; eb++)
                for (int ec = 0; ec < 2; ec++) {
                    const int ei = i - 1 + ea, ej = j - 1 + eb, ek = k - 1 + ec;
                    if (ei < 0 || ei >= nx || ej < 0 || ej >= ny || ek < 0 || ek >= nz) continue;
                    const double ee = E[((long)ny * nz) * ei + (long)nz * ej + ek];
                    const int di = i - ei, dj = j - ej, dk = k - ek;
                    const int me = 4 * dk + (dj == 0 ? di : 3 - di);
                    for (int d = 0; d < 3; d++) dg[d] += ee * K0[(3 * me + d) * 24 + 3 * me + d];
                }
        const uint8_t f = fix[n];
        for (int d = 0; d < 3; d++) D[3 * n + d] = ((f >> d) & 1) ? 1.f : (float)dg[d];
    }
}

// dense free-DOF block of the coarsest level (3 DOFs per node)
__global__ void __launch_bounds__(256) k_mg3_dense(int nx, int ny, int nz, const double* __restrict__ Ke,
                                                   const int* __restrict__ dof, int nf, double* __restrict__ A) {
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t >= (long)nf * nf) return;
    const int a = (int)(t / nf), b = (int)(t - (long)a * nf);
    const int na = dof[a] / 3, da = dof[a] - 3 * na, nb = dof[b] / 3, db = dof[b] - 3 * nb;
    const int pl = (ny + 1) * (nz + 1);
    const int ia = na / pl, ja = (na - ia * pl) / (nz + 1), ka = na - ia * pl - ja * (nz + 1);
    const int ib = nb / pl, jb = (nb - ib * pl) / (nz + 1), kb = nb - ib * pl - jb * (nz + 1);
    double s = 0.0;
    for (int ei = ia - 1; ei <= ia; ei++)
        for (int ej = ja - 1; ej <= ja; ej++)
            for (int ek = ka - 1; ek <= ka; ek++) {
                if (ei < 0 || ei >= nx || ej < 0 || ej >= ny || ek < 0 || ek >= nz) continue;
                int qa = -1, qb = -1;
                for (int q = 0; q < 8; q++) {
                    int qx, qy, qz;
                    mg3_lxyz(q, qx, qy, qz);
                    if (ei + qx == ia && ej + qy == ja && ek + qz == ka) qa = q;
                    if (ei + qx == ib && ej + qy == jb && ek + qz == kb) qb = q;
                }
                if (qa < 0 || qb < 0) continue;
                s += Ke[(((long)ny * nz) * ei + (long)nz * ej + ek) * 576 + (3 * qa + da) * 24 + 3 * qb + db];
            }
    A[t] = s;
}

// level-0 element matrices in FP64 (E_e K0), for a grid that is its own coarsest level
__global__ void __launch_bounds__(256) k_mg3_ke0_full(long ne, const double* __restrict__ E,
                                                      const double* __restrict__ K0, double* __restrict__ Ke) {
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t < ne * 576) Ke[t] = E[t / 576] * K0[t % 576];
}

// ------------------------------------------------------- the small levels ----
// The hex8 V-cycle below a level of at most 1024 nodes in one workgroup of
// 1024 threads (one node per thread), as k_mg_tail does for quad4: the
// levels' vectors and fixities in LDS, the element matrices read from global
// memory, each level's phases (update, residual, restriction; prolongation,
// residual sweeps) separated by barriers; the first level's r restricted
// here from the residual of the level above, its x back to its global
// buffer.  The residual in the element form (elem: y_e = K_e x_e
// into LDS by thread (e, q), then each node's gather) or the node form.
enum { kM3R, kM3X, kM3X2, kM3D, kM3Res, kM3Fix, kM3Ye, kM3Slots };

// Places level (nx, ny, nz)'s arrays in the pool from float offset off (the
// coarsest level keeps r, x and its fixity; the others also x2, D, res and,
// in the element form, y) and returns the next free offset.
inline long mg3_tail_place(int nx, int ny, int nz, bool coarsest, bool elem, long off, int* lo) {
    const long nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    for (int s = 0; s < kM3Slots; s++) lo[s] = -1;
    auto put = [&](int s, long n) {
        lo[s] = (int)off;
        off += (n + 3) & ~3L;
    };
    put(kM3R, 3 * nn);
    put(kM3X, 3 * nn);
    if (!coarsest) {
        put(kM3X2, 3 * nn);
        put(kM3D, 3 * nn);
        put(kM3Res, 3 * nn);
    }
    put(kM3Fix, (nn + 3) / 4);
    if (!coarsest && elem) put(kM3Ye, 24L * nx * ny * nz);
    return off;
}

struct Mg3TailLevel {
    int nx, ny, nz;
    const float* Ke;  // FP32 element matrices (a coarse level)
    const float* D;
    const uint8_t* fix;
    float* x;          // global: the first level's x out
    int lo[kM3Slots];  // the level's arrays in the pool (mg3_tail_place)
};
struct Mg3Tail {
    int nlev;  // levels; the last is the coarsest
    Mg3TailLevel L[kMgTailMax];
    int nf;
    const double* Ainv;
    const int* dof;
    int nu;
    float omega;
    int elem;           // residual in the element form
    const float* pres;  // the residual of the level above the first, restricted into its r here
};

__global__ void __launch_bounds__(1024) k_mg3_tail(Mg3Tail T, const int* __restrict__ done) {
    if (done && *done) return;
    __shared__ float4 pool4[kMgTailPool / 4];
    __shared__ float rf[kMgLdsDense];
    __shared__ double part[kMgTailNodes];  // the coarsest solve's partial sums
    float* const pool = reinterpret_cast<float*>(pool4);
    const int tid = threadIdx.x, nth = (int)blockDim.x;
    const Mg3TailLevel* L = T.L;
    const int c = T.nlev - 1;
    auto sl = [&](int k, int s) { return pool + L[k].lo[s]; };
    auto sfix = [&](int k) { return reinterpret_cast<uint8_t*>(pool + L[k].lo[kM3Fix]); };
    auto nodes = [&](int k) { return (long)(L[k].nx + 1) * (L[k].ny + 1) * (L[k].nz + 1); };
    // the coarsest solve's terms of the inverse and this thread's DOF, loaded
    // with the staging below
    const int nf = T.nf, ng = nth / nf;
    const int ca = tid % nf, cg = tid / nf;
    double ainv[kMgTailTerms];
#pragma unroll
    for (int q = 0; q < kMgTailTerms; q++) {
        const int b = cg + q * ng;
        ainv[q] = (cg < ng && b < nf) ? T.Ainv[(long)b * nf + ca] : 0.0;
    }
    const int mydof = tid < nf ? T.dof[tid] : 0;
    // staging: the first level's r (P^T of the residual of the level above,
    // formed here); every level's fixity and D
#pragma unroll 1
    for (int k = 0; k <= c; k++) {
        const Mg3TailLevel& a = L[k];
        const long nn = nodes(k);
        if (k == 0)
            for (long n = tid; n < nn; n += nth) mg3_restrict_at(n, a.nx, a.ny, a.nz, T.pres, a.fix, sl(0, kM3R));
        if (k < c) {
            float* d = sl(k, kM3D);
            for (long q = tid; q < 3 * nn; q += nth) d[q] = a.D[q];
        }
        uint8_t* f = sfix(k);
        for (long q = tid; q < nn; q += nth) f[q] = a.fix[q];
    }
    __syncthreads();
    const bool pre_x2 = mg_pre_in_x2(T.nu);
    // rout = r - A xin, or with xout, xout = xin + omega D^-1 (r - A xin), on
    // level l, and a barrier
    auto residual = [&](int l, const float* xin, float* rout, float* xout) {
        const Mg3TailLevel& a = L[l];
        const float *r = sl(l, kM3R), *D = sl(l, kM3D);
        const uint8_t* fix = sfix(l);
        if (T.elem) {
            float* ye = sl(l, kM3Ye);
            const long ne = (long)a.nx * a.ny * a.nz;
            const long pl = (long)(a.ny + 1) * (a.nz + 1);
            for (long t = tid; t < 8 * ne; t += nth) {
                const long e = t >> 3;
                const int ei = (int)(e / ((long)a.ny * a.nz));
                const long rem = e - (long)ei * a.ny * a.nz;
                const int ej = (int)(rem / a.nz), ek = (int)(rem - (long)ej * a.nz);
                float xe[24];
#pragma unroll
                for (int p = 0; p < 8; p++) {
                    int px, py, pz;
                    mg3_lxyz(p, px, py, pz);
                    const long m = pl * (ei + px) + (long)(a.nz + 1) * (ej + py) + (ek + pz);
                    xe[3 * p] = xin[3 * m];
                    xe[3 * p + 1] = xin[3 * m + 1];
                    xe[3 * p + 2] = xin[3 * m + 2];
                }
                mg3_elem_rows(a.Ke, e, (int)(t & 7), xe, ye);
            }
            __syncthreads();
            if (tid < nodes(l)) mg3_gather_at(tid, a.nx, a.ny, a.nz, ye, D, fix, T.omega, r, xin, nullptr, rout, xout);
        } else {
            const Mg3KeFull ke{a.Ke};
            if (tid < nodes(l)) mg3_residual_at(tid, a.nx, a.ny, a.nz, ke, D, fix, T.omega, r, xin, rout, xout);
        }
        __syncthreads();
    };
    // down: pre-smoothing and restriction
#pragma unroll 1
    for (int l = 0; l < c; l++) {
        const long nn = nodes(l);
        const float *r = sl(l, kM3R), *D = sl(l, kM3D);
        const uint8_t* fix = sfix(l);
        float *x = sl(l, kM3X), *xo = sl(l, kM3X2), *res = sl(l, kM3Res);
        for (long t = tid; t < 3 * nn; t += nth) mg3_update_at(t, T.omega, nullptr, nullptr, r, D, fix, x);
        __syncthreads();
        residual(l, x, res, nullptr);
#pragma unroll 1
        for (int k = 1; k < T.nu; k++) {
            for (long t = tid; t < 3 * nn; t += nth) mg3_update_at(t, T.omega, x, res, r, D, fix, xo);
            __syncthreads();
            float* t0 = x; x = xo; xo = t0;
            residual(l, x, res, nullptr);
        }
        const Mg3TailLevel& b = L[l + 1];
        if (tid < nodes(l + 1)) mg3_restrict_at(tid, b.nx, b.ny, b.nz, res, sfix(l + 1), sl(l + 1, kM3R));
        __syncthreads();
    }
    // coarsest: x = Ainv r on the free DOFs
    {
        float* cx = sl(c, kM3X);
        const long nv = 3 * nodes(c);
        for (long q = tid; q < nv; q += nth) cx[q] = 0.f;
        if (tid < nf) rf[tid] = sl(c, kM3R)[mydof];
        __syncthreads();
        // x_a = sum_b Ainv[b][a] r_b: group g of threads takes b = g, g + ng,
        // ..., the groups' partial sums then added in group order
        if (cg < ng) {
            double sum = 0.0;
#pragma unroll
            for (int q = 0; q < kMgTailTerms; q++) {
                const int b = cg + q * ng;
                if (b < nf) sum += ainv[q] * (double)rf[b];
            }
            part[cg * nf + ca] = sum;
        }
        __syncthreads();
        if (tid < nf) {
            double sum = 0.0;
            for (int q = 0; q < ng; q++) sum += part[q * nf + tid];
            cx[mydof] = (float)sum;
        }
        __syncthreads();
    }
    // up: prolongation and post-smoothing sweeps
    float* xc = sl(c, kM3X);
#pragma unroll 1
    for (int l = c - 1; l >= 0; l--) {
        const Mg3TailLevel& a = L[l];
        const long nn = nodes(l);
        const uint8_t* fix = sfix(l);
        float *x = pre_x2 ? sl(l, kM3X2) : sl(l, kM3X), *xo = pre_x2 ? sl(l, kM3X) : sl(l, kM3X2);
        if (tid < nn) mg3_prolong_at(tid, a.nx, a.ny, a.nz, x, xc, fix, xo);
        __syncthreads();
        { float* t0 = x; x = xo; xo = t0; }
#pragma unroll 1
        for (int k = 0; k < T.nu; k++) {
            residual(l, x, nullptr, xo);
            float* t0 = x; x = xo; xo = t0;
        }
        xc = x;
    }
    // the first level's x to its global buffer
    {
        float* out = L[0].x;
        const long nv = 3 * nodes(0);
        for (long q = tid; q < nv; q += nth) out[q] = xc[q];
    }
}

}  // namespace pf
