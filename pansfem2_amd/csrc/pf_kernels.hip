// HIP kernels (gfx950) of the SIMP loop on structured quad4 / hex8 grids.
//
// The file is compiled without floating-point contraction: every a*b + c
// rounds twice, as the reference's x86-64 g++ build (no FMA) does, so the
// check-path kernels (element matrices, CSR values, CSR product, diagonal,
// filter, OC step) reproduce the reference's bits.  The matrix-free operator
// and the PCG vector updates, which no result is compared with bit for bit,
// re-enable contraction in their own bodies (half the FP64 instructions).
#pragma clang fp contract(off)

#include "pf_device.h"
#include "pf_internal.h"

namespace pf {

// ===================================================== grid geometry ======
struct Grid2 {
    int nx, ny;
    __device__ int nnode() const { return (nx + 1) * (ny + 1); }
};

// ============================================================ moduli =====
__global__ void k_E_from_rho(long ne, const double* __restrict__ rho, double E1, double E0, double p,
                             double* __restrict__ E, float* __restrict__ Ef) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        double rp = simp_pow(rho[e], p);
        double v = E1 * rp + E0 * (1.0 - rp);  // sample_optimize_density_oc.cpp:123
        E[e] = v;
        Ef[e] = (float)v;
    }
}

// ====================================================== nodal <-> free ====
__global__ void k_free_to_nodal(int N, const int32_t* __restrict__ g2n, const double* __restrict__ xf,
                                double* __restrict__ xn) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < N) xn[g2n[g]] = xf[g];
}

__global__ void k_nodal_to_free(int N, const int32_t* __restrict__ g2n, const double* __restrict__ xn,
                                double* __restrict__ xf) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < N) xf[g] = xn[g2n[g]];
}

template <class T>
__global__ void k_fill(long n, T* __restrict__ p, T v) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

template <class A, class B>
__global__ void k_convert(long n, const A* __restrict__ a, B* __restrict__ b) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = (B)a[i];
}

// ===================================================== 2D EbE operator ====
// Node (i,j) touches elements (i-1,j-1) [as TR, local 2], (i-1,j) [BR, 1],
// (i,j-1) [TL, 3], (i,j) [BL, 0]; contributions are summed in that order,
// which is ascending element id, the order Assembling adds them in.
//
// v[a][b] holds the nodal pair of node (i+a-1, j+b-1).
template <class T>
struct alignas(2 * sizeof(T)) Vec2 { T x, y; };

template <class T, class KP>
__device__ inline void elem_rows_q4(KP K0, int loc, const Vec2<T> n0, const Vec2<T> n1,
                                    const Vec2<T> n2, const Vec2<T> n3, T& ox, T& oy) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    // rows 2*loc, 2*loc+1 of K0 times the element vector (BL, BR, TR, TL)
    const KP r0 = K0 + (2 * loc) * 8;
    const KP r1 = r0 + 8;
    T a = 0, b = 0;
    a += r0[0] * n0.x; a += r0[1] * n0.y; a += r0[2] * n1.x; a += r0[3] * n1.y;
    a += r0[4] * n2.x; a += r0[5] * n2.y; a += r0[6] * n3.x; a += r0[7] * n3.y;
    b += r1[0] * n0.x; b += r1[1] * n0.y; b += r1[2] * n1.x; b += r1[3] * n1.y;
    b += r1[4] * n2.x; b += r1[5] * n2.y; b += r1[6] * n3.x; b += r1[7] * n3.y;
    ox = a;
    oy = b;
}

template <class T>
__device__ inline void apply_q4_node(int nx, int ny, int i, int j, const Vec2<T> (&v)[3][3], const T* __restrict__ E,
                                     const T* __restrict__ K0, T& yx, T& yy) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    T ax = 0, ay = 0, ex, ey;
    if (i >= 1 && j >= 1) {  // element (i-1, j-1): this node is TR
        T Ee = E[(long)ny * (i - 1) + (j - 1)];
        elem_rows_q4<T>(K0, 2, v[0][0], v[1][0], v[1][1], v[0][1], ex, ey);
        ax += Ee * ex; ay += Ee * ey;
    }
    if (i >= 1 && j < ny) {  // element (i-1, j): BR
        T Ee = E[(long)ny * (i - 1) + j];
        elem_rows_q4<T>(K0, 1, v[0][1], v[1][1], v[1][2], v[0][2], ex, ey);
        ax += Ee * ex; ay += Ee * ey;
    }
    if (i < nx && j >= 1) {  // element (i, j-1): TL
        T Ee = E[(long)ny * i + (j - 1)];
        elem_rows_q4<T>(K0, 3, v[1][0], v[2][0], v[2][1], v[1][1], ex, ey);
        ax += Ee * ex; ay += Ee * ey;
    }
    if (i < nx && j < ny) {  // element (i, j): BL
        T Ee = E[(long)ny * i + j];
        elem_rows_q4<T>(K0, 0, v[1][1], v[2][1], v[2][2], v[1][2], ex, ey);
        ax += Ee * ex; ay += Ee * ey;
    }
    yx = ax;
    yy = ay;
}

// One node's pair as a single 16-byte (FP64) or 8-byte (FP32) access.
template <class T>
__device__ inline Vec2<T> load2(const T* __restrict__ a, long n) {
    return reinterpret_cast<const Vec2<T>*>(a)[n];
}

template <class T>
__device__ inline void store2(T* __restrict__ a, long n, Vec2<T> v) {
    reinterpret_cast<Vec2<T>*>(a)[n] = v;
}

// y = K x (nodal vectors), fixed DOFs of y set to zero when mask_fixed.
template <class T>
__global__ void __launch_bounds__(256) k_apply_q4(int nx, int ny, const T* __restrict__ x, T* __restrict__ y,
                                                  const T* __restrict__ E, const T* __restrict__ K0,
                                                  const uint8_t* __restrict__ fix, int mask_fixed) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        Vec2<T> v[3][3];
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                int ii = i + a - 1, jj = j + b - 1;
                if (ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) v[a][b] = load2(x, (long)(ny + 1) * ii + jj);
                else v[a][b] = Vec2<T>{0, 0};
            }
        T yx, yy;
        apply_q4_node(nx, ny, i, j, v, E, K0, yx, yy);
        if (mask_fixed) {
            uint8_t f = fix[n];
            if (f & 1) yx = 0;
            if (f & 2) yy = 0;
        }
        y[2 * n] = yx;
        y[2 * n + 1] = yy;
    }
}

// Jacobi diagonal of the EbE operator: sum of E_e K0(a,a) over the elements
// of the node in ascending element id; fixed DOFs get 1.
template <class T>
__global__ void k_diag_q4(int nx, int ny, const T* __restrict__ E, const T* __restrict__ K0,
                          const uint8_t* __restrict__ fix, T* __restrict__ D) {
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        T dx = 0, dy = 0;
        if (i >= 1 && j >= 1) { T e = E[(long)ny * (i - 1) + j - 1]; dx += e * K0[4 * 8 + 4]; dy += e * K0[5 * 8 + 5]; }
        if (i >= 1 && j < ny) { T e = E[(long)ny * (i - 1) + j]; dx += e * K0[2 * 8 + 2]; dy += e * K0[3 * 8 + 3]; }
        if (i < nx && j >= 1) { T e = E[(long)ny * i + j - 1]; dx += e * K0[6 * 8 + 6]; dy += e * K0[7 * 8 + 7]; }
        if (i < nx && j < ny) { T e = E[(long)ny * i + j]; dx += e * K0[0]; dy += e * K0[1 * 8 + 1]; }
        uint8_t f = fix[n];
        D[2 * n] = (f & 1) ? (T)1 : dx;
        D[2 * n + 1] = (f & 2) ? (T)1 : dy;
    }
}

// =============================================================== PCG =====
// Jacobi-PCG of ScalingCG (CG.h:419-453) as two launches per iteration.
//   K1(k): beta from K2(k-1)'s partials (k > 0; convergence is tested first,
//          as CG.h:443-447 does after iteration k-1), p = beta p + z fused
//          into the operator gather, q = K p, partial p.q.
//   K2(k): alpha = zr / p.q from K1's partials; x += alpha p; r -= alpha q;
//          z = r ./ D; partials z.r and r.r.
// Scalars that a later launch needs are written by workgroup 0 into slot
// k&1, so no workgroup reads a value the same launch is writing.
struct PcgDev {
    double zr[2];
    double bnorm;
    double pq, alpha, beta, rnorm;
    int iterations, status, done, pad;
    double g[2], a[2];  // single-reduction form: gamma = r.u and alpha of the last two steps
};

// beta for K1(k) from the sums (z.r, r.r) of K2(k-1) (init: (z.r, b.b)).
__device__ inline void pcg_head_sums(int k, const double (&v)[2], PcgDev* __restrict__ S, double eps, double& beta,
                                     bool& stop) {
    stop = false;
    if (k == 0) {
        beta = 0.0;
        if (threadIdx.x == 0 && blockIdx.x == 0) {
            S->zr[0] = v[0];
            S->bnorm = sqrt(v[1]);
            S->beta = 0.0;
        }
        return;
    }
    double bnorm = S->bnorm;
    double zr_prev = S->zr[(k - 1) & 1];
    double rnorm = sqrt(v[1]);
    beta = v[0] / zr_prev;
    if (rnorm < eps * bnorm) {
        stop = true;
        if (threadIdx.x == 0 && blockIdx.x == 0) {
            S->rnorm = rnorm;
            S->iterations = k;
            S->status = 1;
            S->done = 1;
        }
        return;
    }
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        S->zr[k & 1] = v[0];
        S->beta = beta;
        S->rnorm = rnorm;
    }
}

__device__ inline void pcg_head(int k, const double* __restrict__ partB, int nbB, PcgDev* __restrict__ S, double eps,
                                double* lds, double& beta, bool& stop) {
    double v[2];
    reduce_partials<2>(partB, nbB, lds, v);
    pcg_head_sums(k, v, S, eps, beta, stop);
}

template <class T>
__global__ void __launch_bounds__(256) k_pcg_k1_q4(int nx, int ny, int k, const T* __restrict__ pold,
                                                   const T* __restrict__ z, T* __restrict__ pnew, T* __restrict__ q,
                                                   const T* __restrict__ E, const T* __restrict__ K0,
                                                   const uint8_t* __restrict__ fix, const double* __restrict__ partB,
                                                   int nbB, double* __restrict__ partA, PcgDev* __restrict__ S,
                                                   double eps) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    __shared__ double lds[32];
    if (S->done) return;
    double beta;
    bool stop;
    pcg_head(k, partB, nbB, S, eps, lds, beta, stop);
    if (stop) return;
    const T tb = (T)beta;
    const long nn = (long)(nx + 1) * (ny + 1);
    double acc[1] = {0.0};
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        Vec2<T> v[3][3];
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                int ii = i + a - 1, jj = j + b - 1;
                if (ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
                    long m = (long)(ny + 1) * ii + jj;
                    Vec2<T> po = load2(pold, m), zz = load2(z, m);
                    v[a][b].x = tb * po.x + zz.x;  // xeaxpy: p = beta p + z (CG.h:42-49)
                    v[a][b].y = tb * po.y + zz.y;
                } else {
                    v[a][b] = Vec2<T>{0, 0};
                }
            }
        T yx, yy;
        apply_q4_node(nx, ny, i, j, v, E, K0, yx, yy);
        uint8_t f = fix[n];
        if (f & 1) yx = 0;
        if (f & 2) yy = 0;
        pnew[2 * n] = v[1][1].x;
        pnew[2 * n + 1] = v[1][1].y;
        q[2 * n] = yx;
        q[2 * n + 1] = yy;
        acc[0] += (double)v[1][1].x * (double)yx;
        acc[0] += (double)v[1][1].y * (double)yy;
    }
    store_partials<1>(acc, lds, partA);
}

// LDS-tiled K1 for quad4 grids.  A tile is TI x TJ nodes (TJ along j, the
// contiguous direction).  For each tile a workgroup stages p_new = beta p_old
// + z for the tile and a one-node halo in LDS (each halo value computed once)
// plus the moduli of the tile's elements; every thread then gathers its 3x3
// neighbourhood from LDS.  Global traffic per node: p_old, z, E read once
// (plus the halo), p_new and q written once.
//
// Launch shape: workgroups are dispatched round-robin over the 8 XCDs, so
// XCD x = blockIdx.x % 8 is given the contiguous tile range [x per, (x+1) per)
// (tile id = tile row * tilesJ + tile column): halo rows shared by
// neighbouring tiles then come through the same L2.  Within its range a
// workgroup takes every (gridDim.x / 8)-th tile and loads the next tile's
// halo and moduli into registers while it computes the current one.
// gridDim.x must be a multiple of 8.
template <class T, int TI, int TJ>
struct K1Tile {
    static constexpr int HALO = (TI + 2) * (TJ + 2);
    static constexpr int PER = (HALO + 255) / 256;
    static constexpr int ES = (TI + 1) * (TJ + 1);
    static constexpr int PE = (ES + 255) / 256;
    Vec2<T> po[PER], zz[PER];
    T ev[PE];

    __device__ inline void load(int t, int tilesJ, int nx, int ny, const T* __restrict__ pold,
                                const T* __restrict__ z, const T* __restrict__ E) {
        const int j0 = (t % tilesJ) * TJ, i0 = (t / tilesJ) * TI;
#pragma unroll
        for (int u = 0; u < PER; u++) {
            int h = threadIdx.x + u * 256;
            int a = h / (TJ + 2), b = h - a * (TJ + 2);
            int ii = i0 - 1 + a, jj = j0 - 1 + b;
            po[u] = Vec2<T>{0, 0};
            zz[u] = Vec2<T>{0, 0};
            if (h < HALO && ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
                long m = (long)(ny + 1) * ii + jj;
                po[u] = load2(pold, m);
                zz[u] = load2(z, m);
            }
        }
#pragma unroll
        for (int u = 0; u < PE; u++) {
            int h = threadIdx.x + u * 256;
            int a = h / (TJ + 1), b = h - a * (TJ + 1);
            int ei = i0 - 1 + a, ej = j0 - 1 + b;
            ev[u] = (h < ES && ei >= 0 && ei < nx && ej >= 0 && ej < ny) ? E[(long)ny * ei + ej] : (T)0;
        }
    }
};

template <class T, int TI, int TJ>
__global__ void __launch_bounds__(256) k_pcg_k1_q4_tile(int nx, int ny, int tilesJ, int ntiles, int k,
                                                        const T* __restrict__ pold, const T* __restrict__ z,
                                                        T* __restrict__ pnew, T* __restrict__ q,
                                                        const T* __restrict__ E, const T* __restrict__ K0,
                                                        const uint8_t* __restrict__ fix,
                                                        const double* __restrict__ partB, int nbB,
                                                        double* __restrict__ partA, PcgDev* __restrict__ S,
                                                        double eps) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    __shared__ double lds[32];
    __shared__ Vec2<T> sp[TI + 2][TJ + 2];
    __shared__ T se[TI + 1][TJ + 1];
    using Tile = K1Tile<T, TI, TJ>;
    const int xcd = blockIdx.x & 7, nb = gridDim.x >> 3;
    const int per = (ntiles + 7) >> 3;
    const int tend = min(ntiles, (xcd + 1) * per);
    int t = xcd * per + (blockIdx.x >> 3);
    // The first tile's loads, the previous launch's partials and the done
    // flag are all issued before the first wait.
    Tile cur;
    if (t < tend) cur.load(t, tilesJ, nx, ny, pold, z, E);
    PartRegs<2, 8> pr;
    load_partials(partB, nbB, pr);
    if (S->done) return;
    double beta;
    bool stop;
    {
        double v[2];
        sum_partials(pr, partB, nbB, lds, v);
        pcg_head_sums(k, v, S, eps, beta, stop);
    }
    if (stop) return;
    const T tb = (T)beta;
    double acc[1] = {0.0};
    for (; t < tend; t += nb) {
        const int j0 = (t % tilesJ) * TJ, i0 = (t / tilesJ) * TI;
        __syncthreads();  // the previous tile's LDS reads are done
#pragma unroll
        for (int u = 0; u < Tile::PER; u++) {
            int h = threadIdx.x + u * 256;
            if (h < Tile::HALO) {
                int a = h / (TJ + 2), b = h - a * (TJ + 2);
                Vec2<T> v;
                v.x = tb * cur.po[u].x + cur.zz[u].x;  // xeaxpy: p = beta p + z (CG.h:42-49)
                v.y = tb * cur.po[u].y + cur.zz[u].y;
                sp[a][b] = v;
            }
        }
#pragma unroll
        for (int u = 0; u < Tile::PE; u++) {
            int h = threadIdx.x + u * 256;
            if (h < Tile::ES) {
                int a = h / (TJ + 1), b = h - a * (TJ + 1);
                se[a][b] = cur.ev[u];
            }
        }
        __syncthreads();
        if (t + nb < tend) cur.load(t + nb, tilesJ, nx, ny, pold, z, E);  // in flight during the compute
        const int c = threadIdx.x % TJ;
        for (int r = threadIdx.x / TJ; r < TI; r += 256 / TJ) {
            const int i = i0 + r, j = j0 + c;
            if (i > nx || j > ny) continue;
            T ax = 0, ay = 0, ex, ey;
            if (i >= 1 && j >= 1) {  // element (i-1, j-1): this node is TR
                elem_rows_q4<T>(K0, 2, sp[r][c], sp[r + 1][c], sp[r + 1][c + 1], sp[r][c + 1], ex, ey);
                T Ee = se[r][c];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i >= 1 && j < ny) {  // element (i-1, j): BR
                elem_rows_q4<T>(K0, 1, sp[r][c + 1], sp[r + 1][c + 1], sp[r + 1][c + 2], sp[r][c + 2], ex, ey);
                T Ee = se[r][c + 1];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j >= 1) {  // element (i, j-1): TL
                elem_rows_q4<T>(K0, 3, sp[r + 1][c], sp[r + 2][c], sp[r + 2][c + 1], sp[r + 1][c + 1], ex, ey);
                T Ee = se[r + 1][c];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j < ny) {  // element (i, j): BL
                elem_rows_q4<T>(K0, 0, sp[r + 1][c + 1], sp[r + 2][c + 1], sp[r + 2][c + 2], sp[r + 1][c + 2], ex, ey);
                T Ee = se[r + 1][c + 1];
                ax += Ee * ex; ay += Ee * ey;
            }
            const long n = (long)(ny + 1) * i + j;
            uint8_t f = fix[n];
            if (f & 1) ax = 0;
            if (f & 2) ay = 0;
            Vec2<T> pv = sp[r + 1][c + 1];
            store2(pnew, n, pv);
            store2(q, n, Vec2<T>{ax, ay});
            acc[0] += (double)pv.x * (double)ax;
            acc[0] += (double)pv.y * (double)ay;
        }
    }
    store_partials<1>(acc, lds, partA);
}

// ------------------------------------------- single-reduction Jacobi-PCG ----
// Chronopoulos & Gear's form of preconditioned CG (J. Comput. Appl. Math. 25,
// 1989), one launch per iteration on quad4 grids.  With u = r ./ D, w = K u
// and s = K p carried as a vector, the recurrences
//   p_i = u_i + beta_i p_{i-1}      s_i = w_i + beta_i s_{i-1}
//   x_{i+1} = x_i + alpha_i p_i     r_{i+1} = r_i - alpha_i s_i
//   gamma_i = r_i.u_i, delta_i = u_i.w_i,
//   beta_i = gamma_i / gamma_{i-1}, alpha_i = gamma_i / (delta_i - beta_i gamma_i / alpha_{i-1})
// generate ScalingCG's iterates (CG.h:397-453) in exact arithmetic (p_i.K p_i
// = delta_i - beta_i gamma_i / alpha_{i-1}), and the three sums of an iterate
// (gamma, delta, r.r) come out of one reduction.
//
// Launch m (m >= 1) reduces the sums of iterate m-1, stops if |r_{m-1}| <
// eps |b| (iterations = m-1, as ScalingCG counts), else forms alpha_{m-1},
// beta_{m-1}, updates p, s, x, r, and computes w_m = K u_m with its sums.
// Launch 0 starts from r = b, x = 0 (alpha = beta = 0, nothing else read).
// A tile needs u_m on its one-node halo, so it recomputes s and r there from
// the previous launch's r, w, s (which neighbouring tiles are rewriting):
// r, w and s alternate between two buffers; p and x are touched only at a
// tile's own nodes and are updated in place.
template <class T>
struct Cg1Vecs {
    const T* rin;  // r_{m-1} (b at m = 0)
    const T* win;  // w_{m-1}
    const T* sin;  // s_{m-2}
    T* rout;       // r_m
    T* wout;       // w_m
    T* sout;       // s_{m-1}
    T* p;          // p_{m-2} -> p_{m-1}
    T* x;          // x_{m-2} -> x_m (even m only; see cg_x_even)
    const T* Dinv; // 1 / D
};

// x is read and written by the even launches only: launch m (even) forms
// x_m = (x_{m-2} + alpha_{m-1} p_{m-2}) + alpha_m p_{m-1} from the p it reads
// (p_{m-2}) and the p it forms (p_{m-1}), where alpha_{m-1} is the previous
// launch's alpha (S->a[m & 1]).  These are the two updates the odd and the
// even launch would each have made, in the same order, so x keeps its
// rounding; x does not enter the recurrences, so the iterates and the
// stopping test are unchanged.  An odd launch saves x's read and write (16 of
// the 88 bytes per DOF of the carried kernel, 16 of 56 of the recomputing
// one); when the last finished launch is odd, k_cg_x_fix adds its update.
__device__ inline bool cg_x_even(int m) { return (m & 1) == 0; }

// the head of launch m >= 1 from the sums v = (gamma, delta, r.r) of iterate m-1
__device__ inline void cg1_head(int m, const double (&v)[3], PcgDev* __restrict__ S, double eps, double& alpha,
                                double& beta, bool& stop) {
    stop = false;
    const bool w0 = threadIdx.x == 0 && blockIdx.x == 0;
    const double rnorm = sqrt(v[2]);
    if (m == 1) {
        beta = 0.0;
        alpha = v[0] / v[1];
        if (w0) S->bnorm = rnorm;
        if (!(v[0] > 0.0)) {  // b = 0: x = 0 is the solution
            stop = true;
            if (w0) {
                S->rnorm = rnorm;
                S->iterations = 0;
                S->status = 1;
                S->done = 1;
            }
            return;
        }
    } else {
        if (rnorm < eps * S->bnorm) {  // CG.h:445-449
            stop = true;
            if (w0) {
                S->rnorm = rnorm;
                S->iterations = m - 1;
                S->status = 1;
                S->done = 1;
            }
            return;
        }
        beta = v[0] / S->g[m & 1];                       // gamma_{m-2} (slot (m-2)&1)
        alpha = v[0] / (v[1] - beta * v[0] / S->a[m & 1]);  // alpha_{m-2}
    }
    if (w0) {
        S->g[(m - 1) & 1] = v[0];
        S->a[(m - 1) & 1] = alpha;
        S->rnorm = rnorm;
    }
}

// One tile of TI x TJ nodes per workgroup (tile (I, J) covers node rows
// [I TI, ...) and columns [J TJ, ...), clipped to the grid); TJ need not
// divide the workgroup: the own nodes are numbered q = r TJ + c and dealt
// out 256 at a time.
// Which tile a workgroup takes.  Full tiles (TI x TJ nodes inside the grid)
// and edge tiles (the last, partial tile row and column) are launched as two
// groups; edgeFirst puts the edge tiles (little work each) first, so that
// the full tiles that do not fit in the first wave of resident workgroups
// start as soon as the edge tiles are done.  Full tiles are given out
// XCD-contiguously (workgroup b runs on XCD b mod 8) as in k_pcg_k1_q4_tile;
// the edge group is padded to a multiple of 8 workgroups to keep that
// correspondence.
struct Cg1Tiles {
    int fullI, fullJ;    // full tile rows and columns
    int tilesI, tilesJ;  // all tile rows and columns
    int perF;            // full tiles per XCD (ceil(fullI fullJ / 8))
    int nEdgePad;        // edge tiles, rounded up to a multiple of 8
    int edgeFirst;
};

// tile (I, J) of workgroup b; false if b has no tile
__device__ inline bool cg1_tile(const Cg1Tiles& G, int b, int& I, int& J) {
    const int nFullPad = 8 * G.perF;
    int f = -1, e = -1;
    if (G.edgeFirst) {
        if (b < G.nEdgePad) e = b; else f = b - G.nEdgePad;
    } else {
        if (b < nFullPad) f = b; else e = b - nFullPad;
    }
    if (f >= 0) {
        const int id = (f & 7) * G.perF + (f >> 3);
        if (id >= G.fullI * G.fullJ) return false;
        I = id / G.fullJ;
        J = id - I * G.fullJ;
        return true;
    }
    const int ec = G.tilesJ - G.fullJ;  // edge columns (0 or 1)
    if (e < G.tilesI * ec) {
        I = e / ec;
        J = G.fullJ + (e - I * ec);
        return true;
    }
    e -= G.tilesI * ec;
    if (e < (G.tilesI - G.fullI) * G.fullJ) {
        I = G.fullI + e / G.fullJ;
        J = e - (I - G.fullI) * G.fullJ;
        return true;
    }
    return false;
}

template <class T, int TI, int TJ, bool XU>
__global__ void __launch_bounds__(256) k_cg1_q4_tile(int nx, int ny, Cg1Tiles G, int m,
                                                     Cg1Vecs<T> V, const T* __restrict__ E,
                                                     const T* __restrict__ K0, const uint8_t* __restrict__ fix,
                                                     const double* __restrict__ partIn, int nbIn,
                                                     double* __restrict__ partOut, PcgDev* __restrict__ S,
                                                     double eps) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    constexpr int PER = ((TI + 2) * (TJ + 2) + 255) / 256;  // staged entries per thread
    constexpr int PE = ((TI + 1) * (TJ + 1) + 255) / 256;   // element moduli per thread
    constexpr int OWN = (TI * TJ + 255) / 256;              // own nodes per thread
    __shared__ double lds[48];  // block_sum<3>: 16 per sum
    __shared__ Vec2<T> su[(TI + 2) * (TJ + 2)];  // u_m on the tile and its halo, row stride tj + 2
    __shared__ Vec2<T> uo[TI * TJ];              // u_{m-1} = r_{m-1} ./ D at the own nodes, stride tj
    __shared__ T se[(TI + 1) * (TJ + 1)];        // moduli of the tile's elements, stride tj + 1
    constexpr int ti = TI, tj = TJ;
    constexpr int halo = (ti + 2) * (tj + 2), es = (ti + 1) * (tj + 1), own = ti * tj;
    int TIr, TJr;
    const bool has = cg1_tile(G, blockIdx.x, TIr, TJr);
    const int i0 = TIr * TI, j0 = TJr * TJ;
    const bool prev = m > 0;  // launch 0 reads only r = b

    // staged entries: r, w, s, D; the tile's elements: E.  p and x (own
    // nodes only) are loaded later, in the operator phase's mapping, so they
    // are not live during the head.
    Vec2<T> rv[PER], wv[PER], sv[PER], dv[PER];
    T ev[PE];
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int h = threadIdx.x + u * 256;
            const int a = h / (tj + 2), b = h - a * (tj + 2);
            const int ii = i0 - 1 + a, jj = j0 - 1 + b;
            rv[u] = wv[u] = sv[u] = Vec2<T>{0, 0};
            dv[u] = Vec2<T>{1, 1};
            if (h < halo && ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
                const long n = (long)(ny + 1) * ii + jj;
                rv[u] = load2(V.rin, n);
                dv[u] = load2(V.Dinv, n);
                if (prev) {
                    wv[u] = load2(V.win, n);
                    sv[u] = load2(V.sin, n);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PE; u++) {
            const int h = threadIdx.x + u * 256;
            const int a = h / (tj + 1), b = h - a * (tj + 1);
            const int ei = i0 - 1 + a, ej = j0 - 1 + b;
            ev[u] = (h < es && ei >= 0 && ei < nx && ej >= 0 && ej < ny) ? E[(long)ny * ei + ej] : (T)0;
        }
    };
    // own nodes in the operator phase: thread t takes column t mod tj of rows
    // 2 (t / tj) and 2 (t / tj) + 1, so the two nodes share six of their nine
    // LDS neighbours and two of their four element moduli
    static_assert(OWN == 2 && TI * TJ == 512 && 256 % TJ == 0, "two vertically adjacent own nodes per thread");
    const int oc = threadIdx.x % tj, orow = 2 * (threadIdx.x / tj);
    constexpr bool xupd = XU;  // cg_x_even(m)
    auto load_px = [&](Vec2<T>(&pv)[OWN], Vec2<T>(&xv)[OWN]) {
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int r = orow + o, c = oc;
            const int q = r * tj + c;
            const int i = i0 + r, j = j0 + c;
            pv[o] = xv[o] = Vec2<T>{0, 0};
            if (prev && has && q < own && i <= nx && j <= ny) {
                const long n = (long)(ny + 1) * i + j;
                pv[o] = load2(V.p, n);
                if (xupd) xv[o] = load2(V.x, n);
            }
        }
    };
    // the first tile's loads, the previous launch's partials and the done
    // flag are issued before the first wait
    if (has) load();
    PartRegs<3, 5> pr;  // 1280 partials in registers, the rest read in sum_partials
    if (prev) load_partials(partIn, nbIn, pr);
    if (S->done) return;
    double alpha = 0.0, beta = 0.0;
    if (prev) {
        double v[3];
        bool stop;
        sum_partials(pr, partIn, nbIn, lds, v);
        cg1_head(m, v, S, eps, alpha, beta, stop);
        if (stop) return;
    }
    // the same in every lane: scalar registers
    const T ta = (T)wave_uniform(alpha), tb = (T)wave_uniform(beta);
    const T tap = (T)(m >= 2 && xupd ? S->a[m & 1] : 0.0);  // the previous launch's alpha
    constexpr int ss = tj + 2;  // LDS row strides
    double acc[3] = {0.0, 0.0, 0.0};  // r.u, u.w, r.r of iterate m
    if (has) {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int h = threadIdx.x + u * 256;
            if (h < halo) {
                const int a = h / (tj + 2), b = h - a * (tj + 2);
                const int ii = i0 - 1 + a, jj = j0 - 1 + b;
                Vec2<T> sn, rn, un;
                sn.x = wv[u].x + tb * sv[u].x;  // s = w + beta s
                sn.y = wv[u].y + tb * sv[u].y;
                rn.x = rv[u].x - ta * sn.x;     // r -= alpha s
                rn.y = rv[u].y - ta * sn.y;
                un.x = rn.x * dv[u].x;          // Scaling (CG.h:412), by 1/D
                un.y = rn.y * dv[u].y;
                su[h] = un;
                if (a >= 1 && a <= ti && b >= 1 && b <= tj && ii <= nx && jj <= ny) {
                    const long n = (long)(ny + 1) * ii + jj;
                    uo[(a - 1) * tj + (b - 1)] = Vec2<T>{rv[u].x * dv[u].x, rv[u].y * dv[u].y};
                    store2(V.sout, n, sn);
                    store2(V.rout, n, rn);
                    acc[0] += (double)rn.x * (double)un.x;
                    acc[0] += (double)rn.y * (double)un.y;
                    acc[2] += (double)rn.x * (double)rn.x;
                    acc[2] += (double)rn.y * (double)rn.y;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PE; u++) {
            const int h = threadIdx.x + u * 256;
            if (h < es) se[h] = ev[u];
        }
        // p_{m-2} and x_{m-1} of this thread's own nodes: in flight during the
        // operator (issued with the other loads they would cost occupancy)
        Vec2<T> pv[OWN], xv[OWN];
        load_px(pv, xv);
        __syncthreads();
        // LDS rows orow .. orow + 3 and columns oc .. oc + 2 (halo coordinates),
        // element moduli rows orow .. orow + 2 and columns oc .. oc + 1
        Vec2<T> v[4][3];
        T em[3][2];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) v[a][b] = su[(orow + a) * ss + oc + b];
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) em[a][b] = se[(orow + a) * (tj + 1) + oc + b];
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int r = orow + o, c = oc;
            const int q = r * tj + c;
            const int i = i0 + r, j = j0 + c;
            if (i > nx || j > ny) continue;
            T ax = 0, ay = 0, ex, ey;
            if (i >= 1 && j >= 1) {  // element (i-1, j-1): this node is TR
                elem_rows_q4<T>(K0, 2, v[o][0], v[o + 1][0], v[o + 1][1], v[o][1], ex, ey);
                const T Ee = em[o][0];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i >= 1 && j < ny) {  // element (i-1, j): BR
                elem_rows_q4<T>(K0, 1, v[o][1], v[o + 1][1], v[o + 1][2], v[o][2], ex, ey);
                const T Ee = em[o][1];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j >= 1) {  // element (i, j-1): TL
                elem_rows_q4<T>(K0, 3, v[o + 1][0], v[o + 2][0], v[o + 2][1], v[o + 1][1], ex, ey);
                const T Ee = em[o + 1][0];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j < ny) {  // element (i, j): BL
                elem_rows_q4<T>(K0, 0, v[o + 1][1], v[o + 2][1], v[o + 2][2], v[o + 1][2], ex, ey);
                const T Ee = em[o + 1][1];
                ax += Ee * ex; ay += Ee * ey;
            }
            const long n = (long)(ny + 1) * i + j;
            const uint8_t f = fix[n];
            if (f & 1) ax = 0;
            if (f & 2) ay = 0;
            const Vec2<T> un = v[o + 1][1];
            store2(V.wout, n, Vec2<T>{ax, ay});
            acc[1] += (double)un.x * (double)ax;
            acc[1] += (double)un.y * (double)ay;
            const Vec2<T> uold = uo[q];
            Vec2<T> pn, xh;
            xh.x = xv[o].x + tap * pv[o].x;  // x += alpha p for the previous launch (even launches)
            xh.y = xv[o].y + tap * pv[o].y;
            pn.x = uold.x + tb * pv[o].x;    // p = u + beta p
            pn.y = uold.y + tb * pv[o].y;
            store2(V.p, n, pn);
            if (xupd) {
                xh.x = xh.x + ta * pn.x;  // and for this one
                xh.y = xh.y + ta * pn.y;
                store2(V.x, n, xh);
            }
        }
    }
    store_partials<3>(acc, lds, partOut);
}

// The same recurrences with s = K p recomputed instead of carried, and w = K u
// used only for its sum.  Launch m forms p_{m-1} = u_{m-1} + beta p_{m-2}
// (u_{m-1} = r_{m-1} ./ D) on the tile and a two-node halo, s_{m-1} = K p_{m-1},
// r_m = r_{m-1} - alpha s_{m-1} and u_m = r_m ./ D on the tile and a one-node
// halo, then w_m = K u_m on the tile for delta_m = u_m.w_m.  x_m = x_{m-1} +
// alpha p_{m-1} at the own nodes.  r and p alternate between two buffers
// (neighbouring tiles read the previous launch's values on their halos); x is
// updated in place.  The Jacobi step multiplies by 1/D (precomputed per
// solve) where ScalingCG divides by D.  A launch reads r, 1/D, p, x and writes
// r, p, x: 56 bytes per free DOF in FP64, against 88 when s and w are carried.
// w_m is not masked at fixed DOFs: u_m is exactly 0 there, so delta_m gets
// nothing from them either way.
template <class T>
struct Cg2Vecs {
    const T* rin;  // r_{m-1} (b at m = 0)
    const T* pin;  // p_{m-2}
    T* rout;       // r_m
    T* pout;       // p_{m-1}
    T* x;          // x_{m-2} -> x_m (even m only; see cg_x_even)
    const T* Dinv; // 1 / D
};

template <class T, int TI, int TJ>
__global__ void __launch_bounds__(256) k_cg2_q4_tile(int nx, int ny, Cg1Tiles G, int m,
                                                     Cg2Vecs<T> V, const T* __restrict__ E,
                                                     const T* __restrict__ K0, const uint8_t* __restrict__ fix,
                                                     const double* __restrict__ partIn, int nbIn,
                                                     double* __restrict__ partOut, PcgDev* __restrict__ S,
                                                     double eps) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    constexpr int w1 = TJ + 2, w2 = TJ + 4, we = TJ + 3;  // row strides of R1, R2 and the elements
    constexpr int n1 = (TI + 2) * w1;   // R1: the tile and a one-node halo
    constexpr int n2 = (TI + 4) * w2;   // R2: the tile and a two-node halo
    constexpr int nel = (TI + 3) * we;  // the elements that touch R1
    constexpr int own = TI * TJ;
    constexpr int P1 = (n1 + 255) / 256, P2 = (n2 + 255) / 256;
    constexpr int PE = (nel + 255) / 256, OWN = (own + 255) / 256;
    __shared__ double lds[48];   // block_sum<3>: 16 per sum
    __shared__ Vec2<T> sp[n2];   // p_{m-1} on R2 (stride w2), then u_m on R1 (stride w1)
    __shared__ T se[nel];        // element (i0 - 2 + a, j0 - 2 + b) at a we + b
    int TIr, TJr;
    const bool has = cg1_tile(G, blockIdx.x, TIr, TJr);
    const int i0 = TIr * TI, j0 = TJr * TJ;
    const bool prev = m > 0;  // launch 0 reads only r = b
    // entry h of R2 -> its R2 coordinates (node (i0 - 2 + a2, j0 - 2 + b2)):
    // the R1 nodes first, row by row, so that a thread's R1 entries are among
    // its R2 entries; then the ring: top row, bottom row, left and right columns
    auto entry = [&](int h, int& a2, int& b2) {
        if (h < n1) {
            const int a = h / w1;
            a2 = a + 1;
            b2 = h - a * w1 + 1;
            return;
        }
        int e = h - n1;
        if (e < w2) { a2 = 0; b2 = e; return; }
        e -= w2;
        if (e < w2) { a2 = TI + 3; b2 = e; return; }
        e -= w2;
        if (e < TI + 2) { a2 = 1 + e; b2 = 0; return; }
        e -= TI + 2;
        a2 = 1 + e;
        b2 = w2 - 1;
    };
    Vec2<T> rv[P2], dv[P2], pv[P2];
    T ev[PE];
    if (has) {
#pragma unroll
        for (int u = 0; u < P2; u++) {
            const int h = threadIdx.x + u * 256;
            rv[u] = pv[u] = Vec2<T>{0, 0};
            dv[u] = Vec2<T>{1, 1};
            if (h < n2) {
                int a2, b2;
                entry(h, a2, b2);
                const int ii = i0 - 2 + a2, jj = j0 - 2 + b2;
                if (ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
                    const long n = (long)(ny + 1) * ii + jj;
                    rv[u] = load2(V.rin, n);
                    dv[u] = load2(V.Dinv, n);
                    if (prev) pv[u] = load2(V.pin, n);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PE; u++) {
            const int h = threadIdx.x + u * 256;
            const int a = h / we, b = h - a * we;
            const int ei = i0 - 2 + a, ej = j0 - 2 + b;
            ev[u] = (h < nel && ei >= 0 && ei < nx && ej >= 0 && ej < ny) ? E[(long)ny * ei + ej] : (T)0;
        }
    }
    PartRegs<3, 5> pr;
    if (prev) load_partials(partIn, nbIn, pr);
    if (S->done) return;
    double alpha = 0.0, beta = 0.0;
    if (prev) {
        double v[3];
        bool stop;
        sum_partials(pr, partIn, nbIn, lds, v);
        cg1_head(m, v, S, eps, alpha, beta, stop);
        if (stop) return;
    }
    const T ta = (T)wave_uniform(alpha), tb = (T)wave_uniform(beta);
    const bool xupd = cg_x_even(m);
    const T tap = (T)(m >= 2 && xupd ? S->a[m & 1] : 0.0);  // the previous launch's alpha
    double acc[3] = {0.0, 0.0, 0.0};  // r.u, u.w, r.r of iterate m
    if (has) {
#pragma unroll
        for (int u = 0; u < P2; u++) {
            const int h = threadIdx.x + u * 256;
            if (h < n2) {
                int a2, b2;
                entry(h, a2, b2);
                Vec2<T> pn;
                pn.x = rv[u].x * dv[u].x + tb * pv[u].x;  // p = u + beta p (CG.h:412, 440)
                pn.y = rv[u].y * dv[u].y + tb * pv[u].y;
                sp[a2 * w2 + b2] = pn;
            }
        }
#pragma unroll
        for (int u = 0; u < PE; u++) {
            const int h = threadIdx.x + u * 256;
            if (h < nel) se[h] = ev[u];
        }
        // x and the fixed-DOF flags of this thread's R1 entries, in flight
        // across the barrier (issued with the first loads they cost more)
        Vec2<T> xv[P1];
        int fv[P1];
#pragma unroll
        for (int u = 0; u < P1; u++) {
            const int h = threadIdx.x + u * 256;
            const int a = h / w1, b = h - a * w1;
            const int ii = i0 - 1 + a, jj = j0 - 1 + b;
            xv[u] = Vec2<T>{0, 0};
            fv[u] = 0;
            if (h < n1 && ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
                const long n = (long)(ny + 1) * ii + jj;
                fv[u] = fix[n];
                if (prev && xupd && a >= 1 && a <= TI && b >= 1 && b <= TJ) xv[u] = load2(V.x, n);
            }
        }
        __syncthreads();
        Vec2<T> un[P1];
#pragma unroll
        for (int u = 0; u < P1; u++) {
            const int h = threadIdx.x + u * 256;
            un[u] = Vec2<T>{0, 0};
            if (h >= n1) continue;
            const int a = h / w1, b = h - a * w1;  // R1 coordinates
            const int ii = i0 - 1 + a, jj = j0 - 1 + b;
            if (ii < 0 || ii > nx || jj < 0 || jj > ny) continue;
            const long n = (long)(ny + 1) * ii + jj;
            const bool mine = a >= 1 && a <= TI && b >= 1 && b <= TJ;
            const Vec2<T>* s0 = sp + a * w2 + b;  // R2 rows a, a+1, a+2 from column b
            T ax = 0, ay = 0, ex, ey;
            if (prev) {  // s = K p (alpha = 0 at launch 0)
                if (ii >= 1 && jj >= 1) {
                    elem_rows_q4<T>(K0, 2, s0[0], s0[w2], s0[w2 + 1], s0[1], ex, ey);
                    const T Ee = se[a * we + b];
                    ax += Ee * ex; ay += Ee * ey;
                }
                if (ii >= 1 && jj < ny) {
                    elem_rows_q4<T>(K0, 1, s0[1], s0[w2 + 1], s0[w2 + 2], s0[2], ex, ey);
                    const T Ee = se[a * we + b + 1];
                    ax += Ee * ex; ay += Ee * ey;
                }
                if (ii < nx && jj >= 1) {
                    elem_rows_q4<T>(K0, 3, s0[w2], s0[2 * w2], s0[2 * w2 + 1], s0[w2 + 1], ex, ey);
                    const T Ee = se[(a + 1) * we + b];
                    ax += Ee * ex; ay += Ee * ey;
                }
                if (ii < nx && jj < ny) {
                    elem_rows_q4<T>(K0, 0, s0[w2 + 1], s0[2 * w2 + 1], s0[2 * w2 + 2], s0[w2 + 2], ex, ey);
                    const T Ee = se[(a + 1) * we + b + 1];
                    ax += Ee * ex; ay += Ee * ey;
                }
                if (fv[u] & 1) ax = 0;
                if (fv[u] & 2) ay = 0;
            }
            Vec2<T> rn;
            rn.x = rv[u].x - ta * ax;  // r -= alpha s
            rn.y = rv[u].y - ta * ay;
            un[u].x = rn.x * dv[u].x;
            un[u].y = rn.y * dv[u].y;
            if (mine) {
                const Vec2<T> pc = s0[w2 + 1];
                store2(V.rout, n, rn);
                store2(V.pout, n, pc);
                if (xupd) {  // pv[u] is p_{m-2} at this R1 node (R1 entries lead the R2 order)
                    Vec2<T> xn;
                    xn.x = (xv[u].x + tap * pv[u].x) + ta * pc.x;  // x += alpha p, two launches' worth
                    xn.y = (xv[u].y + tap * pv[u].y) + ta * pc.y;
                    store2(V.x, n, xn);
                }
                acc[0] += (double)rn.x * (double)un[u].x;
                acc[0] += (double)rn.y * (double)un[u].y;
                acc[2] += (double)rn.x * (double)rn.x;
                acc[2] += (double)rn.y * (double)rn.y;
            }
        }
        __syncthreads();  // every read of p_{m-1} is done: u_m takes its place
        Vec2<T>* su = sp;
#pragma unroll
        for (int u = 0; u < P1; u++) {
            const int h = threadIdx.x + u * 256;
            if (h < n1) su[h] = un[u];
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int q = threadIdx.x + o * 256;
            const int r = q / TJ, c = q - r * TJ;
            const int i = i0 + r, j = j0 + c;
            if (q >= own || i > nx || j > ny) continue;
            const Vec2<T>* s0 = su + r * w1 + c;  // R1 rows r, r+1, r+2 from column c
            T ax = 0, ay = 0, ex, ey;
            if (i >= 1 && j >= 1) {
                elem_rows_q4<T>(K0, 2, s0[0], s0[w1], s0[w1 + 1], s0[1], ex, ey);
                const T Ee = se[(r + 1) * we + c + 1];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i >= 1 && j < ny) {
                elem_rows_q4<T>(K0, 1, s0[1], s0[w1 + 1], s0[w1 + 2], s0[2], ex, ey);
                const T Ee = se[(r + 1) * we + c + 2];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j >= 1) {
                elem_rows_q4<T>(K0, 3, s0[w1], s0[2 * w1], s0[2 * w1 + 1], s0[w1 + 1], ex, ey);
                const T Ee = se[(r + 2) * we + c + 1];
                ax += Ee * ex; ay += Ee * ey;
            }
            if (i < nx && j < ny) {
                elem_rows_q4<T>(K0, 0, s0[w1 + 1], s0[2 * w1 + 1], s0[2 * w1 + 2], s0[w1 + 2], ex, ey);
                const T Ee = se[(r + 2) * we + c + 2];
                ax += Ee * ex; ay += Ee * ey;
            }
            const Vec2<T> uc = s0[w1 + 1];
            acc[1] += (double)uc.x * (double)ax;
            acc[1] += (double)uc.y * (double)ay;
        }
    }
    store_partials<3>(acc, lds, partOut);
}

template <class T>
__global__ void k_recip(long n, const T* __restrict__ D, T* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (T)1 / D[i];
}

__global__ void k_cg1_start(PcgDev* __restrict__ S) {
    S->done = 0;
    S->status = 0;
    S->iterations = 0;
}

// After the host's last launch (M launches: iterate M-1 is the last one):
// the convergence test of that iterate and the itrmax exit (CG.h:451-452).
__global__ void k_cg1_final(int M, const double* __restrict__ partIn, int nbIn, PcgDev* __restrict__ S, double eps) {
    __shared__ double lds[48];  // block_sum<3>: 16 per sum
    if (S->done) return;
    double v[3];
    reduce_partials<3>(partIn, nbIn, lds, v);
    if (threadIdx.x == 0) {
        const double rnorm = sqrt(v[2]);
        S->rnorm = rnorm;
        S->iterations = M - 1;
        S->status = (M > 1 && rnorm < eps * S->bnorm) ? 1 : 2;
        S->done = 1;
    }
}

// After k_cg1_final: when the last finished launch L = S->iterations is odd,
// x holds x_{L-1} and p_{L-1} (the p that launch formed) is in p; add
// alpha_L p_{L-1} (alpha_L in S->a[(L - 1) & 1]) as launch L would have.
template <class T>
__global__ void __launch_bounds__(256) k_cg_x_fix(long n, const T* __restrict__ p, T* __restrict__ x,
                                                  const PcgDev* __restrict__ S) {
#pragma clang fp contract(fast)  // the same contraction as the kernels' own x update
    const int L = S->iterations;
    if (!(L & 1)) return;
    const T a = (T)S->a[(L - 1) & 1];
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = x[i] + a * p[i];
}

// CSR flavour of K1 (free-DOF vectors): q_i = sum_j a_ij (beta pold_j + z_j),
// each row summed in column order from 0 as CSR<T>::operator* does.
__global__ void __launch_bounds__(256) k_pcg_k1_csr(int N, int k, const int32_t* __restrict__ indptr,
                                                    const int32_t* __restrict__ indices,
                                                    const double* __restrict__ data, const double* __restrict__ pold,
                                                    const double* __restrict__ z, double* __restrict__ pnew,
                                                    double* __restrict__ q, const double* __restrict__ partB, int nbB,
                                                    double* __restrict__ partA, PcgDev* __restrict__ S, double eps) {
    __shared__ double lds[32];
    if (S->done) return;
    double beta;
    bool stop;
    pcg_head(k, partB, nbB, S, eps, lds, beta, stop);
    if (stop) return;
    double acc[1] = {0.0};
    for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < N; r += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int jj = indptr[r]; jj < indptr[r + 1]; jj++) {
            int c = indices[jj];
            double pc = beta * pold[c] + z[c];
            s += data[jj] * pc;
        }
        double pr = beta * pold[r] + z[r];
        pnew[r] = pr;
        q[r] = s;
        acc[0] += pr * s;
    }
    store_partials<1>(acc, lds, partA);
}

template <class T>
__global__ void __launch_bounds__(256) k_pcg_k2(long n, int k, T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                const T* __restrict__ p, const T* __restrict__ q,
                                                const T* __restrict__ D, const double* __restrict__ partA, int nbA,
                                                double* __restrict__ partB, PcgDev* __restrict__ S) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    __shared__ double lds[32];
    // first pair of every thread, the partials and the done flag are all
    // loaded before the first wait
    const long n2 = n / 2;
    const long stride = (long)gridDim.x * blockDim.x;
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    Vec2<T> xi{0, 0}, ri{0, 0}, pi{0, 0}, qi{0, 0}, di{1, 1};
    if (i < n2) {
        xi = load2(x, i); ri = load2(r, i); pi = load2(p, i); qi = load2(q, i); di = load2(D, i);
    }
    PartRegs<1, 8> pr;
    load_partials(partA, nbA, pr);
    if (S->done) return;
    double v[1];
    sum_partials(pr, partA, nbA, lds, v);
    const double zr = S->zr[k & 1];
    const double alpha = zr / v[0];  // CG.h:433
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        S->pq = v[0];
        S->alpha = alpha;
    }
    const T ta = (T)alpha, tma = (T)(-alpha);
    double acc[2] = {0.0, 0.0};
    // pairs of entries per access (n is even for nodal vectors); an odd tail
    // (free-numbered CSR vectors) is handled by the scalar step below
    while (i < n2) {
        xi.x = xi.x + ta * pi.x;   // xexpay(x, alpha, p)
        xi.y = xi.y + ta * pi.y;
        ri.x = ri.x + tma * qi.x;  // xexpay(r, -alpha, Ap)
        ri.y = ri.y + tma * qi.y;
        Vec2<T> zi{ri.x / di.x, ri.y / di.y};  // Scaling (CG.h:412)
        store2(x, i, xi);
        store2(r, i, ri);
        store2(z, i, zi);
        acc[0] += (double)zi.x * (double)ri.x;
        acc[0] += (double)zi.y * (double)ri.y;
        acc[1] += (double)ri.x * (double)ri.x;
        acc[1] += (double)ri.y * (double)ri.y;
        i += stride;
        if (i < n2) {
            xi = load2(x, i); ri = load2(r, i); pi = load2(p, i); qi = load2(q, i); di = load2(D, i);
        }
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        long t = n - 1;
        T xt = x[t] + ta * p[t];
        T rt = r[t] + tma * q[t];
        T zt = rt / D[t];
        x[t] = xt;
        r[t] = rt;
        z[t] = zt;
        acc[0] += (double)zt * (double)rt;
        acc[1] += (double)rt * (double)rt;
    }
    store_partials<2>(acc, lds, partB);
}

// x = 0, r = b, z = p0 = b ./ D, pold = 0; partials (z.r, b.b) for K1(0).
template <class T>
__global__ void __launch_bounds__(256) k_pcg_init(long n, const T* __restrict__ b, const T* __restrict__ D,
                                                  T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                  T* __restrict__ pold, double* __restrict__ partB,
                                                  PcgDev* __restrict__ S) {
    __shared__ double lds[32];
    double acc[2] = {0.0, 0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        T bi = b[i];
        T ri = bi - (T)0;  // subtract(b, A*0) (CG.h:424)
        T zi = ri / D[i];
        x[i] = 0;
        r[i] = ri;
        z[i] = zi;
        pold[i] = 0;
        acc[0] += (double)zi * (double)ri;
        acc[1] += (double)bi * (double)bi;
    }
    store_partials<2>(acc, lds, partB);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        S->done = 0;
        S->status = 0;
        S->iterations = 0;
    }
}

// After the host's last K2: test convergence of the final iterate the way
// K1 would, and record the itrmax exit (CG.h:451-452).
__global__ void k_pcg_final(int k, const double* __restrict__ partB, int nbB, PcgDev* __restrict__ S, double eps) {
    __shared__ double lds[32];
    if (S->done) return;
    double v[2];
    reduce_partials<2>(partB, nbB, lds, v);
    if (threadIdx.x == 0) {
        double rnorm = sqrt(v[1]);
        S->rnorm = rnorm;
        S->iterations = k;
        S->status = (k > 0 && rnorm < eps * S->bnorm) ? 1 : 2;
        S->done = 1;
    }
}

// ============================================================= CSR ========
// Closed-form row lengths of the structured quad4 matrix: the free DOFs of
// the 3x3 node block around the row's node (every pair of nodes in that block
// shares an element).
__global__ void k_csr_count_q4(int nx, int ny, const int32_t* __restrict__ n2g, const uint8_t* __restrict__ fix,
                               int32_t* __restrict__ rowlen) {
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        int cnt = 0;
        for (int ii = i - 1; ii <= i + 1; ii++)
            for (int jj = j - 1; jj <= j + 1; jj++) {
                if (ii < 0 || ii > nx || jj < 0 || jj > ny) continue;
                uint8_t f = fix[(long)(ny + 1) * ii + jj];
                cnt += !(f & 1) + !(f & 2);
            }
        for (int d = 0; d < 2; d++) {
            int g = n2g[2 * n + d];
            if (g >= 0) rowlen[g] = cnt;
        }
    }
}

// Values: for row (node n, dof d) and column (node m, dof d'), the sum over
// the elements containing both nodes, in ascending element id, of
// Ke_e(2 loc_n + d, 2 loc_m + d'), starting from 0.0 + first term, exactly as
// LILCSR set/get accumulates (Assembling.h:54-56, LILCSR.h:92-114).
__device__ inline int loc_q4(int ei, int ej, int ni, int nj) {
    // local index of node (ni,nj) in element (ei,ej): BL 0, BR 1, TR 2, TL 3
    int di = ni - ei, dj = nj - ej;
    return dj == 0 ? di : 3 - di;
}

__global__ void k_csr_fill_q4(int nx, int ny, const int32_t* __restrict__ n2g, const int32_t* __restrict__ indptr,
                              const double* __restrict__ ke_all, int32_t* __restrict__ indices,
                              double* __restrict__ data) {
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        for (int d = 0; d < 2; d++) {
            int row = n2g[2 * n + d];
            if (row < 0) continue;
            int pos = indptr[row];
            for (int ii = i - 1; ii <= i + 1; ii++)
                for (int jj = j - 1; jj <= j + 1; jj++) {
                    if (ii < 0 || ii > nx || jj < 0 || jj > ny) continue;
                    long m = (long)(ny + 1) * ii + jj;
                    for (int d2 = 0; d2 < 2; d2++) {
                        int col = n2g[2 * m + d2];
                        if (col < 0) continue;
                        double v = 0.0;
                        // elements containing n and m, ascending id (i-major)
                        int ei0 = max(max(i, ii) - 1, 0), ei1 = min(min(i, ii), nx - 1);
                        int ej0 = max(max(j, jj) - 1, 0), ej1 = min(min(j, jj), ny - 1);
                        for (int ei = ei0; ei <= ei1; ei++)
                            for (int ej = ej0; ej <= ej1; ej++) {
                                const double* Ke = ke_all + ((long)ny * ei + ej) * 64;
                                int a = 2 * loc_q4(ei, ej, i, j) + d, b = 2 * loc_q4(ei, ej, ii, jj) + d2;
                                v = v + Ke[a * 8 + b];
                            }
                        indices[pos] = col;
                        data[pos] = v;
                        pos++;
                    }
                }
        }
    }
}

// CSR<T>::operator* (CSR.h:108-122): row sums from 0 in column order.
__global__ void k_csr_spmv(int N, const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                           const double* __restrict__ data, const double* __restrict__ x, double* __restrict__ y) {
    for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < N; r += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int jj = indptr[r]; jj < indptr[r + 1]; jj++) s += data[jj] * x[indices[jj]];
        y[r] = s;
    }
}

// Partials of ||b - A x||^2 for free-numbered vectors (A assembled).
__global__ void __launch_bounds__(256) k_csr_residual(int N, const int32_t* __restrict__ indptr,
                                                      const int32_t* __restrict__ indices,
                                                      const double* __restrict__ data, const double* __restrict__ b,
                                                      const double* __restrict__ x, double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[1] = {0.0};
    for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < N; r += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int jj = indptr[r]; jj < indptr[r + 1]; jj++) s += data[jj] * x[indices[jj]];
        const double d = b[r] - s;
        acc[0] += d * d;
    }
    store_partials<1>(acc, lds, part);
}

// GetDiagonal via CSR::get (CG.h:397-404, CSR.h:154-167).
__global__ void k_csr_diag(int N, const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                           const double* __restrict__ data, double* __restrict__ D) {
    for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < N; r += (long)gridDim.x * blockDim.x) {
        int lo = indptr[r], hi = indptr[r + 1], end = hi;
        while (lo < hi) {
            int mid = lo + (hi - lo) / 2;
            if (indices[mid] < r) lo = mid + 1; else hi = mid;
        }
        D[r] = (lo < end && indices[lo] == r) ? data[lo] : 0.0;
    }
}

// Exclusive scan of row lengths into indptr (single workgroup, sequential
// chunks; runs once per assembly).
__global__ void k_scan(const int32_t* __restrict__ len, int32_t* __restrict__ out, int n) {
    __shared__ int32_t sums[1024];
    const int t = threadIdx.x, nt = blockDim.x;
    long chunk = (n + nt - 1) / nt;
    long s0 = t * chunk, s1 = min((long)n, s0 + chunk);
    int32_t s = 0;
    for (long i = s0; i < s1; i++) s += len[i];
    sums[t] = s;
    __syncthreads();
    if (t == 0) {
        int32_t run = 0;
        for (int k = 0; k < nt; k++) { int32_t v = sums[k]; sums[k] = run; run += v; }
        out[n] = run;
    }
    __syncthreads();
    int32_t run = sums[t];
    for (long i = s0; i < s1; i++) { out[i] = run; run += len[i]; }
}

// ==================================================== element matrices ====
// PlaneStrainStiffness<T, ShapeFunction4Square, Gauss4Square>
// (PlaneStrain.h:19-58) in the reference's operation order: node
// coordinates lx*(i/(double)nx) (SquareMesh.h:66), dXdr = dNdr X, cofactor
// inverse divided by the determinant, B^T D B J t w0 w1 accumulated per
// Gauss point.  One thread per element.
__device__ inline void mm_dev(const double* A, const double* B, double* C, int m, int k, int n) {
    for (int i = 0; i < m; i++)
        for (int j = 0; j < n; j++) {
            double v = 0.0;
            for (int q = 0; q < k; q++) v += A[i * k + q] * B[q * n + j];
            C[i * n + j] = v;
        }
}

__device__ void ke_q4_ref(const double* X, double E, double nu, double t, double* Ke) {
    const double a = 1.0 / sqrt(3.0);
    const double m = -1.0 / sqrt(3.0);
    const double gp[4][2] = {{m, m}, {a, m}, {m, a}, {a, a}};
    double D[9] = {1.0 - nu, nu, 0.0, nu, 1.0 - nu, 0.0, 0.0, 0.0, 0.5 * (1.0 - 2.0 * nu)};
    double c = E / ((1.0 - 2.0 * nu) * (1.0 + nu));
    for (int k = 0; k < 9; k++) D[k] *= c;
    for (int k = 0; k < 64; k++) Ke[k] = 0.0;
    for (int g = 0; g < 4; g++) {
        double r0 = gp[g][0], r1 = gp[g][1];
        double dN[8] = {-0.25 * (1.0 - r1), 0.25 * (1.0 - r1), 0.25 * (1.0 + r1), -0.25 * (1.0 + r1),
                        -0.25 * (1.0 - r0), -0.25 * (1.0 + r0), 0.25 * (1.0 + r0), 0.25 * (1.0 - r0)};
        double J2[4], inv[4], dNdX[8], B[24], Bt[24], BtD[24], M[64];
        mm_dev(dN, X, J2, 2, 4, 2);
        double det = J2[0] * J2[3] - J2[1] * J2[2];
        inv[0] = J2[3] / det;
        inv[1] = (-J2[1]) / det;
        inv[2] = (-J2[2]) / det;
        inv[3] = J2[0] / det;
        mm_dev(inv, dN, dNdX, 2, 2, 4);
        for (int n = 0; n < 4; n++) {
            B[2 * n] = dNdX[n];         B[2 * n + 1] = 0.0;
            B[8 + 2 * n] = 0.0;         B[8 + 2 * n + 1] = dNdX[4 + n];
            B[16 + 2 * n] = dNdX[4 + n]; B[16 + 2 * n + 1] = dNdX[n];
        }
        for (int r = 0; r < 8; r++)
            for (int s = 0; s < 3; s++) Bt[r * 3 + s] = B[s * 8 + r];
        mm_dev(Bt, D, BtD, 8, 3, 3);
        mm_dev(BtD, B, M, 8, 3, 8);
        for (int k = 0; k < 64; k++) Ke[k] += M[k] * det * t * 1.0 * 1.0;
    }
}

__global__ void k_ke_all_q4(int nx, int ny, double lx, double ly, const double* __restrict__ E, double nu, double t,
                            double* __restrict__ ke_all) {
    const long ne = (long)nx * ny;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        int i = (int)(e / ny), j = (int)(e - (long)i * ny);
        double x0 = lx * (i / (double)nx), x1 = lx * ((i + 1) / (double)nx);
        double y0 = ly * (j / (double)ny), y1 = ly * ((j + 1) / (double)ny);
        double X[8] = {x0, y0, x1, y0, x1, y1, x0, y1};
        double Ke[64];
        ke_q4_ref(X, E[e], nu, t, Ke);
        double* out = ke_all + e * 64;
        for (int k = 0; k < 64; k++) out[k] = Ke[k];
    }
}

// ============================================================ filter ======
// Element centroids as CenterOfGravity computes them (General.h:70-77):
// ((((0 + x_BL) + x_BR) + x_TR) + x_TL) / 4.
__global__ void k_centroids_q4(int nx, int ny, double lx, double ly, double* __restrict__ cg) {
    const long ne = (long)nx * ny;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        int i = (int)(e / ny), j = (int)(e - (long)i * ny);
        double x0 = lx * (i / (double)nx), x1 = lx * ((i + 1) / (double)nx);
        double y0 = ly * (j / (double)ny), y1 = ly * ((j + 1) / (double)ny);
        double cx = 0.0, cy = 0.0;
        cx += x0; cy += y0;
        cx += x1; cy += y0;
        cx += x1; cy += y1;
        cx += x0; cy += y1;
        cg[2 * e] = cx / 4.0;
        cg[2 * e + 1] = cy / 4.0;
    }
}

// Filter weight of the pair (i, j) as the sample driver computes it
// (sample_optimize_density_oc.cpp:55-57, Vector::Norm at Vector.h:297-303).
__device__ inline bool filter_w(const double* __restrict__ cg, long a, long b, double R, double& w) {
    double v0 = cg[2 * a] - cg[2 * b], v1 = cg[2 * a + 1] - cg[2 * b + 1];
    double s = 0.0;
    s += v0 * v0;
    s += v1 * v1;
    double d = sqrt(s);
    if (!(d <= R)) return false;
    w = (R - d) / R;
    return true;
}

// mode 0: rho_i = sum_j w_ij s_j / sum_j w_ij  (DensityFilter.h:45-56)
// mode 1: dfds_i = sum_j dfdrho_j w_ij / sum_j w_ij (DensityFilter.h:60-71)
// Neighbours visited in ascending element id inside a +-win window.
// The filtered value of element e; in(m) gives the input at element m.
template <class IN>
__device__ inline double filter_one_f(int nx, int ny, int win, double R, const double* __restrict__ cg, const IN& in,
                                      long e) {
    int i = (int)(e / ny), j = (int)(e - (long)i * ny);
    double acc = 0.0, wsum = 0.0;
    int i0 = max(i - win, 0), i1 = min(i + win, nx - 1), j0 = max(j - win, 0), j1 = min(j + win, ny - 1);
    for (int ii = i0; ii <= i1; ii++)
        for (int jj = j0; jj <= j1; jj++) {
            long m = (long)ny * ii + jj;
            double w;
            if (filter_w(cg, e, m, R, w)) {
                acc += w * in(m);
                wsum += w;
            }
        }
    return acc / wsum;
}

__device__ inline double filter_one(int nx, int ny, int win, double R, const double* __restrict__ cg,
                                    const double* __restrict__ in, long e) {
    return filter_one_f(nx, ny, win, R, cg, [&](long m) { return in[m]; }, e);
}

__global__ void __launch_bounds__(256) k_filter_q4(int nx, int ny, int win, double R, const double* __restrict__ cg,
                                                   const double* __restrict__ in, double* __restrict__ out) {
    const long ne = (long)nx * ny;
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x)
        out[e] = filter_one(nx, ny, win, R, cg, in, e);
}

// SensitivityFilter<T> (scheme 1, SensitivityFilter.h:44-55):
//   out_i = sum_j (w_ij s_j) df_j / (sum_j w_ij * s_i);
// SensitivityFilter2<T> (scheme 2, SensitivityFilter.h:88-99):
//   out_i = sum_j (w_ij s_j) df_j / sum_j (w_ij s_j);
// sums from zero in neighbour order, as the reference adds them.
__device__ inline void sens_filter_add(int scheme, double w, double sj, double dfj, double& acc, double& den) {
    const double ws = w * sj;
    acc += ws * dfj;
    den += scheme == 2 ? ws : w;
}
__device__ inline double sens_filter_end(int scheme, double acc, double den, double si) {
    return scheme == 2 ? acc / den : acc / (den * si);
}

__global__ void __launch_bounds__(256) k_sensfilter_q4(int nx, int ny, int win, double R,
                                                       const double* __restrict__ cg, const double* __restrict__ s,
                                                       const double* __restrict__ df, int scheme,
                                                       double* __restrict__ out) {
    const long ne = (long)nx * ny;
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x) {
        int i = (int)(e / ny), j = (int)(e - (long)i * ny);
        double acc = 0.0, den = 0.0;
        int i0 = max(i - win, 0), i1 = min(i + win, nx - 1), j0 = max(j - win, 0), j1 = min(j + win, ny - 1);
        for (int ii = i0; ii <= i1; ii++)
            for (int jj = j0; jj <= j1; jj++) {
                long m = (long)ny * ii + jj;
                double w;
                if (filter_w(cg, e, m, R, w)) sens_filter_add(scheme, w, s[m], df[m], acc, den);
            }
        out[e] = sens_filter_end(scheme, acc, den, s[e]);
    }
}

__global__ void __launch_bounds__(256) k_sensfilter_lists(long ne, const int32_t* __restrict__ ptr,
                                                          const int32_t* __restrict__ idx,
                                                          const double* __restrict__ w, const double* __restrict__ s,
                                                          const double* __restrict__ df, int scheme,
                                                          double* __restrict__ out) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        double acc = 0.0, den = 0.0;
        for (int k = ptr[e]; k < ptr[e + 1]; k++) sens_filter_add(scheme, w[k], s[idx[k]], df[idx[k]], acc, den);
        out[e] = sens_filter_end(scheme, acc, den, s[e]);
    }
}

// DensityFilter<T> over caller-given neighbour lists (DensityFilter.h:45-71):
// out_i = (sum_j w_ij in_{idx_ij}) / (sum_j w_ij), both sums from zero in
// list order, as GetFilteredVariables / GetFilteredSensitivitis add them.
__global__ void __launch_bounds__(256) k_filter_lists(long ne, const int32_t* __restrict__ ptr,
                                                      const int32_t* __restrict__ idx, const double* __restrict__ w,
                                                      const double* __restrict__ in, double* __restrict__ out) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        double acc = 0.0, wsum = 0.0;
        for (int k = ptr[e]; k < ptr[e + 1]; k++) {
            double wk = w[k];
            acc = acc + wk * in[idx[k]];
            wsum = wsum + wk;
        }
        out[e] = acc / wsum;
    }
}

// g = sum_i scale1 rho_i / (vf ne) - scale1 (sample...oc.cpp:99-105); the
// per-element terms are summed in a fixed tree order.
__global__ void __launch_bounds__(256) k_volume_partials(long ne, const double* __restrict__ rho, double vf,
                                                         double scale1, double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[1] = {0.0};
    const double den = vf * (double)ne;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x)
        acc[0] += scale1 * rho[e] / den;
    store_partials<1>(acc, lds, part);
}

__global__ void k_reduce_final(const double* __restrict__ part, int nparts, int K, double scale, double shift,
                               double* __restrict__ out) {
    __shared__ double lds[64];
    for (int k = 0; k < K; k++) {
        double v[1] = {0.0};
        for (int i = threadIdx.x; i < nparts; i += blockDim.x) v[0] += part[i * K + k];
        block_sum<1>(v, lds);
        if (threadIdx.x == 0) out[k] = scale * v[0] - shift;
    }
}

// ============================================ compliance / sensitivity ====
// Entry idx (a nodal index, node * ndpn + dof) of the displacement: nodal u
// directly, or (FREE) a free-DOF vector read through nodetoglobal, 0 at
// fixed DOFs -- the same values either way.
template <bool FREE>
__device__ inline double u_entry(const double* __restrict__ u, const int32_t* __restrict__ n2g, long idx) {
    if constexpr (FREE) {
        const int gi = n2g[idx];
        return gi < 0 ? 0.0 : u[gi];
    } else {
        return u[idx];
    }
}

// Per element c_e = u_e^T K0 u_e (Matrix*Vector then Vector*Vector order),
// dfdrho_e = -scale0 p (E1 - E0) rho^(p-1) c_e (sample...oc.cpp:161) and the
// compliance terms E_e c_e (u^T K u = sum_e E_e c_e with fixed DOFs at 0).
template <bool FREE = false>
__global__ void __launch_bounds__(256) k_comp_sens_q4(int nx, int ny, const double* __restrict__ u,
                                                      const double* __restrict__ E, const double* __restrict__ rho,
                                                      const double* __restrict__ K0, double coef, double pm1,
                                                      double* __restrict__ dfdrho, double* __restrict__ part,
                                                      const int32_t* __restrict__ n2g = nullptr) {
    __shared__ double lds[32];
    const long ne = (long)nx * ny;
    double acc[1] = {0.0};
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x) {
        int i = (int)(e / ny), j = (int)(e - (long)i * ny);
        long nbl = (long)(ny + 1) * i + j, nbr = nbl + (ny + 1);
        double ue[8] = {u_entry<FREE>(u, n2g, 2 * nbl),           u_entry<FREE>(u, n2g, 2 * nbl + 1),
                        u_entry<FREE>(u, n2g, 2 * nbr),           u_entry<FREE>(u, n2g, 2 * nbr + 1),
                        u_entry<FREE>(u, n2g, 2 * (nbr + 1)),     u_entry<FREE>(u, n2g, 2 * (nbr + 1) + 1),
                        u_entry<FREE>(u, n2g, 2 * (nbl + 1)),     u_entry<FREE>(u, n2g, 2 * (nbl + 1) + 1)};
        double c = 0.0;
        for (int a = 0; a < 8; a++) {
            double ka = 0.0;
            for (int b = 0; b < 8; b++) ka += K0[a * 8 + b] * ue[b];
            c += ue[a] * ka;
        }
        dfdrho[e] = coef * simp_pow(rho[e], pm1) * c;
        acc[0] += E[e] * c;
    }
    store_partials<1>(acc, lds, part);
}

// ================================================================ OC =====
// OC<T>::UpdateVariables (OC.h:76-107).  One bisection step is two launches:
//   k_oc_xplus(k): decide step k-1 from its volume partials (g > 0 -> l0 =
//     lambda else l1 = lambda), stop when (l1-l0)/(l1+l0) <= lambdaeps, else
//     lambda = (l1+l0)/2 and x+ = clamp(x (-dfdx/(dgdx lambda))^iota);
//   k_oc_volume(k): filter x+ and sum the closure's volume terms.
// The bracket of step k lives in slot k of the history arrays.
// x+ = (-dfdx / (dgdx lambda))^iota x clamped to [max(0, (1-m) x),
// min(1, (1+m) x)] (OC.h:86-91); iota = 0.5 takes the correctly rounded
// sqrt, which glibc's pow(., 0.5) also returns.
__device__ inline double oc_candidate(double xi, double dfdxi, double dgdxi, double lambda, double iota,
                                      double move) {
    double base = -dfdxi / (dgdxi * lambda);
    double v = (iota == 0.5 ? sqrt(base) : pow(base, iota)) * xi;
    double lo = std_max0((1.0 - move) * xi), hi = std_min1((1.0 + move) * xi);
    if (v < lo) v = lo;
    else if (v > hi) v = hi;
    return v;
}

// HeavisideFilter projection of a filtered value st (HeavisideFilter.h:73)
// and its derivative d rho / d st (HeavisideFilter.h:87), in the reference's
// operation order (pow(t, 2.0) is t*t in the reference's build).
__device__ inline double heaviside_rho(double st, double beta) {
    return 0.5 * (tanh(0.5 * beta) + tanh(beta * (st - 0.5))) / tanh(0.5 * beta);
}
__device__ inline double heaviside_drho(double st, double beta) {
    const double t = tanh(beta * (st - 0.5));
    return 0.5 * beta * (1.0 - t * t) / tanh(0.5 * beta);
}

// rho = H(st); dr = H'(st) when dr is non-null.
__global__ void __launch_bounds__(256) k_heaviside(long ne, const double* __restrict__ st, double beta,
                                                   double* __restrict__ rho, double* __restrict__ dr) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < ne; e += (long)gridDim.x * blockDim.x) {
        const double v = st[e];
        rho[e] = heaviside_rho(v, beta);
        if (dr) dr[e] = heaviside_drho(v, beta);
    }
}

// out = a .* b
__global__ void __launch_bounds__(256) k_mul_d(long n, const double* __restrict__ a, const double* __restrict__ b,
                                               double* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = a[i] * b[i];
}

// out = c * b
__global__ void __launch_bounds__(256) k_cmul_d(long n, double c, const double* __restrict__ b,
                                                double* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = c * b[i];
}

struct OcDev {
    double l0i, l1i;  // initial bracket (lambdamin, lambdamax), set by the host
    double l0[2], l1[2], lambda[2];
    double g_last, lambda_last;
    int steps, done, status, pad;  // status: see k_oc_xplus
};

__global__ void __launch_bounds__(256) k_oc_xplus(long ne, int k, const double* __restrict__ x,
                                                  const double* __restrict__ dfdx, const double* __restrict__ dgdx,
                                                  double iota, double move, double leps, double scale1,
                                                  const double* __restrict__ part, int nparts,
                                                  double* __restrict__ xplus, OcDev* __restrict__ S) {
    __shared__ double lds[32];
    if (S->done) return;
    double l0, l1;
    if (k == 0) {
        l0 = S->l0i;
        l1 = S->l1i;
    } else {
        double v[1];
        reduce_partials<1>(part, nparts, lds, v);
        double g = v[0] - 1.0 * scale1;
        l0 = S->l0[(k - 1) & 1];
        l1 = S->l1[(k - 1) & 1];
        double lam = S->lambda[(k - 1) & 1];
        if (g > 0.0) l0 = lam; else l1 = lam;
        if (threadIdx.x == 0 && blockIdx.x == 0) S->g_last = g;
    }
    if (!((l1 - l0) / (l1 + l0) > leps)) {
        if (threadIdx.x == 0 && blockIdx.x == 0) {
            S->steps = k;
            S->done = 1;
            // status 1: every tested lambda left the volume constraint
            // violated (l1 never lowered: the bracket's upper end is too
            // small); 2: every tested lambda satisfied it with a positive
            // lower end (l0 never raised).  The reference returns silently.
            S->status = (k > 0 && l1 == S->l1i) ? 1 : (k > 0 && l0 == S->l0i && l0 > 0.0) ? 2 : 0;
        }
        return;
    }
    const double lambda = 0.5 * (l1 + l0);
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        S->l0[k & 1] = l0;
        S->l1[k & 1] = l1;
        S->lambda[k & 1] = lambda;
        S->lambda_last = lambda;
        S->steps = k + 1;
    }
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ne; i += (long)gridDim.x * blockDim.x)
        xplus[i] = oc_candidate(x[i], dfdx[i], dgdx[i], lambda, iota, move);
}

// One whole bisection step of the quad4 grid rule in one launch: the
// decision of step k-1 from its volume partials (buffer (k-1) & 1), the
// stopping test, lambda, x+ at lambda for this workgroup's elements, and the
// filtered volume of x+ (its neighbours' candidates recomputed rather than
// read, since other workgroups of this launch are writing them) into the
// partials of step k (buffer k & 1, kMaxPartials apart).  The same
// decisions and candidates as k_oc_xplus + k_oc_volume.
__global__ void __launch_bounds__(256) k_oc_step(int nx, int ny, int win, double R, const double* __restrict__ cg,
                                                 int k, const double* __restrict__ x, const double* __restrict__ dfdx,
                                                 const double* __restrict__ dgdx, double iota, double move,
                                                 double leps, double vf, double scale1, double beta,
                                                 double* __restrict__ part, int nparts, double* __restrict__ xplus,
                                                 OcDev* __restrict__ S) {
    __shared__ double lds[32];
    if (S->done) return;
    double l0, l1;
    if (k == 0) {
        l0 = S->l0i;
        l1 = S->l1i;
    } else {
        double v[1];
        reduce_partials<1>(part + ((k - 1) & 1) * kMaxPartials, nparts, lds, v);
        double g = v[0] - 1.0 * scale1;
        l0 = S->l0[(k - 1) & 1];
        l1 = S->l1[(k - 1) & 1];
        double lam = S->lambda[(k - 1) & 1];
        if (g > 0.0) l0 = lam; else l1 = lam;
        if (threadIdx.x == 0 && blockIdx.x == 0) S->g_last = g;
    }
    if (!((l1 - l0) / (l1 + l0) > leps)) {
        if (threadIdx.x == 0 && blockIdx.x == 0) {
            S->steps = k;
            S->done = 1;
            S->status = (k > 0 && l1 == S->l1i) ? 1 : (k > 0 && l0 == S->l0i && l0 > 0.0) ? 2 : 0;
        }
        return;
    }
    const double lambda = 0.5 * (l1 + l0);
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        S->l0[k & 1] = l0;
        S->l1[k & 1] = l1;
        S->lambda[k & 1] = lambda;
        S->lambda_last = lambda;
        S->steps = k + 1;
    }
    const long ne = (long)nx * ny;
    const double den = vf * (double)ne;
    auto cand = [&](long m) { return oc_candidate(x[m], dfdx[m], dgdx[m], lambda, iota, move); };
    double acc[1] = {0.0};
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x) {
        xplus[e] = cand(e);
        double v = filter_one_f(nx, ny, win, R, cg, cand, e);
        if (beta > 0.0) v = heaviside_rho(v, beta);  // HeavisideFilter in the closure
        acc[0] += scale1 * v / den;
    }
    store_partials<1>(acc, lds, part + (k & 1) * kMaxPartials);
}

// One bisection candidate for a given lambda (OC.h:85-92), for callers
// that evaluate the constraint themselves.
__global__ void __launch_bounds__(256) k_oc_candidate(long ne, const double* __restrict__ x,
                                                      const double* __restrict__ dfdx,
                                                      const double* __restrict__ dgdx, double lambda, double iota,
                                                      double move, double* __restrict__ xplus) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ne; i += (long)gridDim.x * blockDim.x)
        xplus[i] = oc_candidate(x[i], dfdx[i], dgdx[i], lambda, iota, move);
}

__global__ void __launch_bounds__(256) k_oc_volume(int nx, int ny, int win, double R, const double* __restrict__ cg,
                                                   const double* __restrict__ xplus, double vf, double scale1,
                                                   double beta, double* __restrict__ part,
                                                   const OcDev* __restrict__ S) {
    __shared__ double lds[32];
    if (S->done) return;
    const long ne = (long)nx * ny;
    const double den = vf * (double)ne;
    double acc[1] = {0.0};
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x) {
        double v = filter_one(nx, ny, win, R, cg, xplus, e);
        if (beta > 0.0) v = heaviside_rho(v, beta);  // HeavisideFilter in the closure
        acc[0] += scale1 * v / den;
    }
    store_partials<1>(acc, lds, part);
}

// ===================================================== true residual =====
// r = b - K x (nodal, FP64) with partials of r.r; used by the refinement
// loop and to report the true residual of every solve.
__global__ void __launch_bounds__(256) k_residual_q4(int nx, int ny, const double* __restrict__ b,
                                                     const double* __restrict__ x, double* __restrict__ r,
                                                     const double* __restrict__ E, const double* __restrict__ K0,
                                                     const uint8_t* __restrict__ fix, double* __restrict__ part) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    __shared__ double lds[32];
    const long nn = (long)(nx + 1) * (ny + 1);
    double acc[1] = {0.0};
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        Vec2<double> v[3][3];
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int bb = 0; bb < 3; bb++) {
                int ii = i + a - 1, jj = j + bb - 1;
                if (ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) v[a][bb] = load2(x, (long)(ny + 1) * ii + jj);
                else v[a][bb] = Vec2<double>{0, 0};
            }
        double yx, yy;
        apply_q4_node(nx, ny, i, j, v, E, K0, yx, yy);
        uint8_t f = fix[n];
        double rx = (f & 1) ? 0.0 : b[2 * n] - yx;
        double ry = (f & 2) ? 0.0 : b[2 * n + 1] - yy;
        r[2 * n] = rx;
        r[2 * n + 1] = ry;
        acc[0] += rx * rx;
        acc[0] += ry * ry;
    }
    store_partials<1>(acc, lds, part);
}

__global__ void k_axpy_d(long n, double a, const double* __restrict__ x, double* __restrict__ y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = y[i] + a * x[i];
}

// y = a x + y written as y += a x (used for accumulating gradients)
__global__ void k_axpby_d(long n, double a, const double* __restrict__ x, double* __restrict__ y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = y[i] + a * x[i];
}

__global__ void k_div_d(long n, const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = a[i] / b[i];
}

__global__ void k_scale_d(long n, double a, double* __restrict__ y) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = a * y[i];
}

// d = a x + c y
__global__ void k_lincomb_d(long n, double a, const double* __restrict__ x, double c, const double* __restrict__ y,
                            double* __restrict__ d) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        d[i] = a * x[i] + c * y[i];
}

// p = z + beta p
__global__ void k_axpby_d2(long n, const double* __restrict__ z, double beta, double* __restrict__ p) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        p[i] = z[i] + beta * p[i];
}

__global__ void k_axpy_f32(long n, const float* __restrict__ d, double* __restrict__ x) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = x[i] + (double)d[i];
}

// One element's PlaneStrainStiffness on the device (check path).
__global__ void k_ke_one_q4(int nx, int ny, double lx, double ly, int e, double E, double nu, double t,
                            double* __restrict__ Ke) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int i = e / ny, j = e - i * ny;
    double x0 = lx * (i / (double)nx), x1 = lx * ((i + 1) / (double)nx);
    double y0 = ly * (j / (double)ny), y1 = ly * ((j + 1) / (double)ny);
    double X[8] = {x0, y0, x1, y0, x1, y1, x0, y1};
    ke_q4_ref(X, E, nu, t, Ke);
}

__global__ void __launch_bounds__(256) k_dot_partials(long n, const double* __restrict__ a, const double* __restrict__ b,
                                                      double* __restrict__ part) {
    __shared__ double lds[32];
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        acc[0] += a[i] * b[i];
    store_partials<1>(acc, lds, part);
}

}  // namespace pf
