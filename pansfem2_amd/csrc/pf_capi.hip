// C-ABI of libpansfem2_amd: context, grids, DOF maps, operators, solvers,
// filter, OC and the device-resident SIMP loop.  Declarations and the
// reference routine each entry point replaces: include/pansfem2_amd.h.
#include <algorithm>
#include <cmath>

#include "pf_kernels.hip"
#include "pf_resident.hip"
#include "pf_mma.hip"
#include "pf_hex8.hip"
#include "pf_resident3.hip"
#include "pf_learned.hip"
#include "pf_mg.hip"
#include "pf_mg3.hip"

#include <chrono>
#include <type_traits>
#include <cstdlib>
#include <cstring>
#include <mutex>

using namespace pf;

namespace {

// workgroups of the grid-stride 1D kernels
constexpr int grid_cap() { return 1024; }

// nodes per LDS tile of the quad4 PCG operator kernel (TI rows x TJ along j)
#ifndef PF_K1_TI
#define PF_K1_TI 8
#endif
#ifndef PF_K1_TJ
#define PF_K1_TJ 64
#endif
constexpr int kTileJ = PF_K1_TJ, kTileI = PF_K1_TI;
// tile of the single-reduction kernel (k_cg1_q4_tile)
#ifndef PF_CG1_TI
#define PF_CG1_TI 8
#endif
#ifndef PF_CG1_TJ
#define PF_CG1_TJ 64
#endif

constexpr int kCg1TI = PF_CG1_TI, kCg1TJ = PF_CG1_TJ;
// the single-reduction form's carried kernel runs while its working set
// stays below this many bytes; beyond, the recomputing kernel's smaller
// per-iteration traffic wins (measured crossover near 125 MB; the last-level
// cache holds 256 MB)
constexpr double kCg1CacheBytes = 150e6;
// tile of the recomputing single-reduction kernel (k_cg2_q4_tile)
#ifndef PF_CG2_TI
#define PF_CG2_TI 16
#endif
#ifndef PF_CG2_TJ
#define PF_CG2_TJ 32
#endif
constexpr int kCg2TI = PF_CG2_TI, kCg2TJ = PF_CG2_TJ;

// Launch shape of the quad4 operator kernel: tiles, and workgroups (a
// multiple of 8, one group per XCD), one tile each (several tiles per
// workgroup with the next tile's loads in flight measured slower).
struct K1Shape {
    int tilesJ, ntiles;
    unsigned grid;
};
constexpr int k1_tiles_per_block() { return 1; }
K1Shape k1_shape(int nx, int ny) {
    K1Shape sh;
    sh.tilesJ = (ny + 1 + kTileJ - 1) / kTileJ;
    sh.ntiles = sh.tilesJ * ((nx + 1 + kTileI - 1) / kTileI);
    const int per = (sh.ntiles + 7) / 8;
    const int tpb = k1_tiles_per_block();
    sh.grid = 8u * (unsigned)((per + tpb - 1) / tpb);
    return sh;
}

// Hex8 K1 with the fused p update (k_pcg_k1_h8_tile): kH8Slab-node slabs of a
// node plane, chunks of PF_H8_PLANES planes per workgroup (doubled until the
// grid fits the reduction scratch).  per == 0: the plane is too long for the
// kernel's registers (nz > 211), and the three-launch form runs instead.
#ifndef PF_H8_PLANES
#define PF_H8_PLANES 4
#endif
struct H8Shape {
    int nslab, planes, nwork, per;
    unsigned grid;
    size_t lds;
    // the operator on MFMA (k_pcg_k1_h8_mfma): mJ node lines per workgroup,
    // mnjb line blocks, chunks of mplanes node planes, one work item per
    // (chunk, line block); mJ = 0: not selected or the plane does not fit
    int mJ, mnjb, mplanes, mnwork;
    unsigned mgrid;
    size_t mlds;
    bool fused() const { return per || mJ; }             // K1 in one launch
    unsigned k1grid() const { return mJ ? mgrid : grid; }  // K1's partials
};
// Node lines per workgroup of k_pcg_k1_h8_mfma: the J (at most 8, LDS within
// 64 KB, a plane's range within the kernel's registers) with the fewest batch
// rounds over a plane, counting a colour's batches in rounds of the
// workgroup's waves.  Planes per workgroup: the chunk length with the least
// per-CU work, counting a workgroup's plane loads (its planes and the two
// halo planes) in rounds of the 256 CUs.
constexpr int kH8mPerMax = 12;
constexpr int kH8mThreads = 512;  // eight waves share a colour's batches
void h8m_pick(const pf_ctx* ctx, size_t tsize, H8Shape& sh) {
    long best = -1;
    for (int J = 1; J <= 8; J++) {
        const size_t bytes = (size_t)h8m_lds_entries(J, ctx->nz) * tsize;
        const int njb = (ctx->ny + J) / J;
        const long nv = 3L * (J + 2) * (ctx->nz + 1);  // one plane's range
        if (bytes > 65536 || nv > kH8mThreads * kH8mPerMax || (long)(J + 1) * ctx->nz > 2 * kH8mThreads ||
            3L * J * (ctx->nz + 1) > 4 * kH8mThreads)
            continue;
        long rounds = 0;
        for (int pj = 0; pj < 2; pj++)
            for (int pk = 0; pk < 2; pk++) {
                const int nl = (J + 1 - pj + 1) / 2;  // element lines of parity pj in a full block
                const int nbl = ((ctx->nz - pk + 1) / 2 + 15) / 16;
                rounds += (nl * nbl + kH8mThreads / 64 - 1) / (kH8mThreads / 64);
            }
        const long cost = rounds * njb;
        if (best < 0 || cost < best) {
            best = cost;
            sh.mJ = J;
            sh.mnjb = njb;
            sh.mlds = bytes;
        }
    }
    if (!sh.mJ) return;
    long bestc = -1;
    for (int P = 1; P <= 16; P++) {
        const long nwork = (long)sh.mnjb * ((ctx->nx + 1 + P - 1) / P);
        const long grid = 8 * ((nwork + 7) / 8);
        if (grid > kMaxPartials) continue;
        const long cost = ((nwork + 255) / 256) * (P + 2);
        if (bestc < 0 || cost < bestc) {
            bestc = cost;
            sh.mplanes = P;
            sh.mnwork = (int)nwork;
            sh.mgrid = (unsigned)grid;
        }
    }
    if (bestc < 0) sh.mJ = 0;
}
H8Shape h8_shape(const pf_ctx* ctx, size_t tsize) {
    H8Shape sh{};
    const long pl = (long)(ctx->ny + 1) * (ctx->nz + 1);
    const int nv = 3 * (kH8Slab + 2 * (ctx->nz + 2));
    sh.per = nv <= 5 * 256 ? 5 : (nv <= 8 * 256 ? 8 : 0);
    sh.nslab = (int)((pl + kH8Slab - 1) / kH8Slab);
    sh.planes = PF_H8_PLANES;
    for (;;) {
        const long nwork = (long)sh.nslab * ((ctx->nx + 1 + sh.planes - 1) / sh.planes);
        const long grid = 8 * ((nwork + 7) / 8);
        if (grid <= kMaxPartials || sh.planes > ctx->nx) {
            sh.nwork = (int)nwork;
            sh.grid = (unsigned)grid;
            break;
        }
        sh.planes *= 2;
    }
    if (sh.grid > (unsigned)kMaxPartials || !ctx->d_K0g) sh.per = 0;
    sh.lds = (size_t)3 * nv * tsize;
    if (ctx->h8_op == PF_H8_OP_MFMA && ctx->d_K0m) h8m_pick(ctx, tsize, sh);
    return sh;
}

// workgroups of the streaming PCG vector kernel (few, so that the operator
// kernel's redundant read of its partials stays small)
constexpr int k2_cap() { return 512; }

unsigned gsize(long n) { return (unsigned)std::max(1L, std::min((long)grid_cap(), (n + kBlock - 1) / kBlock)); }
// gsize rounded up to a multiple of 8, for kernels that split their range
// XCD-contiguously (xcd_block_range)
unsigned gsize8(long n) { return (gsize(n) + 7u) & ~7u; }

template <class T>
int dalloc(pf_ctx* ctx, T** p, long n) {
    if (*p) {
        hipFree(*p);
        *p = nullptr;
    }
    if (n <= 0) return PF_OK;
    hipError_t e = hipMalloc((void**)p, sizeof(T) * (size_t)n);
    if (e != hipSuccess) {
        ctx->err = std::string("hipMalloc: ") + hipGetErrorString(e);
        *p = nullptr;
        return PF_ERR_NOMEM;
    }
    return PF_OK;
}

template <class T>
void dfree(T*& p) {
    if (p) hipFree(p);
    p = nullptr;
}

int set_device(pf_ctx* ctx) {
    PF_HIP(hipSetDevice(ctx->device));
    return PF_OK;
}

int sync(pf_ctx* ctx) {
    PF_HIP(hipStreamSynchronize(ctx->stream));
    return PF_OK;
}

int check_launch(pf_ctx* ctx) {
    PF_HIP(hipGetLastError());
    return PF_OK;
}

bool is2d(pf_ctx* ctx) { return ctx->dim == 2; }
void release_net(pf_ctx* ctx);
G3 g3(pf_ctx* ctx) { return G3{ctx->nx, ctx->ny, ctx->nz}; }

// the hex8 multigrid's finest level runs k_mg3_residual0_tile on this shape
struct Mg3KeTile {
    const H8Shape* sh;
};

template <class T>
void launch_h8_k1_tile(pf_ctx* ctx, const H8Shape& sh, int k, const T* pold, const T* z, T* pnew, T* q, const T* Ev,
                       const T* Kg, const double* partB, int nbB, double* partA, PcgDev* S, double eps) {
    if (sh.mJ) {
        const T* Ka = std::is_same<T, float>::value ? (const T*)ctx->d_K0mf : (const T*)ctx->d_K0m;
        const long nv = 3L * (sh.mJ + 2) * (ctx->nz + 1);
        auto go = [&](auto kern) {
            kern<<<sh.mgrid, kH8mThreads, sh.mlds, ctx->stream>>>(g3(ctx), sh.mJ, sh.mnjb, sh.mplanes, sh.mnwork, k,
                                                                   pold, z, pnew, q, Ev, Ka, ctx->d_fix, partB, nbB,
                                                                   partA, S, eps);
        };
        if (nv <= kH8mThreads * 4)
            go(k_pcg_k1_h8_mfma<T, 4, kH8mThreads>);
        else if (nv <= kH8mThreads * 7)
            go(k_pcg_k1_h8_mfma<T, 7, kH8mThreads>);
        else
            go(k_pcg_k1_h8_mfma<T, kH8mPerMax, kH8mThreads>);
    } else if (sh.per == 5)
        k_pcg_k1_h8_tile<T, 5><<<sh.grid, kBlock, sh.lds, ctx->stream>>>(
            g3(ctx), sh.nslab, sh.planes, sh.nwork, k, pold, z, pnew, q, Ev, Kg, ctx->d_fix, partB, nbB, partA, S, eps);
    else
        k_pcg_k1_h8_tile<T, 8><<<sh.grid, kBlock, sh.lds, ctx->stream>>>(
            g3(ctx), sh.nslab, sh.planes, sh.nwork, k, pold, z, pnew, q, Ev, Kg, ctx->d_fix, partB, nbB, partA, S, eps);
}

void mg_free(pf_ctx* ctx);
void free_grid(pf_ctx* ctx) {
    mg_free(ctx);
    dfree(ctx->d_n2g); dfree(ctx->d_g2n); dfree(ctx->d_fix);
    dfree(ctx->d_rho); dfree(ctx->d_E); dfree(ctx->d_Ef);
    dfree(ctx->d_x); dfree(ctx->d_r); dfree(ctx->d_z); dfree(ctx->d_q); dfree(ctx->d_p0); dfree(ctx->d_p1);
    dfree(ctx->d_D); dfree(ctx->d_b); dfree(ctx->d_t0); dfree(ctx->d_t1);
    dfree(ctx->f_x); dfree(ctx->f_r); dfree(ctx->f_z); dfree(ctx->f_q); dfree(ctx->f_p0); dfree(ctx->f_p1);
    dfree(ctx->d_s0); dfree(ctx->d_s1); dfree(ctx->f_s0); dfree(ctx->f_s1); dfree(ctx->d_Dinv);
    dfree(ctx->f_D); dfree(ctx->f_b);
    dfree(ctx->res_halo);
    dfree(ctx->res_loc);
    ctx->res_halo_n = ctx->res_loc_n = 0;
    if (ctx->res_backoff) ctx->res_pause = ctx->res_backoff = 0;
    dfree(ctx->d_e0); dfree(ctx->d_e1); dfree(ctx->d_e2); dfree(ctx->d_e3); dfree(ctx->d_e4); dfree(ctx->d_e5);
    dfree(ctx->d_e6);
    dfree(ctx->d_cg); dfree(ctx->d_load);
    dfree(ctx->d_indptr); dfree(ctx->d_indices); dfree(ctx->d_data); dfree(ctx->d_ke_all);
    dfree(ctx->d_fptr); dfree(ctx->d_fidx); dfree(ctx->d_fw);
    ctx->nnz = -1;
    ctx->N = 0;
    ctx->have_E = false;
    ctx->have_filter = false;
    ctx->have_lists = false;
    dfree(ctx->d_fcol);
    ctx->fcol_n = 0;
    ctx->have_fcol = false;
    release_net(ctx);
}

int alloc_grid(pf_ctx* ctx) {
    long nv = ctx->nv, ne = ctx->ne, nn = ctx->nn;
    PF_TRY(dalloc(ctx, &ctx->d_fix, nn));
    PF_TRY(dalloc(ctx, &ctx->d_n2g, nv));
    PF_TRY(dalloc(ctx, &ctx->d_rho, ne));
    PF_TRY(dalloc(ctx, &ctx->d_E, ne));
    PF_TRY(dalloc(ctx, &ctx->d_Ef, ne));
    double** dv[] = {&ctx->d_x, &ctx->d_r, &ctx->d_z, &ctx->d_q, &ctx->d_p0, &ctx->d_p1, &ctx->d_D, &ctx->d_b,
                     &ctx->d_t0, &ctx->d_t1, &ctx->d_load, &ctx->d_s0, &ctx->d_s1, &ctx->d_Dinv};
    for (double** p : dv) PF_TRY(dalloc(ctx, p, nv));
    float** fv[] = {&ctx->f_x, &ctx->f_r, &ctx->f_z, &ctx->f_q, &ctx->f_p0, &ctx->f_p1, &ctx->f_D, &ctx->f_b,
                    &ctx->f_s0, &ctx->f_s1};
    for (float** p : fv) PF_TRY(dalloc(ctx, p, nv));
    double** de[] = {&ctx->d_e0, &ctx->d_e1, &ctx->d_e2, &ctx->d_e3, &ctx->d_e4, &ctx->d_e5, &ctx->d_e6};
    for (double** p : de) PF_TRY(dalloc(ctx, p, ne));
    PF_TRY(dalloc(ctx, &ctx->d_cg, ne * ctx->dim));
    PF_HIP(hipMemsetAsync(ctx->d_load, 0, sizeof(double) * nv, ctx->stream));
    PF_HIP(hipMemsetAsync(ctx->d_fix, 0, nn, ctx->stream));
    return PF_OK;
}

// Host rule of SetDirichlet + Renumbering (BoundaryCondition.h:19-25,
// Assembling.h:175-186), uploaded with the inverse map and fixity bits.
int upload_dofmap(pf_ctx* ctx, const std::vector<uint8_t>& fix) {
    long nv = ctx->nv;
    ctx->h_n2g.assign(nv, 0);
    std::vector<int32_t> g2n;
    g2n.reserve(nv);
    int N = 0;
    for (long n = 0; n < ctx->nn; n++)
        for (int d = 0; d < ctx->ndpn; d++) {
            long idx = n * ctx->ndpn + d;
            if (fix[n] & (1u << d)) {
                ctx->h_n2g[idx] = -1;
            } else {
                ctx->h_n2g[idx] = N++;
                g2n.push_back((int32_t)idx);
            }
        }
    ctx->N = N;
    PF_TRY(dalloc(ctx, &ctx->d_g2n, std::max(N, 1)));
    PF_HIP(hipMemcpyAsync(ctx->d_n2g, ctx->h_n2g.data(), sizeof(int32_t) * nv, hipMemcpyHostToDevice, ctx->stream));
    if (N > 0)
        PF_HIP(hipMemcpyAsync(ctx->d_g2n, g2n.data(), sizeof(int32_t) * N, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_fix, fix.data(), ctx->nn, hipMemcpyHostToDevice, ctx->stream));
    ctx->nnz = -1;
    return sync(ctx);
}

// need_E: the matrix-free operators (element matrix and moduli); the
// assembled-CSR operator needs only the grid and the DOF map.
int require_ready(pf_ctx* ctx, bool need_E) {
    PF_CHECK(ctx->dim == 2 || ctx->dim == 3, PF_ERR_STATE, "no grid: call pf_grid2d/pf_grid3d first");
    PF_CHECK(ctx->N > 0, PF_ERR_STATE, "no DOF map: call pf_set_dirichlet first");
    if (need_E) {
        PF_CHECK(!ctx->h_K0.empty(), PF_ERR_STATE, "no element matrix: call pf_set_element_matrix first");
        PF_CHECK(ctx->have_E, PF_ERR_STATE, "no element moduli: call pf_set_density or pf_set_moduli first");
    }
    return PF_OK;
}

// ------------------------------------------------------------ operators ---
int apply_nodal(pf_ctx* ctx, bool f32, const void* x, void* y, bool mask) {
    if (is2d(ctx)) {
        if (f32)
            k_apply_q4<float><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, (const float*)x, (float*)y,
                                                                        ctx->d_Ef, ctx->d_K0f, ctx->d_fix, mask);
        else
            k_apply_q4<double><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, (const double*)x,
                                                                         (double*)y, ctx->d_E, ctx->d_K0, ctx->d_fix,
                                                                         mask);
        return check_launch(ctx);
    }
    if (f32)
        k_apply_h8<float><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), (const float*)x, (float*)y, ctx->d_Ef,
                                                                    ctx->d_K0f, ctx->d_fix, mask, nullptr, nullptr);
    else
        k_apply_h8<double><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), (const double*)x, (double*)y,
                                                                     ctx->d_E, ctx->d_K0, ctx->d_fix, mask, nullptr,
                                                                     nullptr);
    return check_launch(ctx);
}

int diag_nodal(pf_ctx* ctx, bool f32) {
    if (is2d(ctx)) {
        if (f32)
            k_diag_q4<float><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->d_Ef, ctx->d_K0f,
                                                                       ctx->d_fix, ctx->f_D);
        else
            k_diag_q4<double><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->d_E, ctx->d_K0,
                                                                        ctx->d_fix, ctx->d_D);
        return check_launch(ctx);
    }
    if (f32)
        k_diag_h8<float><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->d_Ef, ctx->d_K0f, ctx->d_fix,
                                                                   ctx->f_D);
    else
        k_diag_h8<double><<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->d_E, ctx->d_K0, ctx->d_fix,
                                                                    ctx->d_D);
    return check_launch(ctx);
}

int to_nodal(pf_ctx* ctx, const double* xf_dev, double* xn_dev) {
    PF_HIP(hipMemsetAsync(xn_dev, 0, sizeof(double) * ctx->nv, ctx->stream));
    k_free_to_nodal<<<nblocks(ctx->N), kBlock, 0, ctx->stream>>>(ctx->N, ctx->d_g2n, xf_dev, xn_dev);
    return check_launch(ctx);
}

int to_free(pf_ctx* ctx, const double* xn_dev, double* xf_dev) {
    k_nodal_to_free<<<nblocks(ctx->N), kBlock, 0, ctx->stream>>>(ctx->N, ctx->d_g2n, xn_dev, xf_dev);
    return check_launch(ctx);
}

// ---------------------------------------------------------------- PCG -----
struct PcgRun {
    int iterations = 0, status = 0;
    double rnorm = 0, bnorm = 0;
};

// Jacobi-PCG on device vectors: nodal (EbE, n = nv) or free-numbered (CSR,
// n = N).  b, x, D are of the matching layout; x receives the solution.
// Optional capture of (x_k) during a solve: every `every` chunks the iterate
// is copied (stream-ordered) into slot `count` of `xs` (nv doubles each).
struct SnapHook {
    int every = 0, max = 0, count = 0;
    double* xs = nullptr;
    std::vector<int> iters;
};

// Two events (no timing), destroyed on every return path.
struct EventPair {
    hipEvent_t e[2] = {nullptr, nullptr};
    hipError_t create() {
        hipError_t r = hipEventCreateWithFlags(&e[0], hipEventDisableTiming);
        return r != hipSuccess ? r : hipEventCreateWithFlags(&e[1], hipEventDisableTiming);
    }
    hipEvent_t& operator[](int i) { return e[i]; }
    ~EventPair() {
        for (hipEvent_t x : e)
            if (x) hipEventDestroy(x);
    }
};

// ------------------------------------------------- resident solves -----
// Tiles of a resident solve: gi x gj workgroups of nt threads, S node rows
// per thread.  gi == 0: the grid does not fit.
struct ResShape {
    int gi = 0, gj = 0, nt = 0, S = 0;
    size_t lds = 0;
};
constexpr size_t kResLds = 150 * 1024;  // of a CU's 160 KB, beside the static part
constexpr int kResConfigs[][2] = {{256, 1}, {256, 2}, {512, 2}, {512, 4}, {512, 5}};

// The tiling with the least estimated time per iteration, in microseconds over
// what every tiling pays: 0.0012 per node (with the rows that pad a tile to S),
// up to half as much again where a wave spans several short tile rows (LDS
// conflicts: 1024x512 as 16x16 tiles of 65x33 nodes 7.2, as 32x8 of 33x65
// 6.1), 0.003 per halo node pair, 0.4 for the longer pause of more than 64
// workgroups (res_pause), and 1.2 less for a single one, which waits for nobody (31x15:
// 2.0 against 3.1).
template <class T>
ResShape res_pick(const pf_ctx* ctx) {
    ResShape best;
    double bestc = 0.0;
    const int ni = ctx->nx + 1, nj = ctx->ny + 1;
    for (const auto& cfg : kResConfigs) {
        const int nt = cfg[0], S = cfg[1];
        for (int gi = 1; gi <= std::min(ni, ctx->res_wgs); gi++)
            for (int gj = 1; gj <= std::min(nj, ctx->res_wgs / gi); gj++) {
                const int ti = (ni + gi - 1) / gi, tj = (nj + gj - 1) / gj;
                const int rows = (ti + S - 1) / S * S;
                const size_t lds = res_lds_bytes<T>(ti, tj, S, nt);
                if (rows / S * tj > nt || 2 * (tj + 2) + 2 * ti > nt || lds > kResLds) continue;
                const double split = std::min(1.0, std::max(0.0, 64.0 / tj - 1.0));
                const double cost = 0.0012 * rows * tj * (1.0 + 0.5 * split) + 0.003 * (ti + tj) + 0.0002 * S * nt +
                                    (gi * gj == 1 ? -1.2 : gi * gj > 64 ? 0.4 : 0.0);
                if (best.gi == 0 || cost < bestc) {
                    bestc = cost;
                    best.gi = gi;
                    best.gj = gj;
                    best.nt = nt;
                    best.S = S;
                    best.lds = lds;
                }
            }
    }
    return best;
}

template <class T, bool SR>
const void* res_kernel(const ResShape& sh) {
#define PF_RES_CASE(NT_, S_) \
    if (sh.nt == NT_ && sh.S == S_) return (const void*)k_pcg_q4_resident<T, S_, NT_, SR>;
    PF_RES_CASE(256, 1)
    PF_RES_CASE(256, 2)
    PF_RES_CASE(512, 2)
    PF_RES_CASE(512, 4)
    PF_RES_CASE(512, 5)
#undef PF_RES_CASE
    return nullptr;
}

// whether this context's solves and updates may run resident
bool res_on(const pf_ctx* ctx) {
    return ctx->res_wgs >= 1 && ctx->res_mode != PF_RESIDENT_OFF && ctx->res_pause == 0;
}
// At the start of a solve, update or bisection that may: one call less to wait
// after a stall.
void res_enter(pf_ctx* ctx) {
    if (ctx->res_pause > 0) ctx->res_pause--;
}
// Before launch number `launch` of a resident solve: PF_RESIDENT_STALL's flag.
void res_force(pf_ctx* ctx, int launch) {
    if (ctx->res_mode == PF_RESIDENT_STALL && launch >= ctx->res_after) k_res_stall<<<1, 1, 0, ctx->stream>>>(ctx->d_res);
}
// After a resident launch (h_res copied back): whether a workgroup gave up.  The
// next call is then launched, after a second stall in a row the next two, and
// so on up to 1024: what keeps the GPU busy may end, and a stall costs 2 s.
bool res_gave_up(pf_ctx* ctx) {
    if (!ctx->h_res->stall) return false;
    ctx->res_backoff = std::min(1024, std::max(1, 2 * ctx->res_backoff));
    ctx->res_pause = ctx->res_backoff + 1;  // res_enter of the call that tries again takes the last one
    ctx->res_gave++;
    return true;
}
void res_ended(pf_ctx* ctx) {
    ctx->res_backoff = 0;
    ctx->res_done++;
}
// A cooperative launch.  Refused (false), the next 1024 calls are launched: the
// runtime takes 40 ms to refuse (a 16x8 solve takes 2 ms launched), and it does
// so as long as another process that has made such a launch lives.
bool res_launch(pf_ctx* ctx, const void* kern, unsigned wgs, int nt, void** args, size_t lds) {
    if (ctx->res_mode != PF_RESIDENT_REFUSED) {
        if (hipLaunchCooperativeKernel(kern, dim3(wgs), dim3(nt), args, (unsigned)lds, ctx->stream) == hipSuccess)
            return true;
        (void)hipGetLastError();
    }
    ctx->res_backoff = 0;  // not a stall: a new grid does not end the pause
    ctx->res_pause = 1024 + 1;
    ctx->res_gave++;
    return false;
}

constexpr int kResChunk = 2048;  // iterations per launch: other streams get the GPU in between

// A buffer that only a resident kernel needs, of at least n values (*have: its
// size); false when it cannot be had, which is no error: the launched kernels
// do without.
template <class T>
bool res_alloc(pf_ctx* ctx, T** p, long n, long* have) {
    if (*have >= n) return true;
    dfree(*p);
    *have = 0;
    if (ctx->res_mode == PF_RESIDENT_NOMEM) {
        if (ctx->res_after <= 0) return false;
        ctx->res_after--;
    }
    if (hipMalloc((void**)p, sizeof(T) * (size_t)n) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return false;
    }
    *have = n;
    return true;
}

// Before a launch, none of whose words are read by the next one: no word may
// carry a tag that is still to come (a launch takes at most 5.2 million tags).
void res_tags(pf_ctx* ctx) {
    if (ctx->res_tag <= 0xf0000000u) return;
    k_fill<u64><<<gsize(ctx->res_halo_n), kBlock, 0, ctx->stream>>>(ctx->res_halo_n, ctx->res_halo, 0ull);
    k_fill<u64><<<1, kBlock, 0, ctx->stream>>>(2L * 4 * kResMaxWg * 2, ctx->res_slots, 0ull);
    ctx->res_tag = 1;
}

// Exchange buffer of `words` words for a solve that starts now, and the
// solve's scalars; *ok false: it cannot be had.
int res_begin(pf_ctx* ctx, long words, bool* ok) {
    const bool fresh = ctx->res_halo_n < words;
    *ok = res_alloc(ctx, &ctx->res_halo, words, &ctx->res_halo_n);
    if (!*ok) return PF_OK;
    if (fresh) ctx->res_tag = 0xffffffffu;  // whatever the new words hold
    res_tags(ctx);
    k_res_start<<<1, 1, 0, ctx->stream>>>((PcgDev*)ctx->d_pcg, ctx->d_res);
    return check_launch(ctx);
}

// Launches `kern` (cooperatively) over iterations 0 .. end in chunks until the
// solve is done; *ran is false, and nothing has been solved, when the launch
// cannot be made or stalled: the caller then launches per iteration.
template <class ARGS>
int res_run(pf_ctx* ctx, const void* kern, int wgs, int nt, size_t lds, ARGS& A, long end, PcgRun& out, bool* ran) {
    A.slots = ctx->res_slots;
    A.S = (PcgDev*)ctx->d_pcg;
    A.R = ctx->d_res;
    A.fix = ctx->d_fix;
    const PcgDev* H = (const PcgDev*)ctx->h_pcg;
    int launch = 0;
    for (long m = 0;;) {
        res_tags(ctx);
        res_force(ctx, launch++);
        A.m0 = (int)m;
        A.m1 = (int)std::min(end, m + kResChunk);
        A.last = A.m1 == end;
        A.tag = ctx->res_tag;
        ctx->res_tag += 2 * (A.m1 - A.m0) + 2;
        void* args[] = {&A};
        if (!res_launch(ctx, kern, wgs, nt, args, lds)) return PF_OK;
        PF_HIP(hipMemcpyAsync(ctx->h_pcg, A.S, sizeof(PcgDev), hipMemcpyDeviceToHost, ctx->stream));
        PF_HIP(hipMemcpyAsync(ctx->h_res, ctx->d_res, sizeof(ResDev), hipMemcpyDeviceToHost, ctx->stream));
        PF_TRY(sync(ctx));
        if (res_gave_up(ctx)) return PF_OK;
        m = A.m1;
        if (H->done || m >= end) break;
    }
    *ran = true;
    res_ended(ctx);
    out.iterations = H->iterations;
    out.status = H->status;
    out.rnorm = H->rnorm;
    out.bnorm = H->bnorm;
    return PF_OK;
}

// LDS beyond the default limit; false: the kernel cannot have it
bool res_lds_ok(const void* kern, size_t lds) {
    if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

// Jacobi-PCG on a quad4 grid resident on the chip (k_pcg_q4_resident); *ran as
// in res_run, also false when the grid does not fit.  D: the diagonal, or its
// inverse for the single-reduction form (sr).
template <class T>
int pcg_resident(pf_ctx* ctx, bool sr, const T* b, T* x, const T* D, T* r, T* s, T* p, T* w, double eps, int itrmax,
                 PcgRun& out, bool* ran) {
    *ran = false;
    if (!res_on(ctx)) return PF_OK;
    const ResShape sh = res_pick<T>(ctx);
    if (!sh.gi) return PF_OK;
    const void* kern = sr ? res_kernel<T, true>(sh) : res_kernel<T, false>(sh);
    if (!res_lds_ok(kern, sh.lds)) return PF_OK;
    bool ok;
    PF_TRY(res_begin(ctx, 2 * ctx->nn * 4, &ok));
    if (!ok) return PF_OK;
    const bool f32 = std::is_same<T, float>::value;
    ResArgs<T> A{};
    A.nx = ctx->nx; A.ny = ctx->ny; A.gi = sh.gi; A.gj = sh.gj;
    A.b = b; A.D = D;
    A.E = f32 ? (const T*)ctx->d_Ef : (const T*)ctx->d_E;
    A.K0 = f32 ? (const T*)ctx->d_K0f : (const T*)ctx->d_K0;
    A.x = x; A.r = r; A.s = s; A.p = p; A.w = w;
    A.halo = ctx->res_halo;
    A.eps = eps;
    const long end = std::max(itrmax, 0);  // pf_simp_run takes any cg_itrmax; the tags must go up
    // sr: step m finishes iterate m
    return res_run(ctx, kern, sh.gi * sh.gj, sh.nt, sh.lds, A, sr ? end + 1 : end, out, ran);
}

// Boxes of a hex8 resident solve.  gi == 0: the grid does not fit.
struct Res3Shape {
    int gi = 0, gj = 0, gk = 0, slots = 0, box = 0, fb[3] = {0, 0, 0};
    size_t lds = 0;
};
// The split with the least estimated time per iteration in microseconds:
// 1.5 per pass over a layer of each half box (two waves per SIMD from 9 element
// rows on), 0.001 per node value, 1.8 per split axis (an exchange), 0.0008 per
// exchanged face value.  60x30x30: 30x4x2 boxes 13.2, 15x4x4 15.0, 12x3x3 21.0;
// 128x64x64: 16x4x4 31.6, 8x8x4 39 to 44.  Values per thread: 4 while they
// suffice, else 16, the most that a box of 16 x 16 rows and 8 layers has; sizes
// between (80x40x40 has 5, 100x40x40 6, 100x50x50 10) pay for 16: 25.5, 26.5 and
// 31.6 us, launched 48.7, 48.7 and 55.8.
template <class T>
Res3Shape res3_pick(const pf_ctx* ctx) {
    Res3Shape best;
    double bestc = 0.0;
    for (int gi = 1; gi <= std::min(ctx->nx, ctx->res_wgs); gi++)
        for (int gj = 1; gj <= std::min(ctx->ny, ctx->res_wgs / gi); gj++)
            for (int gk = 1; gk <= std::min(ctx->nz, ctx->res_wgs / (gi * gj)); gk++) {
                const int ei = (ctx->nx + gi - 1) / gi, ej = (ctx->ny + gj - 1) / gj, ek = (ctx->nz + gk - 1) / gk;
                const int di = ei + 1, dj = ej + 1, dk = ek + 1;
                const long nv = 3L * di * dj * dk;
                if (ej > 16 || ek > 16 || nv > kRes3Threads * kRes3Slots) continue;
                int box = 0, most = 0, fb[3];
                for (int ax = 0; ax < 3; ax++) {
                    const int F = res3_face(ax, di, dj, dk);
                    fb[ax] = box;
                    box += 2 * F * (int)(sizeof(T) / 4);
                    most = std::max(most, 2 * F);
                }
                if (most > kRes3Threads * kRes3Items) continue;
                double cost = 1.5 * ((ei + 1) / 2 + 1) * (ej > 8 ? 1.5 : 1.0) + 0.001 * nv;
                const int gd[3] = {gi, gj, gk};
                for (int ax = 0; ax < 3; ax++)
                    if (gd[ax] > 1) cost += 1.8 + 0.0008 * 2 * res3_face(ax, di, dj, dk);
                if (best.gi && cost >= bestc) continue;
                bestc = cost;
                best.gi = gi;
                best.gj = gj;
                best.gk = gk;
                best.slots = nv <= kRes3Threads * 4 ? 4 : kRes3Slots;
                best.box = box;
                std::copy(fb, fb + 3, best.fb);
                best.lds = sizeof(T) * 2 * kRes3Threads * best.slots;
            }
    return best;
}

bool res3_applies(const pf_ctx* ctx) {
    return res_on(ctx) && ctx->d_K0p && ctx->h8_op == PF_H8_OP_AUTO;
}

// The same for hex8 (k_pcg_h8_resident), ScalingCG's order; only for an
// element matrix with parity blocks and the default operator.
template <class T>
int pcg_resident3(pf_ctx* ctx, const T* b, T* x, const T* D, T* r, T* p, double eps, int itrmax, PcgRun& out,
                  bool* ran) {
    *ran = false;
    if (!res3_applies(ctx)) return PF_OK;
    const Res3Shape sh = res3_pick<T>(ctx);
    if (!sh.gi) return PF_OK;
    const void* kern = sh.slots == 4 ? (const void*)k_pcg_h8_resident<T, 4>
                                     : (const void*)k_pcg_h8_resident<T, kRes3Slots>;
    if (!res_lds_ok(kern, sh.lds)) return PF_OK;
    const int wgs = sh.gi * sh.gj * sh.gk;
    const long local = (long)wgs * kRes3Threads * sh.slots;  // x of every workgroup's values
    bool ok;
    PF_TRY(res_begin(ctx, 2L * wgs * sh.box, &ok));
    if (!ok || !res_alloc(ctx, &ctx->res_loc, local, &ctx->res_loc_n)) return PF_OK;
    const bool f32 = std::is_same<T, float>::value;
    Res3Args<T> A{};
    A.nx = ctx->nx; A.ny = ctx->ny; A.nz = ctx->nz;
    A.gi = sh.gi; A.gj = sh.gj; A.gk = sh.gk;
    A.box = sh.box;
    std::copy(sh.fb, sh.fb + 3, A.fb);
    A.b = b; A.D = D;
    A.E = f32 ? (const T*)ctx->d_Ef : (const T*)ctx->d_E;
    A.Kp = f32 ? (const T*)ctx->d_K0pf : (const T*)ctx->d_K0p;
    A.x = x; A.r = r; A.p = p;
    A.edge = ctx->res_halo;
    A.loc = (T*)ctx->res_loc;
    A.eps = eps;
    return res_run(ctx, kern, wgs, kRes3Threads, sh.lds, A, std::max(itrmax, 0), out, ran);
}

// Workgroups of k_cg1_q4_tile: full tiles, then edge tiles (launched first).
Cg1Tiles cg1_tiles(const pf_ctx* ctx, unsigned* grid, int ti = kCg1TI, int tj = kCg1TJ) {
    Cg1Tiles G;
    G.fullI = (ctx->nx + 1) / ti;
    G.fullJ = (ctx->ny + 1) / tj;
    G.tilesI = (ctx->nx + 1 + ti - 1) / ti;
    G.tilesJ = (ctx->ny + 1 + tj - 1) / tj;
    G.perF = (G.fullI * G.fullJ + 7) / 8;
    G.nEdgePad = 8 * ((G.tilesI * G.tilesJ - G.fullI * G.fullJ + 7) / 8);
    G.edgeFirst = 1;
    *grid = (unsigned)(8 * G.perF + G.nEdgePad);
    return G;
}

// Single-reduction forms on quad4 grids, one launch per iteration.
// Carried (k_cg1_q4_tile): x and p in place; r, w = K u and s = K p each in
// two buffers that alternate between launches (r|z, p1|q, s0|s1).
// Recomputed (k_cg2_q4_tile): x in place; r and p alternate (r|z, p1|q).
// Both scale by 1/D (d_Dinv, formed at the start of each solve), and both
// update x in the even launches only (k_cg_x_fix completes an odd last one).
template <class T>
int pcg_device_cg1(pf_ctx* ctx, const T* b, T* x, const T* D, T* r, T* z, T* p0, T* p1, T* q, double eps,
                   int itrmax, PcgRun& out) {
    PcgDev* S = (PcgDev*)ctx->d_pcg;
    double* part[2] = {ctx->red.partials, ctx->red.partials + 3 * kMaxPartials};
    unsigned g1;
    // carried kernel: r, w, s (two buffers each), p, x, 1/D and the moduli
    const double carried = 8.0 * (9.0 * ctx->nv + ctx->ne);
    const bool kp = ctx->pcg_form == PF_PCG_SINGLE_REDUCTION_RECOMPUTED ||
                    (ctx->pcg_form == PF_PCG_SINGLE_REDUCTION && carried > kCg1CacheBytes);
    const Cg1Tiles G = kp ? cg1_tiles(ctx, &g1, kCg2TI, kCg2TJ) : cg1_tiles(ctx, &g1);
    PF_CHECK(g1 <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    const bool f32 = std::is_same<T, float>::value;
    const T* Ev = f32 ? (const T*)ctx->d_Ef : (const T*)ctx->d_E;
    const T* Kv = f32 ? (const T*)ctx->d_K0f : (const T*)ctx->d_K0;
    T* s0 = f32 ? (T*)ctx->f_s0 : (T*)ctx->d_s0;
    T* s1 = f32 ? (T*)ctx->f_s1 : (T*)ctx->d_s1;
    T* R[2] = {r, z};
    T* W[2] = {p1, q};
    T* Sv[2] = {s0, s1};
    T* Dinv = (T*)ctx->d_Dinv;
    k_recip<T><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, D, Dinv);
    if (ctx->pcg_form != PF_PCG_SINGLE_REDUCTION_RECOMPUTED) {
        bool ran;
        PF_TRY(pcg_resident<T>(ctx, true, b, x, Dinv, r, s0, p0, q, eps, itrmax, out, &ran));
        if (ran) return PF_OK;
    }
    k_cg1_start<<<1, 1, 0, ctx->stream>>>(S);
    PF_TRY(check_launch(ctx));
    const int chunk = 32;
    const int mmax = itrmax + 1;  // launch m finishes iterate m; iterate itrmax is the last
    int m = 0;
    EventPair ev;
    PF_HIP(ev.create());
    volatile int* hflag = (volatile int*)ctx->h_red;
    hflag[0] = hflag[1] = 0;
    int slot = 0, pending = 0;
    bool done = false;
    while (!done && m < mmax) {
        const int mend = std::min(mmax, m + chunk);
        for (; m < mend; m++) {
            const int c = m & 1, o = c ^ 1;
            if (kp) {
                Cg2Vecs<T> V{m == 0 ? b : R[o], W[o], R[c], W[c], x, Dinv};
                k_cg2_q4_tile<T, kCg2TI, kCg2TJ><<<g1, kBlock, 0, ctx->stream>>>(
                    ctx->nx, ctx->ny, G, m, V, Ev, Kv, ctx->d_fix, part[o], (int)g1, part[c], S, eps);
                continue;
            }
            Cg1Vecs<T> V{m == 0 ? b : R[o], W[o], Sv[o], R[c], W[c], Sv[c], p0, x, Dinv};
            if (c)
                k_cg1_q4_tile<T, kCg1TI, kCg1TJ, false><<<g1, kBlock, 0, ctx->stream>>>(
                    ctx->nx, ctx->ny, G, m, V, Ev, Kv, ctx->d_fix, part[o], (int)g1, part[c], S, eps);
            else
                k_cg1_q4_tile<T, kCg1TI, kCg1TJ, true><<<g1, kBlock, 0, ctx->stream>>>(
                    ctx->nx, ctx->ny, G, m, V, Ev, Kv, ctx->d_fix, part[o], (int)g1, part[c], S, eps);
        }
        PF_TRY(check_launch(ctx));
        PF_HIP(hipMemcpyAsync((void*)&hflag[slot], &S->done, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        PF_HIP(hipEventRecord(ev[slot], ctx->stream));
        if (pending) {
            PF_HIP(hipEventSynchronize(ev[slot ^ 1]));
            if (hflag[slot ^ 1]) done = true;
        }
        pending = 1;
        slot ^= 1;
    }
    PF_HIP(hipStreamSynchronize(ctx->stream));
    k_cg1_final<<<1, kBlock, 0, ctx->stream>>>(m, part[(m - 1) & 1], (int)g1, S, eps);
    // x is updated by the even launches: the odd last one's update (its p is
    // p0 in place, or W[1] where p alternates)
    k_cg_x_fix<T><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, kp ? W[1] : p0, x, S);
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(ctx->h_pcg, S, sizeof(PcgDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    const PcgDev* H = (const PcgDev*)ctx->h_pcg;
    out.iterations = H->iterations;
    out.status = H->status;
    out.rnorm = H->rnorm;
    out.bnorm = H->bnorm;
    return PF_OK;
}

template <class T>
int pcg_device(pf_ctx* ctx, bool csr, const T* b, T* x, const T* D, T* r, T* z, T* p0, T* p1, T* q, double eps,
               int itrmax, PcgRun& out, SnapHook* snap = nullptr) {
    // FP32 solves keep ScalingCG's order: with FP32 vectors the carried s = K p
    // drifts and the single-reduction form needs about a third more iterations
    if (!csr && is2d(ctx) && ctx->pcg_form != PF_PCG_SCALINGCG && !snap && std::is_same<T, double>::value)
        return pcg_device_cg1<T>(ctx, b, x, D, r, z, p0, p1, q, eps, itrmax, out);
    if (!csr && !snap) {
        bool ran;
        if (is2d(ctx)) PF_TRY(pcg_resident<T>(ctx, false, b, x, D, r, z, p0, q, eps, itrmax, out, &ran));
        else PF_TRY(pcg_resident3<T>(ctx, b, x, D, r, p0, eps, itrmax, out, &ran));
        if (ran) return PF_OK;
    }
    const long n = csr ? ctx->N : ctx->nv;
    PcgDev* S = (PcgDev*)ctx->d_pcg;
    double* partA = ctx->red.partials;
    double* partB = ctx->red.partials + 2 * kMaxPartials;
    const bool h8 = !csr && !is2d(ctx);
    const K1Shape sh = k1_shape(ctx->nx, ctx->ny);
    const H8Shape s8 = h8 ? h8_shape(ctx, sizeof(T)) : H8Shape{};
    const unsigned g1 = csr ? gsize(ctx->N) : (h8 ? (s8.fused() ? s8.k1grid() : gsize(ctx->nn)) : sh.grid);
    const unsigned g2 = std::min<unsigned>(gsize(n), (unsigned)k2_cap());
    PF_CHECK(g1 <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    k_pcg_init<T><<<g2, kBlock, 0, ctx->stream>>>(n, b, D, x, r, z, p0, partB, S);
    PF_TRY(check_launch(ctx));
    const int chunk = 32;
    int k = 0;
    // one chunk is kept in flight while the previous chunk's flag is read
    EventPair ev;
    PF_HIP(ev.create());
    volatile int* hflag = (volatile int*)ctx->h_red;  // two ints: done flags of chunks in flight
    hflag[0] = hflag[1] = 0;
    int slot = 0, pending = 0;
    bool done = false;
    auto enqueue_chunk = [&](int kend) -> int {
        for (; k < kend; k++) {
            T* pold = (k & 1) ? p1 : p0;
            T* pnew = (k & 1) ? p0 : p1;
            if (h8) {
                const T* Ev = std::is_same<T, float>::value ? (const T*)ctx->d_Ef : (const T*)ctx->d_E;
                const T* Kv = std::is_same<T, float>::value ? (const T*)ctx->d_K0f : (const T*)ctx->d_K0;
                if (s8.fused()) {
                    const T* Kg = std::is_same<T, float>::value ? (const T*)ctx->d_K0gf : (const T*)ctx->d_K0g;
                    launch_h8_k1_tile<T>(ctx, s8, k, pold, z, pnew, q, Ev, Kg, partB, (int)g2, partA, S, eps);
                    k_pcg_k2<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, x, r, z, pnew, q, D, partA, (int)g1, partB, S);
                    continue;
                }
                // three launches: p = beta p + z in place (head + convergence), q = K p, update
                k_pcg_k3<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, p0, z, partB, (int)g2, S, eps);
                k_pcg_k1_h8<T><<<g1, kBlock, 0, ctx->stream>>>(g3(ctx), p0, q, Ev, Kv, ctx->d_fix, partA, S);
                k_pcg_k2<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, x, r, z, p0, q, D, partA, (int)g1, partB, S);
                continue;
            }
            if (csr) {
                k_pcg_k1_csr<<<g1, kBlock, 0, ctx->stream>>>(ctx->N, k, ctx->d_indptr, ctx->d_indices, ctx->d_data,
                                                            (const double*)pold, (const double*)z, (double*)pnew,
                                                            (double*)q, partB, (int)g2, partA, S, eps);
            } else if (is2d(ctx)) {
                const T* Ev = std::is_same<T, float>::value ? (const T*)ctx->d_Ef : (const T*)ctx->d_E;
                const T* Kv = std::is_same<T, float>::value ? (const T*)ctx->d_K0f : (const T*)ctx->d_K0;
                k_pcg_k1_q4_tile<T, kTileI, kTileJ><<<g1, kBlock, 0, ctx->stream>>>(
                    ctx->nx, ctx->ny, sh.tilesJ, sh.ntiles, k, pold, z, pnew, q, Ev, Kv, ctx->d_fix, partB, (int)g2,
                    partA, S, eps);
            }
            k_pcg_k2<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, x, r, z, pnew, q, D, partA, (int)g1, partB, S);
        }
        PF_TRY(check_launch(ctx));
        if (snap && std::is_same<T, double>::value && snap->count < snap->max && (k / chunk) % snap->every == 0) {
            PF_HIP(hipMemcpyAsync(snap->xs + (size_t)snap->count * n, x, sizeof(double) * n, hipMemcpyDeviceToDevice,
                                  ctx->stream));
            snap->iters.push_back(k);
            snap->count++;
        }
        PF_HIP(hipMemcpyAsync((void*)&hflag[slot], &S->done, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        PF_HIP(hipEventRecord(ev[slot], ctx->stream));
        return PF_OK;
    };
    while (!done && k < itrmax) {
        PF_TRY(enqueue_chunk(std::min(itrmax, k + chunk)));
        if (pending) {
            PF_HIP(hipEventSynchronize(ev[slot ^ 1]));
            if (hflag[slot ^ 1]) done = true;
        }
        pending = 1;
        slot ^= 1;
    }
    // drain
    PF_HIP(hipStreamSynchronize(ctx->stream));
    k_pcg_final<<<1, kBlock, 0, ctx->stream>>>(k, partB, (int)g2, S, eps);
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(ctx->h_pcg, S, sizeof(PcgDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    const PcgDev* H = (const PcgDev*)ctx->h_pcg;
    out.iterations = H->iterations;
    out.status = H->status;
    out.rnorm = H->rnorm;
    out.bnorm = H->bnorm;
    return PF_OK;
}

double reduce_host(pf_ctx* ctx, const double* part, int nparts, double scale, double shift, int* rc) {
    k_reduce_final<<<1, kBlock, 0, ctx->stream>>>(part, nparts, 1, scale, shift, ctx->red.out);
    hipMemcpyAsync(ctx->h_red + 8, ctx->red.out, sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        ctx->err = std::string("reduce: ") + hipGetErrorString(e);
        *rc = PF_ERR_HIP;
        return 0.0;
    }
    *rc = PF_OK;
    return ctx->h_red[8];
}

// True FP64 residual ||b - K x|| of nodal vectors (EbE operator).
int true_residual(pf_ctx* ctx, const double* b, const double* x, double* r, double* out_norm) {
    const unsigned g = gsize(ctx->nn);
    if (is2d(ctx))
        k_residual_q4<<<g, kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, b, x, r, ctx->d_E, ctx->d_K0, ctx->d_fix,
                                                    ctx->red.partials);
    else
        k_apply_h8<double><<<g, kBlock, 0, ctx->stream>>>(g3(ctx), x, r, ctx->d_E, ctx->d_K0, ctx->d_fix, 1, b,
                                                        ctx->red.partials);
    PF_TRY(check_launch(ctx));
    int rc;
    double rr = reduce_host(ctx, ctx->red.partials, (int)g, 1.0, 0.0, &rc);
    PF_TRY(rc);
    *out_norm = std::sqrt(rr);
    return PF_OK;
}

double norm_nodal(pf_ctx* ctx, const double* a, int* rc) {
    const unsigned g = gsize(ctx->nv);
    k_dot_partials<<<g, kBlock, 0, ctx->stream>>>(ctx->nv, a, a, ctx->red.partials);
    return std::sqrt(reduce_host(ctx, ctx->red.partials, (int)g, 1.0, 0.0, rc));
}

// Mixed precision: FP32 matrix-free Jacobi-PCG inner solves (FP32 vectors
// and operator, FP64 dot accumulation) inside FP64 iterative refinement:
// r = b - K x in FP64, solve K d = r in FP32 to inner_eps (relative, at most
// kInnerCap iterations), x += d in FP64, until ||b - K x|| <= eps ||b||.
// Each outer step gains at most about -log10(cond(K) * 6e-8) digits, whatever
// inner_eps is.  A step that does not halve the true residual (FP32 cannot
// resolve the system: moduli contrasts of 1e9 between neighbours) is undone
// and the refinement continues with FP64 Jacobi-PCG corrections from the
// current iterate (counted in st.fallbacks).
//
// With the parity operator (hex8, resident) an FP32 solve's true residual
// follows its recursive one further than with the direct operator, so that the
// refinement ends in fewer steps with less to spare: at inner_eps and eps
// themselves the solutions at 60x30x30 (eps = 1e-8, six density fields) were
// 2.3e-8 off in the mean, 1.9e-9 with the direct operator in one more step.
// There both are tightened to an eighth, which gives 8e-10 in 23 to 39 ms
// (launched 102 to 143 ms, untightened 18 to 35 ms); a last step solves no
// further than it has to, and one that starts with the caller's tolerance met
// takes no more iterations than the longest before it (where FP32 cannot
// reach the eighth it would run to kInnerCap to be undone).
int pcg_ir(pf_ctx* ctx, const double* b, double* x, double eps, int itrmax, double inner_eps, pf_solve_stats& st) {
    constexpr int kInnerCap = 20000;
    const bool parity = !is2d(ctx) && res3_applies(ctx) && res3_pick<float>(ctx).gi > 0;
    double goal = parity ? 0.125 * eps : eps;
    PF_TRY(diag_nodal(ctx, true));
    int rc;
    const double bn = norm_nodal(ctx, b, &rc);
    PF_TRY(rc);
    PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * ctx->nv, ctx->stream));
    double rn = bn;
    int outer = 0, total = 0, status = 2, fallbacks = 0, longest = 0;
    bool fp64 = false;
    const int max_outer = 60;
    double* r64 = ctx->d_t0;
    double* d64 = ctx->d_t1;
    PF_TRY(true_residual(ctx, b, x, r64, &rn));
    while (outer < max_outer) {
        const bool met = rn <= eps * bn;
        if (rn <= goal * bn || (met && outer == 0)) break;
        if (total >= itrmax) break;
        PcgRun run;
        if (!fp64) {
            const int cap = std::min(met ? longest : kInnerCap, itrmax - total);
            const double inner = parity ? std::max(0.125 * inner_eps, std::min(0.1, 0.1 * goal * bn / rn)) : inner_eps;
            k_convert<double, float><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, r64, ctx->f_b);
            PF_TRY(pcg_device<float>(ctx, false, ctx->f_b, ctx->f_x, ctx->f_D, ctx->f_r, ctx->f_z, ctx->f_p0,
                                     ctx->f_p1, ctx->f_q, inner, cap, run));
            total += run.iterations;
            longest = std::max(longest, run.iterations);
            outer++;
            PF_HIP(hipMemcpyAsync(d64, x, sizeof(double) * ctx->nv, hipMemcpyDeviceToDevice, ctx->stream));
            k_axpy_f32<<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->f_x, x);
            PF_TRY(check_launch(ctx));
            double rnew;
            PF_TRY(true_residual(ctx, b, x, r64, &rnew));
            if (std::isfinite(run.rnorm) && std::isfinite(rnew) && rnew <= 0.5 * rn) {
                rn = rnew;
                continue;
            }
            // undo the step: x and its true residual as they were
            PF_HIP(hipMemcpyAsync(x, d64, sizeof(double) * ctx->nv, hipMemcpyDeviceToDevice, ctx->stream));
            PF_TRY(true_residual(ctx, b, x, r64, &rn));
            goal = eps;
            if (rn <= eps * bn) break;
            fp64 = true;
            fallbacks++;
            continue;
        }
        // FP64 correction: K d = r to the relative tolerance that brings the
        // true residual to eps ||b||
        PF_TRY(diag_nodal(ctx, false));
        const double rel = std::min(0.5, eps * bn / rn);
        PF_TRY(pcg_device<double>(ctx, false, r64, d64, ctx->d_D, ctx->d_r, ctx->d_z, ctx->d_p0, ctx->d_p1,
                                  ctx->d_q, rel, itrmax - total, run));
        total += run.iterations;
        outer++;
        k_axpy_d<<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, 1.0, d64, x);
        PF_TRY(check_launch(ctx));
        PF_TRY(true_residual(ctx, b, x, r64, &rn));
    }
    if (rn <= eps * bn) status = 1;
    st.iterations = total;
    st.status = status;
    st.outer = outer;
    st.fallbacks = fallbacks;
    st.rel_residual = bn > 0 ? rn / bn : 0.0;
    return PF_OK;
}


// ----------------------------------------------------- learned network ----
}  // namespace

struct NetLayer {
    int cin = 0, cout = 0, level = 0, relu = 1;
    int ntap = 9;  // 3x3 (quad4) or 3x3x3 (hex8)
    float *W = nullptr, *m = nullptr, *v = nullptr, *g = nullptr;
    bf16 *Wb = nullptr, *Wtb = nullptr;
    long size() const { return (long)ntap * cin * cout; }
};

// Levels of the V-cycle (k_mg_* kernels): level 0 is the grid (E, K0, the
// context's fixity); coarser levels hold FP64 and FP32 element matrices.
struct MgLevel {
    int nx = 0, ny = 0, nz = 0;  // nz > 0: hex8
    long nn = 0, nv = 0, ne = 0;
    double* Ke64 = nullptr;  // levels >= 1, and level 0 when it is the coarsest (64 or 576 per element)
    float* Ke32 = nullptr;   // levels >= 1
    float* ye = nullptr;     // hex8 levels in the two-pass residual: 24 values per element
    float* D = nullptr;
    uint8_t* fix = nullptr;  // levels >= 1 (level 0 uses the context's)
    float *r = nullptr, *x = nullptr, *x2 = nullptr, *res = nullptr, *res2 = nullptr;
    // operator-dependent prolongation from the next coarser level (quad4,
    // levels with a coarser one): edge and centre weights in FP64 (for the
    // coarsening) and FP32 (for the V-cycle)
    double *wh64 = nullptr, *wv64 = nullptr, *wc64 = nullptr;
    float *wh = nullptr, *wv = nullptr, *wc = nullptr;
    MgProl prol(bool on) const { return on ? MgProl{wh, wv, wc} : MgProl{}; }
};
struct MgState {
    const int* done = nullptr;  // while set, the V-cycle's kernels return at once when *done
    // while set (quad4, nu = 1), the finest level's last sweep also writes z in
    // FP64 with the sums z.r, r.r (r64) into zpart, one per tile
    const double* r64 = nullptr;
    double* z64 = nullptr;
    double* zpart = nullptr;
    int tail = -1;              // first level of the one-workgroup tail (k_mg_tail), -1: none
    const float* tail_res = nullptr;  // the residual of the level above the tail (which restricts it)
    int prolong = PF_MG_PROLONG_STIFFNESS;  // quad4 prolongation (hex8: trilinear)
    int nu = 1;
    float omega = 0.6f;
    std::vector<MgLevel> L;
    int nf = 0;             // free DOFs of the coarsest level
    int* dof = nullptr;     // their nodal indices
    double* A = nullptr;    // coarsest free-DOF block, inverted in place
    double* W = nullptr;    // inversion scratch
    double* M = nullptr;    // hex8: the children's contributions to a coarse element (k_mg3_child_matrices), behind W
    std::vector<void*> owned;
};
// pixels per workgroup of a weight-gradient launch
constexpr int kWgradPixels = 4096;
// dot products one batched reduction holds (multidot_batch), and its grid
constexpr int kMpartDots = 128;
constexpr int kMpartGrid = 1024;

struct LearnedNet {
    int dim = 2;                            // 2: quad4 nodes (H x Wd), 3: hex8 nodes (H x Wd x Dz)
    int H[4] = {0}, Wd[4] = {0}, Dz[4] = {1, 1, 1, 1};
    std::vector<NetLayer> L;  // c0a c0b c1a c1b c2a c2b c3a c3b d2 d1 d0 out
    // activations (level, channels) and their gradients
    bf16 *x0, *a0, *e0, *x1, *a1, *e1, *x2, *a2, *e2, *x3, *a3, *b3, *u2, *d2, *u1, *d1, *u0, *d0;
    bf16 *gy, *gd0, *gu0, *gd1, *gu1, *gd2, *gu2, *gb3, *ga3, *gx3, *ge2, *ga2, *gx2, *ge1, *ga1, *gx1, *ge0, *ga0;
    float* y = nullptr;
    float* wpart = nullptr;
    long wpart_n = 0;
    // the network's stream beside a V-cycle, and its fork and join (made on first use)
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    // dataset (FP32): residual, error (nodal) and element densities per pair
    int cap = 0, nsamp = 0;
    float *ds_r = nullptr, *ds_e = nullptr, *ds_rho = nullptr;
    double* snap_x = nullptr;
    int snap_cap = 0;
    // the caller's densities and moduli, kept aside while training swaps in
    // each pair's
    double *keep_rho = nullptr, *keep_E = nullptr;
    float* keep_Ef = nullptr;
    // FP64 scratch (nodal)
    double *w = nullptr, *Kw = nullptr, *gd = nullptr, *rr = nullptr, *ee = nullptr, *dd = nullptr;
    int adam_t = 0;
    std::vector<void*> allocs;
    bool trained = false;
    // flexible CG: stored directions and their operator images
    int fcg_m = 0;
    std::vector<double*> fP, fQ;
    double* mpart = nullptr;  // multi-dot partials (grid x dots), then three blocks of sums
    FcgDev* fcg = nullptr;       // device state of the flexible CG
    FcgDev* fcg_host = nullptr;  // two pinned copies of it
};

namespace {

int moduli_from_rho(pf_ctx* ctx);

long lvl_px(LearnedNet* N, int lv) { return (long)N->H[lv] * N->Wd[lv] * N->Dz[lv]; }

void net_free(LearnedNet* N) {
    if (!N) return;
    if (N->side) {
        hipStreamSynchronize(N->side);
        hipStreamDestroy(N->side);
    }
    if (N->fork) hipEventDestroy(N->fork);
    if (N->join) hipEventDestroy(N->join);
    for (void* p : N->allocs) hipFree(p);
    if (N->fcg_host) hipHostFree(N->fcg_host);
    delete N;
}

void release_net(pf_ctx* ctx) {
    net_free(ctx->net);
    ctx->net = nullptr;
}

template <class T>
int net_alloc(pf_ctx* ctx, LearnedNet* N, T** p, long n) {
    PF_HIP(hipMalloc((void**)p, sizeof(T) * (size_t)std::max(1L, n)));
    N->allocs.push_back((void*)*p);
    PF_HIP(hipMemsetAsync(*p, 0, sizeof(T) * (size_t)std::max(1L, n), ctx->stream));
    return PF_OK;
}

uint64_t splitmix(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
double urand(uint64_t& s) { return (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0); }

int net_refresh_bf16(pf_ctx* ctx, LearnedNet* N) {
    for (NetLayer& l : N->L) {
        k_weights_bf16<<<nblocks(l.size()), kBlock, 0, ctx->stream>>>(l.ntap, l.cout, l.cin, l.W, l.Wb, l.Wtb);
    }
    return check_launch(ctx);
}

int net_build(pf_ctx* ctx, uint64_t seed) {
    net_free(ctx->net);
    LearnedNet* N = new LearnedNet();
    ctx->net = N;
    N->dim = is2d(ctx) ? 2 : 3;
    N->H[0] = ctx->nx + 1;
    N->Wd[0] = ctx->ny + 1;
    N->Dz[0] = N->dim == 3 ? ctx->nz + 1 : 1;
    for (int lv = 1; lv < 4; lv++) {
        N->H[lv] = (N->H[lv - 1] + 1) / 2;
        N->Wd[lv] = (N->Wd[lv - 1] + 1) / 2;
        N->Dz[lv] = N->dim == 3 ? (N->Dz[lv - 1] + 1) / 2 : 1;
    }
    const int ntap = N->dim == 3 ? 27 : 9;
    const int spec[kNetLayers][4] = {  // cin, cout, level, relu
        {16, 16, 0, 1}, {16, 16, 0, 1}, {16, 32, 1, 1}, {32, 32, 1, 1}, {32, 32, 2, 1}, {32, 32, 2, 1},
        {32, 64, 3, 1}, {64, 32, 3, 1}, {32, 32, 2, 1}, {32, 16, 1, 1}, {16, 16, 0, 1}, {16, 16, 0, 0}};
    uint64_t rs = seed ? seed : 20261204ull;
    long maxw = 0;
    for (int i = 0; i < kNetLayers; i++) {
        NetLayer l;
        l.cin = spec[i][0];
        l.cout = spec[i][1];
        l.level = spec[i][2];
        l.relu = spec[i][3];
        l.ntap = ntap;
        long n = l.size();
        maxw = std::max(maxw, n);
        PF_TRY(net_alloc(ctx, N, &l.W, n));
        PF_TRY(net_alloc(ctx, N, &l.m, n));
        PF_TRY(net_alloc(ctx, N, &l.v, n));
        PF_TRY(net_alloc(ctx, N, &l.g, n));
        PF_TRY(net_alloc(ctx, N, &l.Wb, n));
        PF_TRY(net_alloc(ctx, N, &l.Wtb, n));
        // He-uniform initialisation; the output layer starts near zero so that
        // the preconditioner starts at Jacobi
        std::vector<float> w(n);
        double a = std::sqrt(6.0 / ((double)ntap * l.cin)) * (i == kNetLayers - 1 ? 0.01 : 1.0);
        for (long q = 0; q < n; q++) w[q] = (float)((2.0 * urand(rs) - 1.0) * a);
        PF_HIP(hipMemcpyAsync(l.W, w.data(), sizeof(float) * n, hipMemcpyHostToDevice, ctx->stream));
        PF_TRY(sync(ctx));
        N->L.push_back(l);
    }
    PF_TRY(net_refresh_bf16(ctx, N));
    const long p0 = lvl_px(N, 0), p1 = lvl_px(N, 1), p2 = lvl_px(N, 2), p3 = lvl_px(N, 3);
    struct A { bf16** p; long n; } acts[] = {
        {&N->x0, p0 * 16}, {&N->a0, p0 * 16}, {&N->e0, p0 * 16}, {&N->x1, p1 * 16}, {&N->a1, p1 * 32},
        {&N->e1, p1 * 32}, {&N->x2, p2 * 32}, {&N->a2, p2 * 32}, {&N->e2, p2 * 32}, {&N->x3, p3 * 32},
        {&N->a3, p3 * 64}, {&N->b3, p3 * 32}, {&N->u2, p2 * 32}, {&N->d2, p2 * 32}, {&N->u1, p1 * 32},
        {&N->d1, p1 * 16}, {&N->u0, p0 * 16}, {&N->d0, p0 * 16},
        {&N->gy, p0 * 16}, {&N->gd0, p0 * 16}, {&N->gu0, p0 * 16}, {&N->gd1, p1 * 16}, {&N->gu1, p1 * 32},
        {&N->gd2, p2 * 32}, {&N->gu2, p2 * 32}, {&N->gb3, p3 * 32}, {&N->ga3, p3 * 64}, {&N->gx3, p3 * 32},
        {&N->ge2, p2 * 32}, {&N->ga2, p2 * 32}, {&N->gx2, p2 * 32}, {&N->ge1, p1 * 32}, {&N->ga1, p1 * 32},
        {&N->gx1, p1 * 16}, {&N->ge0, p0 * 16}, {&N->ga0, p0 * 16}};
    for (auto& a : acts) PF_TRY(net_alloc(ctx, N, a.p, a.n));
    PF_TRY(net_alloc(ctx, N, &N->y, p0 * 16));
    N->wpart_n = ((p0 + kWgradPixels - 1) / kWgradPixels) * maxw;
    PF_TRY(net_alloc(ctx, N, &N->wpart, N->wpart_n));
    const long nv = ctx->nv;
    PF_TRY(net_alloc(ctx, N, &N->mpart, (long)kMpartGrid * kMpartDots + 3 * kMpartDots));
    PF_TRY(net_alloc(ctx, N, &N->fcg, 1));
    PF_HIP(hipHostMalloc((void**)&N->fcg_host, 2 * sizeof(FcgDev)));
    double** sc[] = {&N->w, &N->Kw, &N->gd, &N->rr, &N->ee, &N->dd};
    for (double** q : sc) PF_TRY(net_alloc(ctx, N, q, nv));
    return sync(ctx);
}

constexpr long kConvFwdGrid = 768;  // workgroups of the tiled convolution
// yn (with fix): the nodal FP64 output of the network's last layer
// (kConvOutNodal), 16 -> 16 channels only
template <int CI, int CO>
int conv_fwd_t(pf_ctx* ctx, int H, int W, const bf16* X, const bf16* Wt, bf16* Y, float* Yf, int relu,
               const uint8_t* fix, double* yn) {
    // the tiled kernel addresses its tensors with 31-bit byte offsets
    if ((double)H * W * std::max(CI, CO) * 4 >= 2147483648.0) {
        ctx->err = "conv: image too large for the tiled convolution (2^31 bytes per tensor)";
        return PF_ERR_UNSUPPORTED;
    }
    // a few workgroups per CU, each looping over tiles of four rows (two
    // rows per wave measured slower for 16 -> 16 channels: 19.6 against
    // 18.8 us at 1025 x 513)
    constexpr int RPW = 1;
    const long ntiles = (long)((H + 4 * RPW - 1) / (4 * RPW)) * ((W + kConvTW - 1) / kConvTW);
    const unsigned grid = (unsigned)std::min<long>(ntiles, kConvFwdGrid);
    if (yn) {
        if constexpr (CI == 16 && CO == 16) {
            k_conv_fwd<CI, CO, RPW, kConvOutNodal>
                <<<grid, 256, 0, ctx->stream>>>(H, W, X, Wt, Y, Yf, relu, fix, yn);
            return PF_OK;
        }
        ctx->err = "conv: nodal output from 16 -> 16 channels only";
        return PF_ERR_UNSUPPORTED;
    }
    if (Yf)
        k_conv_fwd<CI, CO, RPW, kConvOutF32><<<grid, 256, 0, ctx->stream>>>(H, W, X, Wt, Y, Yf, relu, nullptr, nullptr);
    else
        k_conv_fwd<CI, CO, RPW, kConvOutBf16><<<grid, 256, 0, ctx->stream>>>(H, W, X, Wt, Y, Yf, relu, nullptr, nullptr);
    return PF_OK;
}

// One workgroup per kWgradPixels pixels.  The trained network depends on the
// gradients' rounding, and so does how well it preconditions (at 96x48 a
// different split of the pixels, with the same loss to 1%, took flexible CG
// from 405 to 1058 iterations), so the split is kept fixed.
template <int CI, int CO>
void conv_wgrad_t(pf_ctx* ctx, float* wpart, int H, int W, const bf16* X, const bf16* dZ, float* dW) {
    const int ppb = kWgradPixels;
    const long npx = (long)H * W;
    const int nb = (int)((npx + ppb - 1) / ppb);
    k_conv_wgrad<2, CI, CO><<<dim3(nb, 3, wgrad_tiles(CI, CO)), 64 * wgrad_waves(CI, CO), 0, ctx->stream>>>(
        H, W, 1, X, dZ, wpart, ppb);
    const int n = 9 * CI * CO;
    k_wgrad_reduce<<<nblocks(n), kBlock, 0, ctx->stream>>>(wpart, nb, n, dW);
}

// dispatch on (cin, cout) in {16, 32, 64}
int conv_fwd(pf_ctx* ctx, int cin, int cout, int H, int W, const bf16* X, const bf16* Wt, bf16* Y, float* Yf,
             int relu, const uint8_t* fix = nullptr, double* yn = nullptr) {
#define PF_CONV_CASE(a, b)                                                             \
    if (cin == a && cout == b) {                                                       \
        PF_TRY((conv_fwd_t<a, b>(ctx, H, W, X, Wt, Y, Yf, relu, fix, yn)));           \
        return check_launch(ctx);                                                      \
    }
    PF_CONV_CASE(16, 16) PF_CONV_CASE(16, 32) PF_CONV_CASE(32, 16) PF_CONV_CASE(32, 32) PF_CONV_CASE(32, 64)
    PF_CONV_CASE(64, 32) PF_CONV_CASE(16, 64) PF_CONV_CASE(64, 16) PF_CONV_CASE(64, 64)
#undef PF_CONV_CASE
    ctx->err = "conv: unsupported channel counts";
    return PF_ERR_UNSUPPORTED;
}

// wpart: FP32 partials of ceil(H W / kWgradPixels) workgroups x 9 cin cout
int conv_wgrad(pf_ctx* ctx, int cin, int cout, int H, int W, const bf16* X, const bf16* dZ, float* dW,
               float* wpart = nullptr) {
    if (!wpart) wpart = ctx->net->wpart;
#define PF_WG_CASE(a, b) \
    if (cin == a && cout == b) { conv_wgrad_t<a, b>(ctx, wpart, H, W, X, dZ, dW); return check_launch(ctx); }
    PF_WG_CASE(16, 16) PF_WG_CASE(16, 32) PF_WG_CASE(32, 16) PF_WG_CASE(32, 32) PF_WG_CASE(32, 64) PF_WG_CASE(64, 32)
#undef PF_WG_CASE
    ctx->err = "wgrad: unsupported channel counts";
    return PF_ERR_UNSUPPORTED;
}

// hex8 networks: 3x3x3 convolutions on an H x W x Dp node grid
// At most 32 channels in and out: the LDS-tiled kernel (k_conv3_fwd_tile,
// up to 768 workgroups looping over tiles of 16 NQ nodes along k); else one
// line per workgroup (k_conv3_fwd).  yn (with fix): the nodal FP64 output of
// the network's last layer, 16 -> 16.
constexpr long kConv3Grid = 768;
template <int CI, int CO, int NQ>
int conv3_tile_t(pf_ctx* ctx, int H, int W, int Dp, const bf16* X, const bf16* Wt, bf16* Y, float* Yf, int relu,
                 const uint8_t* fix, double* yn) {
    const long ntiles = (long)H * ((W + kConv3TJ - 1) / kConv3TJ) * ((Dp + 16 * NQ - 1) / (16 * NQ));
    const unsigned grid = (unsigned)std::min<long>(ntiles, kConv3Grid);
    if (yn) {
        if constexpr (CO == 16) {
            k_conv3_fwd_tile<CI, CO, kConvOutNodal, NQ>
                <<<grid, 256, 0, ctx->stream>>>(H, W, Dp, X, Wt, Y, Yf, relu, fix, yn);
            return PF_OK;
        }
        ctx->err = "conv3: nodal output from 16 -> 16 channels only";
        return PF_ERR_UNSUPPORTED;
    }
    if (Yf)
        k_conv3_fwd_tile<CI, CO, kConvOutF32, NQ>
            <<<grid, 256, 0, ctx->stream>>>(H, W, Dp, X, Wt, Y, Yf, relu, nullptr, nullptr);
    else
        k_conv3_fwd_tile<CI, CO, kConvOutBf16, NQ>
            <<<grid, 256, 0, ctx->stream>>>(H, W, Dp, X, Wt, Y, Yf, relu, nullptr, nullptr);
    return PF_OK;
}
template <int CI, int CO>
int conv3_fwd_t(pf_ctx* ctx, int H, int W, int Dp, const bf16* X, const bf16* Wt, bf16* Y, float* Yf, int relu,
                const uint8_t* fix, double* yn) {
    if constexpr (CI <= 32 && CO <= 32) {
        if ((double)H * W * Dp * std::max(CO * 4, 24) >= 2147483648.0) {
            ctx->err = "conv3: grid too large for the tiled convolution (2^31 bytes per tensor)";
            return PF_ERR_UNSUPPORTED;
        }
        // one tile along k for lines of at most 80 nodes (64 with 32 input
        // channels: its 80-node tile would hold 96 prefetch registers), else
        // 64-node tiles
        const int nq = (Dp + 15) / 16;
        auto go = [&](auto NQc) {
            return conv3_tile_t<CI, CO, decltype(NQc)::value>(ctx, H, W, Dp, X, Wt, Y, Yf, relu, fix, yn);
        };
        if (nq <= 1) return go(std::integral_constant<int, 1>{});
        if (nq == 2) return go(std::integral_constant<int, 2>{});
        if (nq == 3) return go(std::integral_constant<int, 3>{});
        if constexpr (CI == 16)
            if (nq == 5) return go(std::integral_constant<int, 5>{});
        return go(std::integral_constant<int, 4>{});
    }
    if (yn) {
        ctx->err = "conv3: nodal output from 16 -> 16 channels only";
        return PF_ERR_UNSUPPORTED;
    }
    dim3 grid((unsigned)(H * W), (Dp + 63) / 64);
    k_conv3_fwd<CI, CO><<<grid, 256, 0, ctx->stream>>>(H, W, Dp, X, Wt, Y, Yf, relu);
    return PF_OK;
}

template <int CI, int CO>
void conv3_wgrad_t(pf_ctx* ctx, float* wpart, int H, int W, int Dp, const bf16* X, const bf16* dZ, float* dW) {
    const int ppb = kWgradPixels;
    const long npx = (long)H * W * Dp;
    const int nb = (int)((npx + ppb - 1) / ppb);
    k_conv_wgrad<3, CI, CO><<<dim3(nb, 9, wgrad_tiles(CI, CO)), 64 * wgrad_waves(CI, CO), 0, ctx->stream>>>(
        H, W, Dp, X, dZ, wpart, ppb);
    const int n = 27 * CI * CO;
    k_wgrad_reduce<<<nblocks(n), kBlock, 0, ctx->stream>>>(wpart, nb, n, dW);
}

int conv3_fwd(pf_ctx* ctx, int cin, int cout, int H, int W, int Dp, const bf16* X, const bf16* Wt, bf16* Y,
              float* Yf, int relu, const uint8_t* fix = nullptr, double* yn = nullptr) {
#define PF_CONV3_CASE(a, b)                                                            \
    if (cin == a && cout == b) {                                                       \
        PF_TRY((conv3_fwd_t<a, b>(ctx, H, W, Dp, X, Wt, Y, Yf, relu, fix, yn)));      \
        return check_launch(ctx);                                                      \
    }
    PF_CONV3_CASE(16, 16) PF_CONV3_CASE(16, 32) PF_CONV3_CASE(32, 16) PF_CONV3_CASE(32, 32) PF_CONV3_CASE(32, 64)
    PF_CONV3_CASE(64, 32)
#undef PF_CONV3_CASE
    ctx->err = "conv3: unsupported channel counts";
    return PF_ERR_UNSUPPORTED;
}

int conv3_wgrad(pf_ctx* ctx, int cin, int cout, int H, int W, int Dp, const bf16* X, const bf16* dZ, float* dW,
                float* wpart = nullptr) {
    if (!wpart) wpart = ctx->net->wpart;
#define PF_WG3_CASE(a, b) \
    if (cin == a && cout == b) { conv3_wgrad_t<a, b>(ctx, wpart, H, W, Dp, X, dZ, dW); return check_launch(ctx); }
    PF_WG3_CASE(16, 16) PF_WG3_CASE(16, 32) PF_WG3_CASE(32, 16) PF_WG3_CASE(32, 32) PF_WG3_CASE(32, 64)
    PF_WG3_CASE(64, 32)
#undef PF_WG3_CASE
    ctx->err = "wgrad3: unsupported channel counts";
    return PF_ERR_UNSUPPORTED;
}

// The network's forward pass on N->x0.  nodal: the output field as the nodal
// FP64 vector N->w (DOFs fixed by ctx->d_fix zeroed), else the 16-channel
// FP32 output N->y.
int net_forward(pf_ctx* ctx, bool nodal) {
    LearnedNet* N = ctx->net;
    auto& L = N->L;
    const bool d3 = N->dim == 3;
    auto lay = [&](int li, const bf16* X, bf16* Y, float* Yf) {
        NetLayer& l = L[li];
        if (d3)
            return conv3_fwd(ctx, l.cin, l.cout, N->H[l.level], N->Wd[l.level], N->Dz[l.level], X, l.Wb, Y, Yf,
                             l.relu);
        return conv_fwd(ctx, l.cin, l.cout, N->H[l.level], N->Wd[l.level], X, l.Wb, Y, Yf, l.relu);
    };
    auto pool = [&](int lv, int C, const bf16* in, bf16* out) {
        long n = lvl_px(N, lv + 1) * C / 8;  // 8 channels per thread
        if (d3)
            k_pool3<<<gsize(n), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], N->Dz[lv], C, in, out);
        else
            k_pool2<<<gsize(n), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], C, in, out);
    };
    auto upadd = [&](int lv, int C, const bf16* coarse, const bf16* skip, bf16* out) {
        long n = lvl_px(N, lv) * C / 8;
        if (d3)
            k_up3_add<<<gsize(n), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], N->Dz[lv], C, coarse, skip, out);
        else
            k_up2_add<<<gsize(n), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], C, coarse, skip, out);
    };
    PF_TRY(lay(0, N->x0, N->a0, nullptr));
    PF_TRY(lay(1, N->a0, N->e0, nullptr));
    pool(0, 16, N->e0, N->x1);
    PF_TRY(lay(2, N->x1, N->a1, nullptr));
    PF_TRY(lay(3, N->a1, N->e1, nullptr));
    pool(1, 32, N->e1, N->x2);
    PF_TRY(lay(4, N->x2, N->a2, nullptr));
    PF_TRY(lay(5, N->a2, N->e2, nullptr));
    pool(2, 32, N->e2, N->x3);
    PF_TRY(lay(6, N->x3, N->a3, nullptr));
    PF_TRY(lay(7, N->a3, N->b3, nullptr));
    upadd(2, 32, N->b3, N->e2, N->u2);
    PF_TRY(lay(8, N->u2, N->d2, nullptr));
    upadd(1, 32, N->d2, N->e1, N->u1);
    PF_TRY(lay(9, N->u1, N->d1, nullptr));
    upadd(0, 16, N->d1, N->e0, N->u0);
    PF_TRY(lay(10, N->u0, N->d0, nullptr));
    if (nodal) {
        // the last layer writes the nodal vector itself (kConvOutNodal)
        NetLayer& l = L[11];
        if (d3)
            PF_TRY(conv3_fwd(ctx, l.cin, l.cout, N->H[l.level], N->Wd[l.level], N->Dz[l.level], N->d0, l.Wb, nullptr,
                             nullptr, l.relu, ctx->d_fix, N->w));
        else
            PF_TRY(conv_fwd(ctx, l.cin, l.cout, N->H[l.level], N->Wd[l.level], N->d0, l.Wb, nullptr, nullptr, l.relu,
                            ctx->d_fix, N->w));
        return check_launch(ctx);
    }
    PF_TRY(lay(11, N->d0, nullptr, N->y));
    return check_launch(ctx);
}

// gradients of all layer weights for the output gradient N->gy
int net_backward(pf_ctx* ctx) {
    LearnedNet* N = ctx->net;
    auto& L = N->L;
    // layer li: output gradient gz (already masked by ReLU), input X -> dW, and
    // the input gradient gx (if non-null)
    const bool d3 = N->dim == 3;
    auto back = [&](int li, const bf16* X, bf16* gz, bf16* gx) -> int {
        NetLayer& l = L[li];
        const int H = N->H[l.level], W = N->Wd[l.level], Dp = N->Dz[l.level];
        if (d3) {
            PF_TRY(conv3_wgrad(ctx, l.cin, l.cout, H, W, Dp, X, gz, l.g));
            if (gx) PF_TRY(conv3_fwd(ctx, l.cout, l.cin, H, W, Dp, gz, l.Wtb, gx, nullptr, 0));
            return PF_OK;
        }
        PF_TRY(conv_wgrad(ctx, l.cin, l.cout, H, W, X, gz, l.g));
        if (gx) PF_TRY(conv_fwd(ctx, l.cout, l.cin, H, W, gz, l.Wtb, gx, nullptr, 0));
        return PF_OK;
    };
    auto relu_bwd = [&](int lv, int C, const bf16* Y, bf16* g) {
        const long n8 = lvl_px(N, lv) * C / 8;
        k_relu_bwd<<<gsize(n8), kBlock, 0, ctx->stream>>>(n8, (const uint4*)Y, (uint4*)g);
    };
    auto depth = [&](int lv) { return d3 ? N->Dz[lv] : 1; };
    // gradient of the decoder output Y on level lv + 1 (C channels) from that of its upsampled sum on level lv
    auto up_bwd = [&](int lv, int C, const bf16* gfine, const bf16* Y, bf16* g) {
        k_up_bwd<<<gsize(lvl_px(N, lv + 1) * C / 8), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], depth(lv), C, gfine,
                                                                             Y, g);
    };
    // gradient of the encoder output Y on level lv from its skip and pooled branches
    auto skip_pool_bwd = [&](int lv, int C, const bf16* gskip, const bf16* gcoarse, const bf16* Y, bf16* g) {
        k_skip_pool_bwd<<<gsize(lvl_px(N, lv) * C / 8), kBlock, 0, ctx->stream>>>(N->H[lv], N->Wd[lv], depth(lv), C,
                                                                                gskip, gcoarse, Y, g);
    };
    PF_TRY(back(11, N->d0, N->gy, N->gd0));
    relu_bwd(0, 16, N->d0, N->gd0);
    PF_TRY(back(10, N->u0, N->gd0, N->gu0));
    up_bwd(0, 16, N->gu0, N->d1, N->gd1);
    PF_TRY(back(9, N->u1, N->gd1, N->gu1));
    up_bwd(1, 32, N->gu1, N->d2, N->gd2);
    PF_TRY(back(8, N->u2, N->gd2, N->gu2));
    up_bwd(2, 32, N->gu2, N->b3, N->gb3);
    PF_TRY(back(7, N->a3, N->gb3, N->ga3));
    relu_bwd(3, 64, N->a3, N->ga3);
    PF_TRY(back(6, N->x3, N->ga3, N->gx3));
    skip_pool_bwd(2, 32, N->gu2, N->gx3, N->e2, N->ge2);
    PF_TRY(back(5, N->a2, N->ge2, N->ga2));
    relu_bwd(2, 32, N->a2, N->ga2);
    PF_TRY(back(4, N->x2, N->ga2, N->gx2));
    skip_pool_bwd(1, 32, N->gu1, N->gx2, N->e1, N->ge1);
    PF_TRY(back(3, N->a1, N->ge1, N->ga1));
    relu_bwd(1, 32, N->a1, N->ga1);
    PF_TRY(back(2, N->x1, N->ga1, N->gx1));
    skip_pool_bwd(0, 16, N->gu0, N->gx1, N->e0, N->ge0);
    PF_TRY(back(1, N->a0, N->ge0, N->ga0));
    relu_bwd(0, 16, N->a0, N->ga0);
    PF_TRY(back(0, N->x0, N->ga0, nullptr));
    return check_launch(ctx);
}


// ------------------------------------------------------------ multigrid ----
// levels with at least this many nodes use the LDS-tiled sweep
constexpr long kMgTileNodes = 16384;
// the finest level's tiles (1024x512: 11.0 us per sweep; 4x64 tiles 11.5 us)
constexpr int kMgTile0TI = 8, kMgTile0TJ = 64;
// coarse levels of kMgMidNodes nodes or more: tiles of kMgMidTI x kMgMidTJ
// nodes (1024x512, levels 3-4: 5.2 us per sweep against 8.2 us for the
// untiled sweep, 16x16 and 8x32 tiles 5.35 and 5.34 us; levels 1-2: 4x64
// tiles took the solve from 7.00 to 6.68 ms against 8x64 tiles)
constexpr long kMgMidNodes = 2048;
constexpr int kMgMidTI = 4, kMgMidTJ = 64;
// coarsening stops at the first level with at most this many nodal DOFs (a
// 8 x 4 level: its free block is inverted in LDS)
constexpr long kMgCoarse = 90;

void mg_free(pf_ctx* ctx) {
    if (!ctx->mg) return;
    for (void* p : ctx->mg->owned) hipFree(p);
    delete ctx->mg;
    ctx->mg = nullptr;
}

template <class T>
int mg_alloc(pf_ctx* ctx, T** p, long n) {
    if (hipMalloc((void**)p, sizeof(T) * (size_t)std::max(1L, n)) != hipSuccess) {
        ctx->err = "hipMalloc failed for the multigrid hierarchy";
        return PF_ERR_NOMEM;
    }
    ctx->mg->owned.push_back(*p);
    return PF_OK;
}

// the hex8 tail forms its residual element-wise unless the node form is
// asked for (its levels are below kMg3ElemMin elements, but in one workgroup
// the element form's matrix reads are independent of one another)
inline bool mg3_tail_elem(const pf_ctx* ctx) { return ctx->mg_resid != PF_MG_RESIDUAL_NODE; }

// levels and their storage for the current grid
int mg_plan(pf_ctx* ctx, int nu, float omega, int prolong) {
    mg_free(ctx);
    ctx->mg = new MgState;
    MgState* S = ctx->mg;
    S->nu = nu;
    S->omega = omega;
    S->prolong = prolong;
    const bool h8 = !is2d(ctx);
    int nx = ctx->nx, ny = ctx->ny, nz = h8 ? ctx->nz : 0;
    for (;;) {
        MgLevel a;
        a.nx = nx;
        a.ny = ny;
        a.nz = nz;
        a.nn = (long)(nx + 1) * (ny + 1) * (h8 ? nz + 1 : 1);
        a.nv = (h8 ? 3 : 2) * a.nn;
        a.ne = (long)nx * ny * (h8 ? nz : 1);
        S->L.push_back(a);
        if (a.nv <= kMgCoarse || nx % 2 || ny % 2 || (h8 && nz % 2)) break;
        nx /= 2;
        ny /= 2;
        nz /= 2;
    }
    const int c = (int)S->L.size() - 1;
    PF_CHECK(S->L[c].nv <= kMgDenseMax, PF_ERR_UNSUPPORTED,
             "multigrid: the grid does not coarsen to a small enough level (element counts must be divisible by "
             "powers of two)");
    const long kes = h8 ? 576 : 64;
    for (int l = 0; l <= c; l++) {
        MgLevel& a = S->L[l];
        if (l > 0 || l == c) PF_TRY(mg_alloc(ctx, &a.Ke64, a.ne * kes));
        if (l > 0) {
            PF_TRY(mg_alloc(ctx, &a.Ke32, a.ne * kes));
            PF_TRY(mg_alloc(ctx, &a.fix, a.nn));
            const bool elem = ctx->mg_resid == PF_MG_RESIDUAL_ELEMENT ||
                              (ctx->mg_resid == PF_MG_RESIDUAL_AUTO && a.ne >= kMg3ElemMin);
            if (h8 && elem) PF_TRY(mg_alloc(ctx, &a.ye, a.ne * 24));
        }
        float** v[] = {&a.D, &a.r, &a.x, &a.x2, &a.res, &a.res2};
        for (float** q : v) PF_TRY(mg_alloc(ctx, q, a.nv));
        if (!h8 && l < c && prolong == PF_MG_PROLONG_STIFFNESS) {
            const long cnx = a.nx / 2, cny = a.ny / 2;
            const long nh = cnx * (cny + 1), nvv = (cnx + 1) * cny, ncw = cnx * cny * 16;
            PF_TRY(mg_alloc(ctx, &a.wh64, nh));
            PF_TRY(mg_alloc(ctx, &a.wv64, nvv));
            PF_TRY(mg_alloc(ctx, &a.wc64, ncw));
            PF_TRY(mg_alloc(ctx, &a.wh, nh));
            PF_TRY(mg_alloc(ctx, &a.wv, nvv));
            PF_TRY(mg_alloc(ctx, &a.wc, ncw));
        }
    }
    // the small levels (and the coarsest solve) run in one workgroup
    if (!h8 && S->L[c].nv <= kMgLdsDense) {
        int t = c;
        // LDS the tail kernel needs for levels t .. c
        auto pool = [&](int t0) {
            long off = 0;
            int lo[kMtSlots];
            for (int k = t0; k <= c; k++)
                off = mg_tail_place(S->L[k].nx, S->L[k].ny, k == c, prolong == PF_MG_PROLONG_STIFFNESS, off, lo);
            return off;
        };
        while (t - 1 >= 1 && S->L[t - 1].nn <= kMgTailNodes && c - (t - 1) + 1 <= kMgTailMax &&
               pool(t - 1) <= kMgTailPool)
            t--;
        if (S->L[t].nn <= kMgTailNodes && t >= 1 && pool(t) <= kMgTailPool) S->tail = t;
    }
    if (h8 && S->L[c].nv <= kMgLdsDense) {
        int t = c;
        auto pool = [&](int t0) {
            long off = 0;
            int lo[kM3Slots];
            for (int k = t0; k <= c; k++)
                off = mg3_tail_place(S->L[k].nx, S->L[k].ny, S->L[k].nz, k == c, mg3_tail_elem(ctx), off, lo);
            return off;
        };
        while (t - 1 >= 1 && S->L[t - 1].nn <= kMgTailNodes && c - (t - 1) + 1 <= kMgTailMax &&
               pool(t - 1) <= kMgTailPool)
            t--;
        if (S->L[t].nn <= kMgTailNodes && t >= 1 && pool(t) <= kMgTailPool) S->tail = t;
    }
    const long nvc = S->L[c].nv;
    PF_TRY(mg_alloc(ctx, &S->dof, nvc));
    PF_TRY(mg_alloc(ctx, &S->A, nvc * nvc));
    PF_TRY(mg_alloc(ctx, &S->W, nvc * nvc + (h8 ? 8L * 576 : 0)));
    S->M = S->W + nvc * nvc;
    return PF_OK;
}

// coarse operators, diagonals and the coarsest inverse for the current moduli
int mg_build(pf_ctx* ctx) {
    MgState* S = ctx->mg;
    PF_CHECK(S, PF_ERR_STATE, "multigrid not set up: call pf_mg_setup first");
    const int c = (int)S->L.size() - 1;
    const bool h8 = S->L[0].nz > 0;
    const int ndpn = h8 ? 3 : 2;
    MgLevel& l0 = S->L[0];
    if (h8)
        k_mg3_diag0<<<gsize(l0.nn), kBlock, 0, ctx->stream>>>(l0.nx, l0.ny, l0.nz, ctx->d_E, ctx->d_K0, ctx->d_fix,
                                                             l0.D);
    else
        k_mg_diag0<<<gsize(l0.nn), kBlock, 0, ctx->stream>>>(l0.nx, l0.ny, ctx->d_E, ctx->d_K0, ctx->d_fix, l0.D);
    for (int l = 1; l <= c; l++) {
        MgLevel& a = S->L[l];
        const double* Kf = l == 1 ? nullptr : S->L[l - 1].Ke64;
        if (h8) {
            if (l == 1) {
                k_mg3_child_matrices<<<18, kBlock, 0, ctx->stream>>>(ctx->d_K0, S->M);
                k_mg3_coarsen0<<<(unsigned)std::min(a.ne, 4096L), kMg3C0Threads, 0, ctx->stream>>>(
                    a.nx, a.ny, a.nz, ctx->d_E, ctx->d_K0, S->M, ctx->d_fix, a.Ke64, a.Ke32);
            } else {
                const long t = a.ne * 24;
                k_mg3_coarsen<<<(unsigned)((t + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(a.nx, a.ny, a.nz, Kf,
                                                                                                 a.Ke64, a.Ke32);
            }
            k_mg3_diag_full<<<gsize(a.nn), kBlock, 0, ctx->stream>>>(a.nx, a.ny, a.nz, a.Ke64, a.D, a.fix);
        } else {
            const long t = a.ne * 8;
            MgLevel& f = S->L[l - 1];
            if (f.wh64) {
                const long ne_w = (long)a.nx * (a.ny + 1) + (long)(a.nx + 1) * a.ny;
                k_mg_edge_weights<<<gsize(ne_w), kBlock, 0, ctx->stream>>>(f.nx, f.ny, ctx->d_E, ctx->d_K0,
                                                                          ctx->d_fix, Kf, f.wh64, f.wv64, f.wh, f.wv);
                k_mg_centre_weights<<<gsize(a.ne), kBlock, 0, ctx->stream>>>(a.nx, a.ny, ctx->d_E, ctx->d_K0,
                                                                            ctx->d_fix, Kf, f.wh64, f.wv64, f.wc64,
                                                                            f.wc);
                k_mg_coarsen_w<<<(unsigned)((t + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(
                    a.nx, a.ny, ctx->d_E, ctx->d_K0, ctx->d_fix, Kf, f.wh64, f.wv64, f.wc64, a.Ke64, a.Ke32);
            } else {
                k_mg_coarsen<<<(unsigned)((t + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(
                    a.nx, a.ny, ctx->d_E, ctx->d_K0, ctx->d_fix, Kf, a.Ke64, a.Ke32);
            }
            k_mg_diag_full<<<gsize(a.nn), kBlock, 0, ctx->stream>>>(a.nx, a.ny, a.Ke64, a.D, a.fix);
        }
    }
    MgLevel& C = S->L[c];
    if (c == 0) {
        const long t = C.ne * (h8 ? 576 : 64);
        if (h8)
            k_mg3_ke0_full<<<(unsigned)((t + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(C.ne, ctx->d_E,
                                                                                          ctx->d_K0, C.Ke64);
        else
            k_mg_ke0_full<<<(unsigned)((t + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(C.ne, ctx->d_E,
                                                                                         ctx->d_K0, C.Ke64);
    }
    PF_TRY(check_launch(ctx));
    // free DOFs of the coarsest level (its fixity is known only now)
    std::vector<uint8_t> hf(C.nn);
    PF_HIP(hipMemcpyAsync(hf.data(), c == 0 ? ctx->d_fix : C.fix, C.nn, hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    std::vector<int> dof;
    for (long n = 0; n < C.nn; n++)
        for (int d = 0; d < ndpn; d++)
            if (!((hf[n] >> d) & 1)) dof.push_back((int)(ndpn * n + d));
    S->nf = (int)dof.size();
    PF_CHECK(S->nf > 0, PF_ERR_STATE, "multigrid: no free DOFs on the coarsest level");
    PF_HIP(hipMemcpyAsync(S->dof, dof.data(), sizeof(int) * dof.size(), hipMemcpyHostToDevice, ctx->stream));
    const long nf2 = (long)S->nf * S->nf;
    if (h8)
        k_mg3_dense<<<(unsigned)((nf2 + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(C.nx, C.ny, C.nz, C.Ke64,
                                                                                        S->dof, S->nf, S->A);
    else
        k_mg_dense<<<(unsigned)((nf2 + kBlock - 1) / kBlock), kBlock, 0, ctx->stream>>>(C.nx, C.ny, C.Ke64,
                                                                                       S->dof, S->nf, S->A);
    if (S->nf <= kMgLdsDense)
        k_mg_invert_lds<<<1, 1024, 0, ctx->stream>>>(S->nf, S->A);
    else
        k_mg_invert<<<1, kBlock, 0, ctx->stream>>>(S->nf, S->A, S->W);
    PF_TRY(check_launch(ctx));
    return sync(ctx);  // dof (host vector) must outlive its copy
}

// one V-cycle from level l on S->L[l].r; returns the buffer holding x
float* mg_cycle(pf_ctx* ctx, int l) {
    MgState* S = ctx->mg;
    MgLevel& a = S->L[l];
    const int c = (int)S->L.size() - 1;
    if (l == S->tail && a.nz > 0) {  // hex8
        Mg3Tail T{};
        T.nlev = c - l + 1;
        long off = 0;
        for (int k = 0; k < T.nlev; k++) {
            MgLevel& b = S->L[l + k];
            Mg3TailLevel& t = T.L[k];
            t.nx = b.nx;
            t.ny = b.ny;
            t.nz = b.nz;
            t.Ke = b.Ke32;
            t.D = b.D;
            t.fix = b.fix;
            t.x = b.x;
            // fits, as mg_plan checked
            off = mg3_tail_place(b.nx, b.ny, b.nz, k == T.nlev - 1, mg3_tail_elem(ctx), off, t.lo);
        }
        T.elem = mg3_tail_elem(ctx) ? 1 : 0;
        T.pres = S->tail_res;
        T.nf = S->nf;
        T.Ainv = S->A;
        T.dof = S->dof;
        T.nu = S->nu;
        T.omega = S->omega;
        k_mg3_tail<<<1, kMgTailNodes, 0, ctx->stream>>>(T, S->done);
        return a.x;
    }
    if (l == S->tail) {
        MgTail T{};
        T.nlev = c - l + 1;
        long off = 0;
        for (int k = 0; k < T.nlev; k++) {
            MgLevel& b = S->L[l + k];
            MgTailLevel& t = T.L[k];
            t.nx = b.nx;
            t.ny = b.ny;
            t.Ke = b.Ke32;
            t.D = b.D;
            t.fix = b.fix;
            t.x = b.x;
            t.x2 = b.x2;
            t.P = b.prol(true);
            // the weights exist exactly when mg_plan counted them, so the
            // levels fit the pool as planned
            off = mg_tail_place(b.nx, b.ny, k == T.nlev - 1, t.P.wh != nullptr, off, t.lo);
        }
        T.nf = S->nf;
        T.Ainv = S->A;
        T.dof = S->dof;
        T.nu = S->nu;
        T.omega = S->omega;
        T.pres = S->tail_res;
        T.pP = S->L[l - 1].prol(true);
        k_mg_tail<<<1, kMgTailNodes, 0, ctx->stream>>>(T, S->done);
        if (T.nlev == 1) return a.x;
        return mg_tail_final_is_x2(S->nu) ? a.x2 : a.x;
    }
    if (l == c) {
        k_fill<float><<<gsize(a.nv), kBlock, 0, ctx->stream>>>(a.nv, a.x, 0.f);
        k_mg_coarse_solve<<<(unsigned)((S->nf + 63) / 64), 256, 0, ctx->stream>>>(S->nf, S->A, S->dof, a.r, a.x,
                                                                                S->done);
        return a.x;
    }
    if (a.nz > 0) {  // hex8: two-pass sweeps
        const uint8_t* fx3 = l == 0 ? ctx->d_fix : a.fix;
        float *x = a.x, *res = a.res, *xo = a.x2;
        auto run3 = [&](auto ke) {
            const unsigned gv = gsize(a.nv), gn = gsize(a.nn);
            // the two-pass residual (element pass, node pass) with its input
            // formed as MODE says (kMg3InUpdate: xout receives the update)
            auto elem2 = [&](auto mode, const float* Ke, const float* xin, const float* xc, float* rout,
                             float* xout) {
                constexpr int MODE = decltype(mode)::value;
                k_mg3_elem_apply<MODE><<<gsize8((a.ne + 31) / 32 * kBlock), kBlock, 0, ctx->stream>>>(
                    a.nx, a.ny, a.nz, Ke, xin, xc, a.r, a.D, fx3, S->omega, a.ye, S->done);
                k_mg3_node_gather<MODE><<<gsize8(a.nn), kBlock, 0, ctx->stream>>>(
                    a.nx, a.ny, a.nz, a.ye, a.D, fx3, S->omega, a.r, xin, xc, rout, xout, S->done);
            };
            // res = r - A xin, or with xout, xout = xin + omega D^-1 (r - A xin)
            auto residual = [&](const float* xin, float* rout, float* xout) {
                if constexpr (std::is_same<decltype(ke), Mg3KeTile>::value) {
                    const H8Shape& t = *ke.sh;
                    if (t.per == 5)
                        k_mg3_residual0_tile<5><<<t.grid, kBlock, t.lds, ctx->stream>>>(
                            g3(ctx), t.nslab, t.planes, t.nwork, ctx->d_Ef, ctx->d_K0gf, a.D, fx3, S->omega, a.r, xin,
                            rout, xout, S->done);
                    else
                        k_mg3_residual0_tile<8><<<t.grid, kBlock, t.lds, ctx->stream>>>(
                            g3(ctx), t.nslab, t.planes, t.nwork, ctx->d_Ef, ctx->d_K0gf, a.D, fx3, S->omega, a.r, xin,
                            rout, xout, S->done);
                } else if constexpr (std::is_same<decltype(ke), Mg3KeFull>::value) {
                    if (a.ye) {  // large level: element pass, then node pass
                        elem2(std::integral_constant<int, kMg3In>{}, ke.Ke, xin, nullptr, rout, xout);
                    } else {
                        k_mg3_residual<<<gsize8(a.nn), kBlock, 0, ctx->stream>>>(
                            a.nx, a.ny, a.nz, ke, a.D, fx3, S->omega, a.r, xin, rout, xout, S->done);
                    }
                } else {
                    k_mg3_residual<<<gsize8(a.nn), kBlock, 0, ctx->stream>>>(a.nx, a.ny, a.nz, ke, a.D, fx3,
                                                                             S->omega, a.r, xin, rout, xout, S->done);
                }
            };
            // the element form on a coarse level takes the first pre-smoothing
            // update and the prolongation into its element and node passes
            constexpr bool fuse = std::is_same<decltype(ke), Mg3KeFull>::value;
            if (fuse && a.ye) {
                elem2(std::integral_constant<int, kMg3InUpdate>{}, a.Ke32, nullptr, nullptr, res, x);
            } else {
                k_mg3_update<<<gv, kBlock, 0, ctx->stream>>>(a.nv, S->omega, nullptr, nullptr, a.r, a.D, fx3, x,
                                                             S->done);
                residual(x, res, nullptr);
            }
            for (int k = 1; k < S->nu; k++) {
                k_mg3_update<<<gv, kBlock, 0, ctx->stream>>>(a.nv, S->omega, x, res, a.r, a.D, fx3, xo, S->done);
                std::swap(x, xo);
                residual(x, res, nullptr);
            }
            MgLevel& b = S->L[l + 1];
            if (l + 1 == S->tail)  // the tail kernel restricts res into its first level itself
                S->tail_res = res;
            else
                k_mg3_restrict<<<gsize8(b.nn), kBlock, 0, ctx->stream>>>(b.nx, b.ny, b.nz, res, b.fix, b.r,
                                                                         S->done);
            const float* xc = mg_cycle(ctx, l + 1);
            int k0 = 0;
            if (fuse && a.ye) {  // x + P xc formed where the first post-sweep reads it
                elem2(std::integral_constant<int, kMg3InProlong>{}, a.Ke32, x, xc, nullptr, xo);
                k0 = 1;
            } else {
                k_mg3_prolong<<<gn, kBlock, 0, ctx->stream>>>(a.nx, a.ny, a.nz, x, xc, fx3, xo, S->done);
            }
            std::swap(x, xo);
            for (int k = k0; k < S->nu; k++) {
                residual(x, nullptr, xo);
                std::swap(x, xo);
            }
        };
        if (l == 0) {
            const H8Shape s8 = h8_shape(ctx, sizeof(float));
            if (s8.per)
                run3(Mg3KeTile{&s8});
            else
                run3(Mg3KeShared{ctx->d_Ef, ctx->d_K0f});
        } else {
            run3(Mg3KeFull{a.Ke32});
        }
        return x;
    }
    const uint8_t* fx = l == 0 ? ctx->d_fix : a.fix;
    const unsigned g = gsize(a.nn);
    float *x = a.x, *res = a.res, *xo = a.x2, *ro = a.res2;
    auto sweep = [&](auto ke, const float* xi, const float* ri, const float* xc, float* xout, float* rout) {
        if (l == 0 && a.nn >= kMgTileNodes) {  // a large finest level: LDS-tiled
            constexpr int TI = kMgTile0TI, TJ = kMgTile0TJ;
            const int tilesJ = (a.ny + 1 + TJ - 1) / TJ, tiles = tilesJ * ((a.nx + 1 + TI - 1) / TI);
            const bool zf = l == 0 && xc && S->z64 && S->nu == 1;  // the cycle's last sweep
            k_mg_sweep_tile<decltype(ke), TI, TJ><<<tiles, kBlock, 0, ctx->stream>>>(
                a.nx, a.ny, tilesJ, ke, a.D, fx, S->omega, a.r, xi, ri, xc, xout, rout, S->done,
                zf ? S->r64 : nullptr, zf ? S->z64 : nullptr, zf ? S->zpart : nullptr, a.prol(true));
        } else if (a.nn >= kMgMidNodes) {  // coarse levels: smaller tiles, more workgroups
            constexpr int TI = kMgMidTI, TJ = kMgMidTJ;
            const int tilesJ = (a.ny + 1 + TJ - 1) / TJ, tiles = tilesJ * ((a.nx + 1 + TI - 1) / TI);
            k_mg_sweep_tile<decltype(ke), TI, TJ><<<tiles, kBlock, 0, ctx->stream>>>(
                a.nx, a.ny, tilesJ, ke, a.D, fx, S->omega, a.r, xi, ri, xc, xout, rout, S->done, nullptr, nullptr,
                nullptr, a.prol(true));
        } else {
            k_mg_sweep<<<g, kBlock, 0, ctx->stream>>>(a.nx, a.ny, ke, a.D, fx, S->omega, a.r, xi, ri, xc, xout,
                                                      rout, S->done, a.prol(true));
        }
    };
    auto jac = [&](auto ke, const float* xi, float* xout) {
        k_mg_jacobi<<<g, kBlock, 0, ctx->stream>>>(a.nx, a.ny, ke, a.D, fx, S->omega, a.r, xi, xout, S->done);
    };
    auto run = [&](auto ke) {
        sweep(ke, nullptr, nullptr, nullptr, x, res);
        for (int k = 1; k < S->nu; k++) {
            sweep(ke, x, res, nullptr, xo, ro);
            std::swap(x, xo);
            std::swap(res, ro);
        }
        MgLevel& b = S->L[l + 1];
        if (l + 1 == S->tail)  // the tail kernel restricts res into its first level itself
            S->tail_res = res;
        else
            k_mg_restrict<<<gsize(b.nn), kBlock, 0, ctx->stream>>>(b.nx, b.ny, res, b.fix, b.r, S->done,
                                                                   a.prol(true));
        const float* xc = mg_cycle(ctx, l + 1);
        sweep(ke, x, nullptr, xc, xo, nullptr);
        std::swap(x, xo);
        for (int k = 1; k < S->nu; k++) {
            jac(ke, x, xo);
            std::swap(x, xo);
        }
    };
    if (l == 0)
        run(MgKeShared{ctx->d_Ef, ctx->d_K0f});
    else
        run(MgKeFull{a.Ke32});
    return x;
}

// PCG with z = V(r) (the hierarchy built for the current moduli), stream
// ordered like pcg_device: k_pcg_k1_q4_tile (beta, convergence test on the
// recursive residual, p, K p), k_mg_pcg_update (alpha, x, r, r in FP32), the
// V-cycle, k_mg_pcg_z (z and the sums z.r, r.r); the host reads the done
// flag once per chunk.  b, x nodal; x starts at 0.  T = double: the FP64
// solve (work vectors d_*); T = float: the inner solve of pcg_ir_mg (work
// vectors f_*, the FP32 operator and diagonal).
template <class T>
int pcg_mg_device(pf_ctx* ctx, const T* b, T* x, double eps, int itrmax, PcgRun& out) {
    constexpr bool f32 = std::is_same<T, float>::value;
    MgState* M = ctx->mg;
    const long n = ctx->nv;
    PcgDev* S = (PcgDev*)ctx->d_pcg;
    double* partA = ctx->red.partials;
    double* partB = ctx->red.partials + 2 * kMaxPartials;
    const bool h8 = !is2d(ctx);
    const K1Shape sh = h8 ? K1Shape{0, 0, 0u} : k1_shape(ctx->nx, ctx->ny);
    const H8Shape s8 = h8 ? h8_shape(ctx, sizeof(T)) : H8Shape{};
    const unsigned g1 = h8 ? (s8.fused() ? s8.k1grid() : gsize(ctx->nn)) : sh.grid;
    const unsigned g2 = std::min<unsigned>(gsize(n), (unsigned)k2_cap());
    PF_CHECK(g1 <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    T *r, *z, *p0, *p1, *q;
    const T *Ev, *Kv, *Kg, *D;
    if constexpr (f32) {
        r = ctx->f_r, z = ctx->f_z, p0 = ctx->f_p0, p1 = ctx->f_p1, q = ctx->f_q;
        Ev = ctx->d_Ef, Kv = ctx->d_K0f, Kg = ctx->d_K0gf, D = ctx->f_D;
    } else {
        r = ctx->d_r, z = ctx->d_z, p0 = ctx->d_p0, p1 = ctx->d_p1, q = ctx->d_q;
        Ev = ctx->d_E, Kv = ctx->d_K0, Kg = ctx->d_K0g, D = ctx->d_D;
    }
    float* r32 = M->L[0].r;
    // the finest level's last V-cycle sweep writes z and its sums itself when
    // it is the LDS-tiled quad4 sweep (one sweep per side), else k_mg_pcg_z does
    const bool zfused = !f32 && !h8 && M->nu == 1 && M->L[0].nn >= kMgTileNodes && (int)M->L.size() > 1;
    const unsigned gz = zfused ? (unsigned)(((ctx->ny + kMgTile0TJ) / kMgTile0TJ) *
                                            ((ctx->nx + kMgTile0TI) / kMgTile0TI))
                               : g2;
    PF_CHECK(gz <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    auto cycle_z = [&](const int* done_flag) {
        if (zfused) {
            M->r64 = (const double*)r;
            M->z64 = (double*)z;
            M->zpart = partB;
            mg_cycle(ctx, 0);
            M->r64 = nullptr;
            M->z64 = nullptr;
            M->zpart = nullptr;
        } else {
            k_mg_pcg_z<T><<<g2, kBlock, 0, ctx->stream>>>(n, mg_cycle(ctx, 0), r, z, partB, done_flag);
        }
    };
    // x = 0, r = b (k_pcg_init's z = b ./ D and its sums are replaced by V(b)'s)
    k_pcg_init<T><<<g2, kBlock, 0, ctx->stream>>>(n, b, D, x, r, z, p0, partB, S);
    k_convert<T, float><<<gsize(n), kBlock, 0, ctx->stream>>>(n, b, r32);
    M->done = &S->done;
    cycle_z(nullptr);
    PF_TRY(check_launch(ctx));
    const int chunk = 8;
    int k = 0;
    EventPair ev;
    PF_HIP(ev.create());
    volatile int* hflag = (volatile int*)ctx->h_red;
    hflag[0] = hflag[1] = 0;
    int slot = 0, pending = 0;
    bool done = false;
    int rc = PF_OK;
    while (!done && k < itrmax) {
        const int kend = std::min(itrmax, k + chunk);
        for (; k < kend; k++) {
            T* pold = (k & 1) ? p1 : p0;
            T* pnew = (k & 1) ? p0 : p1;
            if (h8 && s8.fused()) {
                launch_h8_k1_tile<T>(ctx, s8, k, pold, z, pnew, q, Ev, Kg, partB, (int)gz, partA, S, eps);
            } else if (h8) {
                // p = beta p + z in place (head and convergence test), q = K p
                k_pcg_k3<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, p0, z, partB, (int)g2, S, eps);
                k_pcg_k1_h8<T><<<g1, kBlock, 0, ctx->stream>>>(g3(ctx), p0, q, Ev, Kv, ctx->d_fix, partA, S);
                pnew = p0;
            } else {
                k_pcg_k1_q4_tile<T, kTileI, kTileJ><<<g1, kBlock, 0, ctx->stream>>>(
                    ctx->nx, ctx->ny, sh.tilesJ, sh.ntiles, k, pold, z, pnew, q, Ev, Kv, ctx->d_fix, partB, (int)gz,
                    partA, S, eps);
            }
            k_mg_pcg_update<T><<<g2, kBlock, 0, ctx->stream>>>(n, k, x, r, pnew, q, r32, partA, (int)g1, S);
            cycle_z(&S->done);
        }
        if ((rc = check_launch(ctx)) < 0) break;
        if (hipMemcpyAsync((void*)&hflag[slot], &S->done, sizeof(int), hipMemcpyDeviceToHost, ctx->stream) !=
                hipSuccess ||
            hipEventRecord(ev[slot], ctx->stream) != hipSuccess) {
            rc = PF_ERR_HIP;
            break;
        }
        if (pending) {
            hipEventSynchronize(ev[slot ^ 1]);
            if (hflag[slot ^ 1]) done = true;
        }
        pending = 1;
        slot ^= 1;
    }
    M->done = nullptr;
    hipStreamSynchronize(ctx->stream);
    PF_TRY(rc);
    k_pcg_final<<<1, kBlock, 0, ctx->stream>>>(k, partB, (int)gz, S, eps);
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(ctx->h_pcg, S, sizeof(PcgDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    const PcgDev* H = (const PcgDev*)ctx->h_pcg;
    out.iterations = H->iterations;
    out.status = H->status;
    out.rnorm = H->rnorm;
    out.bnorm = H->bnorm;
    return PF_OK;
}

// Multigrid-preconditioned solve to an FP64 true residual eps ||b||: the
// device PCG above stops on its recursive residual; while the true residual
// is above eps ||b|| (at most 4 rounds), a correction K d = b - K x is solved
// the same way and added.
int solve_mg(pf_ctx* ctx, const double* b, double* x, double eps, int itrmax, pf_solve_stats& st) {
    PF_TRY(diag_nodal(ctx, false));
    PF_TRY(mg_build(ctx));
    int rc;
    const double bn = norm_nodal(ctx, b, &rc);
    PF_TRY(rc);
    PcgRun run;
    PF_TRY(pcg_mg_device<double>(ctx, b, x, eps, itrmax, run));
    int total = run.iterations, rounds = 1;
    double tn;
    PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &tn));
    while (tn > eps * bn && rounds < 4 && total < itrmax && std::isfinite(tn)) {
        PF_HIP(hipMemcpyAsync(ctx->d_t1, ctx->d_t0, sizeof(double) * ctx->nv, hipMemcpyDeviceToDevice, ctx->stream));
        double* d = ctx->d_s0;  // the correction (the single-reduction form's buffer, free here)
        PF_TRY(pcg_mg_device<double>(ctx, ctx->d_t1, d, eps * bn / tn, itrmax - total, run));
        k_axpy_d<<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, 1.0, d, x);
        PF_TRY(check_launch(ctx));
        total += run.iterations;
        rounds++;
        PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &tn));
    }
    st.iterations = total;
    st.outer = rounds;
    st.status = (tn <= eps * bn) ? 1 : 2;
    st.rel_residual = bn > 0 ? tn / bn : 0.0;
    return PF_OK;
}

// Multigrid PCG in FP32 (FP32 vectors and operator, the same FP32 V-cycle)
// inside FP64 iterative refinement to an FP64 true residual eps ||b||, as
// pcg_ir does with Jacobi-PCG: each outer step solves K d = r to inner_eps
// in FP32 and adds d in FP64; a step that does not halve the true residual
// is undone and the solve continues with FP64 multigrid corrections.
int pcg_ir_mg(pf_ctx* ctx, const double* b, double* x, double eps, int itrmax, double inner_eps,
              pf_solve_stats& st) {
    // an FP32 inner solve that has not reached inner_eps in this many
    // iterations has stagnated (FP32 cannot resolve contrasts of 1e9 between
    // neighbouring elements): its step is checked and the solve goes on in FP64
    constexpr int kInnerCapMg = 500;
    PF_TRY(diag_nodal(ctx, true));
    PF_TRY(diag_nodal(ctx, false));
    PF_TRY(mg_build(ctx));
    int rc;
    const double bn = norm_nodal(ctx, b, &rc);
    PF_TRY(rc);
    PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * ctx->nv, ctx->stream));
    double rn = bn;
    int outer = 0, total = 0, status = 2, fallbacks = 0;
    bool fp64 = false;
    const int max_outer = 60;
    double* r64 = ctx->d_t0;
    double* d64 = ctx->d_t1;
    PF_TRY(true_residual(ctx, b, x, r64, &rn));
    while (outer < max_outer) {
        if (rn <= eps * bn) {
            status = 1;
            break;
        }
        if (total >= itrmax) break;
        PcgRun run;
        if (!fp64) {
            k_convert<double, float><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, r64, ctx->f_b);
            PF_TRY(pcg_mg_device<float>(ctx, ctx->f_b, ctx->f_x, inner_eps, std::min(kInnerCapMg, itrmax - total),
                                        run));
            total += run.iterations;
            outer++;
            PF_HIP(hipMemcpyAsync(d64, x, sizeof(double) * ctx->nv, hipMemcpyDeviceToDevice, ctx->stream));
            k_axpy_f32<<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->f_x, x);
            PF_TRY(check_launch(ctx));
            double rnew;
            PF_TRY(true_residual(ctx, b, x, r64, &rnew));
            if (std::isfinite(run.rnorm) && std::isfinite(rnew) && rnew <= 0.5 * rn) {
                rn = rnew;
                continue;
            }
            PF_HIP(hipMemcpyAsync(x, d64, sizeof(double) * ctx->nv, hipMemcpyDeviceToDevice, ctx->stream));
            PF_TRY(true_residual(ctx, b, x, r64, &rn));
            fp64 = true;
            fallbacks++;
            continue;
        }
        // FP64 multigrid correction to the relative tolerance that brings the
        // true residual to eps ||b||
        const double rel = std::min(0.5, eps * bn / rn);
        PF_TRY(pcg_mg_device<double>(ctx, r64, d64, rel, itrmax - total, run));
        total += run.iterations;
        outer++;
        k_axpy_d<<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, 1.0, d64, x);
        PF_TRY(check_launch(ctx));
        PF_TRY(true_residual(ctx, b, x, r64, &rn));
    }
    st.iterations = total;
    st.status = status;
    st.outer = outer;
    st.fallbacks = fallbacks;
    st.rel_residual = bn > 0 ? rn / bn : 0.0;
    return PF_OK;
}

// z = V(r) for nodal FP64 vectors (the hierarchy built for the current moduli)
int mg_apply(pf_ctx* ctx, const double* r, double* z) {
    MgLevel& a = ctx->mg->L[0];
    k_d2f<<<gsize(a.nv), kBlock, 0, ctx->stream>>>(a.nv, r, a.r);
    const float* x = mg_cycle(ctx, 0);
    k_f2d<<<gsize(a.nv), kBlock, 0, ctx->stream>>>(a.nv, x, z);
    return check_launch(ctx);
}

double dot_nodal(pf_ctx* ctx, const double* a, const double* b, int* rc);
int optimal_pair(pf_ctx* ctx, const double* r, double* a, double* c);

// M(r) for a nodal FP64 residual r with the current moduli (D, the FP64
// Jacobi diagonal, in ctx->d_D):  t = r ./ D,  y = network field for
// (rho, r / s),  d = a t + c y  with (a, c) minimising the energy norm of the
// error of d over span{t, y}:  [t.Kt t.Ky; t.Ky y.Ky] (a, c) = (t.r, y.r)
// (K e = r makes this computable without e).  d is never worse, in that
// norm, than the best-scaled Jacobi step.  N->w holds y, N->Kw K y, N->dd t
// and N->gd K t on return.
// The pieces of M(r) (stream-ordered, no host synchronisation): N->w = y,
// N->dd = t, N->gd = K t, N->Kw = K y.
// the network's input channels for residual r (scale rs, or *rn_dev / sqrtN)
void net_input(pf_ctx* ctx, const double* rho, const double* r, double rs, const double* rn_dev, double sqrtN) {
    LearnedNet* N = ctx->net;
    if (N->dim == 3)
        k_net_input3<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->nz, rho, r, rs, rn_dev, sqrtN,
                                                                 N->x0);
    else
        k_net_input<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, rho, r, rs, rn_dev, sqrtN, N->x0);
}

// rn: |r| on the host, or (rn_dev non-null) on the device.
// Over the V-cycle the two pieces run side by side: its coarse levels occupy a
// few of the CUs, the network's kernels the others.  They share no buffer that
// either writes, and the caller's stream waits for both, so nothing changes but
// the time: a learned solve at 1024 x 512 takes 14.1 ms, 16.5 one after the other,
// in a process with one context; after other contexts' work, whose streams share
// the process's four hardware queues with these two, 17.2 and 18.0.
int net_parts(pf_ctx* ctx, const double* rho, const double* r, double rn, const double* rn_dev = nullptr) {
    LearnedNet* N = ctx->net;
    const long nv = ctx->nv;
    const double sqrtN = std::sqrt((double)std::max(1, ctx->N));
    const double rs = rn > 0 ? rn / sqrtN : 1.0;
    auto network = [&]() -> int {
        net_input(ctx, rho, r, rs, rn_dev, sqrtN);
        PF_TRY(net_forward(ctx, true));                     // y in N->w
        return apply_nodal(ctx, false, N->w, N->Kw, true);  // K y
    };
    if (!ctx->mg) {
        PF_TRY(network());
        k_div_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, r, ctx->d_D, N->dd);  // t = r ./ D
        PF_TRY(apply_nodal(ctx, false, N->dd, N->gd, true));                    // K t
        return check_launch(ctx);
    }
    if (!N->side) PF_HIP(hipStreamCreate(&N->side));
    if (!N->fork) PF_HIP(hipEventCreateWithFlags(&N->fork, hipEventDisableTiming));
    if (!N->join) PF_HIP(hipEventCreateWithFlags(&N->join, hipEventDisableTiming));
    const hipStream_t own = ctx->stream;
    PF_HIP(hipEventRecord(N->fork, own));
    PF_HIP(hipStreamWaitEvent(N->side, N->fork, 0));
    ctx->stream = N->side;
    const int rc = network();
    ctx->stream = own;
    // joined on every path: what follows on the caller's stream, also after an
    // error, comes after the network's kernels
    const hipError_t e0 = hipEventRecord(N->join, N->side);
    int rv = mg_apply(ctx, r, N->dd);                                            // t = V(r)
    if (rv == PF_OK) rv = apply_nodal(ctx, false, N->dd, N->gd, true);           // K t
    const hipError_t e1 = e0 == hipSuccess ? hipStreamWaitEvent(own, N->join, 0) : e0;
    if (e1 != hipSuccess) hipStreamSynchronize(N->side);
    PF_TRY(rc);
    PF_TRY(rv);
    PF_HIP(e1);
    return check_launch(ctx);
}

int net_apply(pf_ctx* ctx, const double* rho, const double* r, double* d, double* rs_out, double rnorm = -1.0) {
    LearnedNet* N = ctx->net;
    const long nv = ctx->nv;
    int rc = PF_OK;
    const double rn = rnorm >= 0.0 ? rnorm : norm_nodal(ctx, r, &rc);
    PF_TRY(rc);
    const double rs = rn > 0 ? rn / std::sqrt((double)std::max(1, ctx->N)) : 1.0;
    PF_TRY(net_parts(ctx, rho, r, rn));
    double a = 1.0, c = 0.0;
    PF_TRY(optimal_pair(ctx, r, &a, &c));
    k_lincomb_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, a, N->dd, c, N->w, d);
    if (rs_out) *rs_out = rs;
    return check_launch(ctx);
}

double dot_nodal(pf_ctx* ctx, const double* a, const double* b, int* rc) {
    const unsigned g = gsize(ctx->nv);
    k_dot_partials<<<g, kBlock, 0, ctx->stream>>>(ctx->nv, a, b, ctx->red.partials);
    return reduce_host(ctx, ctx->red.partials, (int)g, 1.0, 0.0, rc);
}

// Several sets of dot products (a_k . b_kj) in one batch: the partial-sum
// launches (at most 32 vectors each) and one launch that reduces every dot's
// partials on the device in a fixed order; multidot_batch then copies the
// sums to the host (one synchronisation).
struct DotJob {
    const double* a;
    std::vector<const double*> b;
    std::vector<double> out;
};
// The launches of a batch, with the sums left in `sums` on the device, in
// job order (nd of them).
int multidot_enqueue(pf_ctx* ctx, std::vector<DotJob>& jobs, double* sums, int* nd_out) {
    LearnedNet* N = ctx->net;
    const unsigned g = std::min<unsigned>(gsize(ctx->nv / 2), (unsigned)kMpartGrid);
    DotIdx idx{};
    long off = 0;
    int nd = 0;
    for (int j = 0; j < (int)jobs.size(); j++) {
        const int nbj = (int)jobs[j].b.size();
        jobs[j].out.assign(nbj, 0.0);
        for (int f = 0; f < nbj; f += 32) {
            const int nb = std::min(32, nbj - f);
            PF_CHECK(nd + nb <= kMpartDots, PF_ERR_ARG, "too many dot products in one batch");
            PtrPack P{};
            for (int q = 0; q < nb; q++) {
                P.p[q] = jobs[j].b[f + q];
                idx.off[nd] = (int)off;
                idx.nb[nd] = (short)nb;
                idx.q[nd] = (short)q;
                nd++;
            }
            double* part = N->mpart + off;
            const double* a = jobs[j].a;
            if (nb <= 4)
                k_multidot<4><<<g, kBlock, 0, ctx->stream>>>(ctx->nv, nb, a, P, part);
            else if (nb <= 8)
                k_multidot<8><<<g, kBlock, 0, ctx->stream>>>(ctx->nv, nb, a, P, part);
            else
                k_multidot<32><<<g, kBlock, 0, ctx->stream>>>(ctx->nv, nb, a, P, part);
            off += (long)g * nb;
        }
    }
    if (nd > 0) k_multidot_final<<<nd, kBlock, 0, ctx->stream>>>(N->mpart, (int)g, idx, sums);
    *nd_out = nd;
    return check_launch(ctx);
}

int multidot_batch(pf_ctx* ctx, std::vector<DotJob>& jobs) {
    LearnedNet* N = ctx->net;
    double* sums = N->mpart + (long)kMpartGrid * kMpartDots;
    int nd;
    PF_TRY(multidot_enqueue(ctx, jobs, sums, &nd));
    if (nd == 0) return PF_OK;
    std::vector<double> h(nd);
    PF_HIP(hipMemcpyAsync(h.data(), sums, sizeof(double) * nd, hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    int d = 0;
    for (DotJob& jb : jobs)
        for (double& o : jb.out) o = h[d++];
    return PF_OK;
}

// dots of `a` with up to 32 vectors in one pass
int multidot(pf_ctx* ctx, const double* a, const double* const* b, int nb, double* out) {
    std::vector<DotJob> jobs(1);
    jobs[0].a = a;
    jobs[0].b.assign(b, b + nb);
    PF_TRY(multidot_batch(ctx, jobs));
    for (int j = 0; j < nb; j++) out[j] = jobs[0].out[j];
    return PF_OK;
}

// (a, c) minimising ||a t + c y - e||_K with t = N->dd, y = N->w, K t = N->gd,
// K y = N->Kw and K e = r; falls back to the best-scaled t alone when the
// 2x2 Gram matrix is singular.
int optimal_pair(pf_ctx* ctx, const double* r, double* a, double* c) {
    LearnedNet* N = ctx->net;
    double d1[3], d2[2];
    const double* b1[3] = {N->gd, N->Kw, r};
    PF_TRY(multidot(ctx, N->dd, b1, 3, d1));   // t.Kt, t.Ky, t.r
    const double* b2[2] = {N->Kw, r};
    PF_TRY(multidot(ctx, N->w, b2, 2, d2));    // y.Ky, y.r
    pair_from_sums(d1[0], d1[1], d1[2], d2[0], d2[1], a, c);
    return PF_OK;
}

int net_dataset_alloc(pf_ctx* ctx) {
    LearnedNet* N = ctx->net;
    if (N->cap > 0) return PF_OK;
    const long nv = ctx->nv, ne = ctx->ne;
    // dataset capacity: bounded by memory (about 10 bytes per DOF per pair)
    N->cap = (int)std::max(16L, std::min(1024L, (8L << 30) / (10L * nv)));
    PF_TRY(net_alloc(ctx, N, &N->ds_r, (long)N->cap * nv));
    PF_TRY(net_alloc(ctx, N, &N->ds_e, (long)N->cap * nv));
    PF_TRY(net_alloc(ctx, N, &N->ds_rho, (long)N->cap * ne));
    N->snap_cap = 64;
    PF_TRY(net_alloc(ctx, N, &N->snap_x, (long)N->snap_cap * nv));
    return PF_OK;
}





// Solve the current system with plain FP64 Jacobi-PCG, keeping snapshots of
// x_k; then store (true residual b - K x_k, x* - x_k, rho) pairs.
int net_collect(pf_ctx* ctx, const double* b, int every, int max_pairs, int* count, PcgRun* run_out = nullptr) {
    LearnedNet* N = ctx->net;
    PF_CHECK(N, PF_ERR_STATE, "learned preconditioner not initialised: call pf_precond_init first");
    PF_TRY(net_dataset_alloc(ctx));
    const long nv = ctx->nv;
    const long ne = ctx->ne;
    SnapHook hook;
    hook.every = std::max(1, every);
    hook.max = std::min(N->snap_cap, std::max(0, max_pairs));
    hook.xs = N->snap_x;
    PF_TRY(diag_nodal(ctx, false));
    PcgRun run;
    PF_TRY(pcg_device<double>(ctx, false, b, ctx->d_x, ctx->d_D, ctx->d_r, ctx->d_z, ctx->d_p0, ctx->d_p1, ctx->d_q,
                              1e-10, 100000, run, &hook));
    int added = 0;
    for (int s = 0; s < hook.count; s++) {
        if (hook.iters[s] >= run.iterations) continue;  // converged iterate: e = 0
        if (N->nsamp >= N->cap) break;
        // e = x* - x_k and r = K e: an exactly consistent pair (b - K x_k
        // would carry the final residual of x*, which is not small next to a
        // late r_k)
        const double* xs = N->snap_x + (size_t)s * nv;
        const int slot = N->nsamp++;
        k_sub_scale<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, ctx->d_x, xs, 1.0, ctx->d_t1);
        PF_TRY(apply_nodal(ctx, false, ctx->d_t1, ctx->d_t0, true));
        k_pair_store<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, ctx->d_t0, ctx->d_t1, N->ds_r + (size_t)slot * nv,
                                                           N->ds_e + (size_t)slot * nv);
        k_d2f<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, ctx->d_rho, N->ds_rho + (size_t)slot * ne);
        added++;
    }
    PF_TRY(check_launch(ctx));
    PF_TRY(sync(ctx));
    if (count) *count = N->nsamp;
    if (run_out) *run_out = run;
    return PF_OK;
}

// One Adam step on pair `s`; returns the loss of that pair,
//   L = min_{a,c} ||a t + c y - e||_K^2 / ||e||_K^2   (t = r ./ D, y = network),
// whose gradient at the optimal (a, c) is  dL/dy = 2 c (a K t + c K y - r) / e.r.
int net_train_step(pf_ctx* ctx, int s, float lr, double* loss) {
    LearnedNet* N = ctx->net;
    const long nv = ctx->nv, ne = ctx->ne;
    k_f2d<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, N->ds_rho + (size_t)s * ne, ctx->d_rho);
    PF_TRY(moduli_from_rho(ctx));
    PF_TRY(diag_nodal(ctx, false));
    k_f2d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, N->ds_r + (size_t)s * nv, N->rr);
    k_f2d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, N->ds_e + (size_t)s * nv, N->ee);
    int rc;
    const double rn = norm_nodal(ctx, N->rr, &rc);
    PF_TRY(rc);
    const double rs = rn > 0 ? rn / std::sqrt((double)std::max(1, ctx->N)) : 1.0;
    net_input(ctx, ctx->d_rho, N->rr, rs, nullptr, 1.0);
    PF_TRY(net_forward(ctx, true));                                                                // y in N->w
    PF_TRY(apply_nodal(ctx, false, N->w, N->Kw, true));                                           // K y
    if (ctx->mg) {
        PF_TRY(mg_build(ctx));                                                                     // this pair's moduli
        PF_TRY(mg_apply(ctx, N->rr, N->dd));                                                       // t = V(r)
    } else {
        k_div_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, N->rr, ctx->d_D, N->dd);               // t = r ./ D
    }
    PF_TRY(apply_nodal(ctx, false, N->dd, N->gd, true));                                          // K t
    const double er = dot_nodal(ctx, N->ee, N->rr, &rc);
    PF_TRY(rc);
    double a, c;
    PF_TRY(optimal_pair(ctx, N->rr, &a, &c));
    if (!(er > 0.0) || !std::isfinite(a + c)) {
        *loss = NAN;
        return PF_OK;
    }
    // v = a K t + c K y - r (= K (a t + c y - e));  L = (a t + c y - e).v / e.r
    k_lincomb_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, a, N->gd, c, N->Kw, ctx->d_t1);
    k_axpy_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, -1.0, N->rr, ctx->d_t1);
    k_lincomb_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, a, N->dd, c, N->w, ctx->d_t0);
    k_axpy_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, -1.0, N->ee, ctx->d_t0);
    *loss = dot_nodal(ctx, ctx->d_t0, ctx->d_t1, &rc) / er;
    PF_TRY(rc);
    k_scale_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, 2.0 * c / er, ctx->d_t1);
    k_net_dy_from_nodal<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nn, ctx->ndpn, ctx->d_t1, ctx->d_fix, N->gy);
    PF_TRY(net_backward(ctx));
    N->adam_t++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)N->adam_t), c2 = 1.f - std::pow(b2, (float)N->adam_t);
    AdamLayers P;
    long most = 0;
    for (int i = 0; i < kNetLayers; i++) {
        NetLayer& l = N->L[i];
        P.l[i] = {l.W, l.m, l.v, l.g, l.Wb, l.Wtb, l.ntap, l.cout, l.cin};
        most = std::max(most, l.size());
    }
    k_adam<<<dim3(nblocks(most), kNetLayers), kBlock, 0, ctx->stream>>>(P, lr, b1, b2, 1e-8f, c1, c2);
    return check_launch(ctx);
}

// Synthetic pairs (K v, v) for random smooth fields v at the current moduli.
int net_collect_random(pf_ctx* ctx, int count, uint64_t seed, int* total) {
    LearnedNet* N = ctx->net;
    const long nv = ctx->nv, ne = ctx->ne;
    int levels = 1;
    while ((1 << levels) < std::max(std::max(ctx->nx, ctx->ny), N->dim == 3 ? ctx->nz : 0) / 2) levels++;
    for (int q = 0; q < count && N->nsamp < N->cap; q++) {
        const int slot = N->nsamp++;
        if (N->dim == 3)
            k_random_field3<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->nz, seed + 7919ull * q,
                                                                       levels, ctx->d_fix, ctx->d_t0);
        else
            k_random_field<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, seed + 7919ull * q, levels,
                                                                      ctx->d_fix, ctx->d_t0);
        PF_TRY(apply_nodal(ctx, false, ctx->d_t0, ctx->d_t1, true));
        k_pair_store<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, ctx->d_t1, ctx->d_t0, N->ds_r + (size_t)slot * nv,
                                                           N->ds_e + (size_t)slot * nv);
        k_d2f<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, ctx->d_rho, N->ds_rho + (size_t)slot * ne);
    }
    PF_TRY(check_launch(ctx));
    PF_TRY(sync(ctx));
    if (total) *total = N->nsamp;
    return PF_OK;
}

// Stored directions of the flexible CG.  With the network over the Jacobi
// step, m = 8 needs about 1.4x the iterations of m = 32 on the 96 x 48
// cantilever; over the V-cycle the preconditioner varies far less: at
// 1024 x 512, m = 4 needs the iterations of m = 8 (53) at less traffic per
// iteration, m = 2 needs 62.  CoefPack/PtrPack hold 32.
constexpr int kFcgDirections = 32;
#ifndef PF_FCG_DIRECTIONS_MG
#define PF_FCG_DIRECTIONS_MG 4
#endif
constexpr int kFcgDirectionsMg = PF_FCG_DIRECTIONS_MG;

// Flexible CG (Notay's FCG(m)) with M = the network correction over the base
// step (the multigrid V-cycle after pf_mg_setup, else the Jacobi step
// r ./ D): each new direction is made K-conjugate to the last m stored ones,
// which keeps the Krylov-like acceleration that a varying preconditioner
// would otherwise lose.  Per iteration two batched reductions and no
// operator application of its own (K p comes from K t and K y).  FP64
// vectors; stops on the FP64 true residual; when M breaks down, diverges
// (residual 10x above its best) or stagnates (no halving in `stall` steps)
// Jacobi-PCG takes over from the current iterate.
int pcg_learned(pf_ctx* ctx, const double* b, double* x, double eps, int itrmax, pf_solve_stats& st) {
    LearnedNet* N = ctx->net;
    PF_CHECK(N && N->trained, PF_ERR_STATE, "learned preconditioner has not been trained");
    const long nv = ctx->nv;
    const int m = !ctx->mg ? kFcgDirections : kFcgDirectionsMg;
    if (N->fcg_m != m) {
        N->fP.assign(m, nullptr);
        N->fQ.assign(m, nullptr);
        for (int j = 0; j < m; j++) {
            PF_TRY(net_alloc(ctx, N, &N->fP[j], nv));
            PF_TRY(net_alloc(ctx, N, &N->fQ[j], nv));
        }
        N->fcg_m = m;
    }
    int rc;
    PF_TRY(diag_nodal(ctx, false));
    if (ctx->mg) PF_TRY(mg_build(ctx));
    const double bn = norm_nodal(ctx, b, &rc);
    PF_TRY(rc);
    double *r = ctx->d_r, *z = ctx->d_z;
    PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * nv, ctx->stream));
    PF_HIP(hipMemcpyAsync(r, b, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
    FcgDev* S = N->fcg;
    FcgDev* H = N->fcg_host;
    k_fcg_init<<<1, 1, 0, ctx->stream>>>(S, bn, eps);
    double* sums1 = N->mpart + (long)kMpartGrid * kMpartDots + kMpartDots;
    double* sums2 = sums1 + kMpartDots;
    const unsigned gs = gsize(nv);
    PF_CHECK(gs <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    const int stall = 2000;
    EventPair ev;
    PF_HIP(ev.create());
    // iteration k, stream-ordered: t, y and their images; one batch for the
    // pair (a, c) and z.q_j = a t.q_j + c y.q_j (z = a t + c y is never
    // formed); the direction; p.q and p.r; the step with |r|; the decisions;
    // a copy of the state into pinned slot k mod 2
    auto enqueue = [&](int k) -> int {
        const int nst = std::min(k, m);
        const int slot = k % m;
        double* p = N->fP[slot];
        double* q = N->fQ[slot];
        PtrPack Pp{}, Qp{};
        std::vector<DotJob> jobs(2);
        jobs[0].a = N->dd;
        jobs[0].b = {N->gd, N->Kw, r};
        jobs[1].a = N->w;
        jobs[1].b = {N->Kw, r};
        for (int j = 0; j < nst; j++) {
            const int sj = (k - 1 - j + m) % m;
            Pp.p[j] = N->fP[sj];
            Qp.p[j] = N->fQ[sj];
            jobs[0].b.push_back(N->fQ[sj]);
            jobs[1].b.push_back(N->fQ[sj]);
        }
        PF_TRY(net_parts(ctx, ctx->d_rho, r, 0.0, &S->rn));
        int nd;
        PF_TRY(multidot_enqueue(ctx, jobs, sums1, &nd));
        k_fcg_coef<<<1, 64, 0, ctx->stream>>>(S, sums1, k, m, nst);
        k_fcg_direction<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, nst, S, N->dd, N->w, N->gd, N->Kw, Pp, Qp, p, q);
        std::vector<DotJob> step(1);
        step[0].a = p;
        step[0].b = {q, r};
        PF_TRY(multidot_enqueue(ctx, step, sums2, &nd));
        k_fcg_step<<<gs, kBlock, 0, ctx->stream>>>(nv, S, sums2, p, q, x, r, ctx->red.partials);
        k_fcg_check<<<1, kBlock, 0, ctx->stream>>>(S, sums2, ctx->red.partials, (int)gs, slot, stall);
        PF_HIP(hipMemcpyAsync(&H[k & 1], S, sizeof(FcgDev), hipMemcpyDeviceToHost, ctx->stream));
        PF_HIP(hipEventRecord(ev[k & 1], ctx->stream));
        return check_launch(ctx);
    };
    // iteration k is enqueued while k - 1 runs; the host then reads k - 1's
    // state (once done is set, the FCG launches of a later iteration change
    // nothing)
    int k = 0, kq = 0, status = 2, fallbacks = 0;
    double rn = bn;
    bool fallback = false;
    std::vector<int> pend;
    int erc = PF_OK;
    for (;;) {
        if (kq < itrmax) {
            erc = enqueue(kq);
            if (erc != PF_OK) break;
            pend.push_back(kq++);
        }
        if (pend.empty()) break;  // itrmax reached
        if (pend.size() < 2 && kq < itrmax) continue;
        const int kw = pend.front();
        pend.erase(pend.begin());
        if (hipEventSynchronize(ev[kw & 1]) != hipSuccess) {
            erc = PF_ERR_HIP;
            break;
        }
        const FcgDev st_k = H[kw & 1];
        k = st_k.k;
        rn = st_k.rn;
        if (!st_k.done) continue;
        if (st_k.flag == 2) {
            fallback = true;
            break;
        }
        // confirm on the true residual
        PF_HIP(hipStreamSynchronize(ctx->stream));
        double tn;
        PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &tn));
        if (tn <= eps * bn) {
            status = 1;
            rn = tn;
            break;
        }
        PF_HIP(hipMemcpyAsync(r, ctx->d_t0, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
        double best = st_k.best;
        int since = st_k.since_best;
        bool fb = false;
        if (tn < 0.5 * best) {
            best = tn;
            since = 0;
        } else if (++since >= stall || tn > 10.0 * best) {
            fb = true;
        }
        k_fcg_resume<<<1, 1, 0, ctx->stream>>>(S, tn, best, since, fb ? 1 : 0);
        rn = tn;
        if (fb) {
            k -= 1;
            fallback = true;
            break;
        }
        pend.clear();
        kq = k;
    }
    hipStreamSynchronize(ctx->stream);
    PF_TRY(erc);
    if (fallback) {
        // Jacobi-PCG on the correction K dx = b - K x from the current iterate
        // (from x = 0 when the iterate is not finite)
        fallbacks++;
        double tn;
        PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &tn));
        if (!std::isfinite(tn)) {
            PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * nv, ctx->stream));
            PF_HIP(hipMemcpyAsync(ctx->d_t0, b, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
            tn = bn;
        }
        PcgRun run;
        PF_HIP(hipMemcpyAsync(ctx->d_t1, ctx->d_t0, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
        PF_TRY(pcg_device<double>(ctx, false, ctx->d_t1, N->dd, ctx->d_D, r, z, ctx->d_p0, ctx->d_p1, ctx->d_q,
                                  eps * bn / std::max(tn, 1e-300), std::max(1, itrmax - k), run));
        k_axpy_d<<<gsize(nv), kBlock, 0, ctx->stream>>>(nv, 1.0, N->dd, x);
        k += run.iterations;
        PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &rn));
        status = rn <= eps * bn ? 1 : 2;
    }
    st.iterations = k;
    st.status = status;
    st.fallbacks = fallbacks;
    st.rel_residual = bn > 0 ? rn / bn : 0.0;
    return check_launch(ctx);
}

// Solve K x = b for nodal device vectors b, x with the selected operator.
int solve_nodal(pf_ctx* ctx, int op, const double* b, double* x, double eps, int itrmax, double inner_eps,
                pf_solve_stats* st) {
    auto t0 = std::chrono::steady_clock::now();
    pf_solve_stats s{};
    {
        int rc0;
        double bn0 = norm_nodal(ctx, b, &rc0);
        PF_TRY(rc0);
        PF_CHECK(std::isfinite(bn0), PF_ERR_NUMERIC, "non-finite right-hand side (NaN or Inf in b)");
        if (bn0 == 0.0) {
            // b = 0: x = 0 is exact (the reference would divide 0 by 0 here)
            PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * ctx->nv, ctx->stream));
            s.status = 1;
            PF_TRY(sync(ctx));
            s.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (st) *st = s;
            return PF_OK;
        }
    }
    if (op == PF_OP_EBE64 || op == PF_OP_EBE32) res_enter(ctx);
    if (op == PF_OP_EBE64) {
        PF_TRY(diag_nodal(ctx, false));
        PcgRun run;
        PF_TRY(pcg_device<double>(ctx, false, b, x, ctx->d_D, ctx->d_r, ctx->d_z, ctx->d_p0, ctx->d_p1, ctx->d_q, eps,
                                  itrmax, run));
        s.iterations = run.iterations;
        s.status = run.status;
        s.rel_residual = run.bnorm > 0 ? run.rnorm / run.bnorm : 0.0;
    } else if (op == PF_OP_CSR64) {
        PF_CHECK(ctx->nnz >= 0, PF_ERR_STATE, "no assembled CSR: call pf_assemble_csr first");
        // free-numbered work vectors live in the nodal buffers' storage (N <= nv)
        double *bf = ctx->d_t0, *xf = ctx->d_t1;
        PF_TRY(to_free(ctx, b, bf));
        k_csr_diag<<<gsize(ctx->N), kBlock, 0, ctx->stream>>>(ctx->N, ctx->d_indptr, ctx->d_indices, ctx->d_data,
                                                             ctx->d_D);
        PF_TRY(check_launch(ctx));
        PcgRun run;
        PF_TRY(pcg_device<double>(ctx, true, bf, xf, ctx->d_D, ctx->d_r, ctx->d_z, ctx->d_p0, ctx->d_p1, ctx->d_q, eps,
                                  itrmax, run));
        // true residual with the assembled matrix itself
        const unsigned g = gsize(ctx->N);
        k_csr_residual<<<g, kBlock, 0, ctx->stream>>>(ctx->N, ctx->d_indptr, ctx->d_indices, ctx->d_data, bf, xf,
                                                      ctx->red.partials);
        PF_TRY(check_launch(ctx));
        int rc;
        const double rr = reduce_host(ctx, ctx->red.partials, (int)g, 1.0, 0.0, &rc);
        PF_TRY(rc);
        PF_TRY(to_nodal(ctx, xf, x));
        s.iterations = run.iterations;
        s.status = run.status;
        s.rel_residual = run.bnorm > 0 ? run.rnorm / run.bnorm : 0.0;
        s.true_residual = run.bnorm > 0 ? std::sqrt(rr) / run.bnorm : 0.0;
    } else if (op == PF_OP_EBE32) {
        PF_TRY(pcg_ir(ctx, b, x, eps, itrmax, inner_eps, s));
    } else if (op == PF_OP_LEARNED) {
        PF_TRY(pcg_learned(ctx, b, x, eps, itrmax, s));
    } else if (op == PF_OP_MG) {
        PF_CHECK(ctx->mg, PF_ERR_STATE, "multigrid not set up: call pf_mg_setup first");
        PF_TRY(solve_mg(ctx, b, x, eps, itrmax, s));
    } else if (op == PF_OP_MG32) {
        PF_CHECK(ctx->mg, PF_ERR_STATE, "multigrid not set up: call pf_mg_setup first");
        PF_TRY(pcg_ir_mg(ctx, b, x, eps, itrmax, inner_eps, s));
    } else {
        ctx->err = "unknown operator";
        return PF_ERR_ARG;
    }
    if (op != PF_OP_CSR64) {
        double trn;
        int rc;
        PF_TRY(true_residual(ctx, b, x, ctx->d_t0, &trn));
        double bn = norm_nodal(ctx, b, &rc);
        PF_TRY(rc);
        s.true_residual = bn > 0 ? trn / bn : 0.0;
    }
    PF_TRY(sync(ctx));
    s.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    if (st) *st = s;
    return s.status == 1 ? PF_OK : PF_NOT_CONVERGED;
}

// ------------------------------------------------------------------ OC ----
// The bisection in one resident launch (k_oc_resident), its result in h_oc;
// *ran is false, and nothing has been done, with the projection in the closure, a
// volume that is not a number, more elements than the chip's registers hold, no memory for the column sums or
// a launch that cannot be made or stalled.
int oc_resident(pf_ctx* ctx, const pf_oc_params* prm, int max_steps, const double* x, const double* dfdx,
                const double* dgdx, double* xplus, bool* ran) {
    *ran = false;
    constexpr int NT = kOcResThreads;
    const long ne = ctx->ne, most = (long)ctx->res_wgs * NT;
    if (!res_on(ctx) || ne > 16 * most || prm->beta > 0.0 || max_steps > 1000000) return PF_OK;
    // a volume that divides by zero or scales by infinity is NaN where a term is
    // zero: a single density's here, a whole neighbourhood's in the launched form
    if (!(std::fabs(prm->vf * (double)ne) > 0.0) || !std::isfinite(prm->scale1)) return PF_OK;
    if (!ctx->have_fcol) {
        if (!res_alloc(ctx, &ctx->d_fcol, ne, &ctx->fcol_n)) return PF_OK;
        k_filter_colsum<<<gsize(ne), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->dim, ctx->win, ctx->R, ctx->d_cg, nullptr,
                                                               xplus);
        k_filter_colsum<<<gsize(ne), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->dim, ctx->win, ctx->R, ctx->d_cg, xplus,
                                                               ctx->d_fcol);
        PF_TRY(check_launch(ctx));
        ctx->have_fcol = true;
    }
    // one element per thread while the workgroups last, then 2, 4, 8, 16
    int S = 1;
    while (ne > S * most) S *= 2;
    const void* kern = S == 1   ? (const void*)k_oc_resident<1>
                       : S == 2 ? (const void*)k_oc_resident<2>
                       : S == 4 ? (const void*)k_oc_resident<4>
                       : S == 8 ? (const void*)k_oc_resident<8>
                                : (const void*)k_oc_resident<16>;
    bool ok;
    PF_TRY(res_begin(ctx, 0, &ok));  // no buffer of its own
    OcRes A{};
    A.n = ne;
    A.max_steps = max_steps;
    A.tag = ctx->res_tag;
    ctx->res_tag += (unsigned)max_steps + 1;
    A.iota = prm->iota; A.move = prm->movelimit; A.leps = prm->lambdaeps;
    A.vf = prm->vf; A.scale1 = prm->scale1;
    A.l0 = prm->lambdamin; A.l1 = prm->lambdamax;
    A.x = x; A.dfdx = dfdx; A.dgdx = dgdx; A.col = ctx->d_fcol; A.xplus = xplus;
    A.slots = ctx->res_slots;
    A.R = ctx->d_res;
    A.O = (OcDev*)ctx->d_oc;
    res_force(ctx, 0);
    void* args[] = {&A};
    const unsigned wgs = (unsigned)((ne + (long)NT * S - 1) / ((long)NT * S));
    if (!res_launch(ctx, kern, wgs, NT, args, 0)) return PF_OK;
    PF_HIP(hipMemcpyAsync(ctx->h_oc, ctx->d_oc, sizeof(OcDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->h_res, ctx->d_res, sizeof(ResDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    if (res_gave_up(ctx)) return PF_OK;
    res_ended(ctx);
    *ran = true;
    return PF_OK;
}

int oc_device(pf_ctx* ctx, const pf_oc_params* prm, const double* x, const double* dfdx, const double* dgdx,
              double* xplus, double* lambda_out, int* steps_out) {
    PF_CHECK(ctx->have_filter && !ctx->have_lists, PF_ERR_STATE,
             "the device OC closure filters with the grid rule: call pf_filter_setup first");
    OcDev* S = (OcDev*)ctx->d_oc;
    const int max_steps = prm->max_steps > 0 ? prm->max_steps : 200;
    bool resident;
    res_enter(ctx);
    PF_TRY(oc_resident(ctx, prm, max_steps, x, dfdx, dgdx, xplus, &resident));
    if (!resident) {
        OcDev init{};
        init.l0i = prm->lambdamin;
        init.l1i = prm->lambdamax;
        PF_HIP(hipMemcpyAsync(S, &init, sizeof(OcDev), hipMemcpyHostToDevice, ctx->stream));
        PF_HIP(hipMemsetAsync(xplus, 0, sizeof(double) * ctx->ne, ctx->stream));  // xkp1 starts as zeros (OC.h:81)
    }
    const unsigned g = gsize(ctx->ne);
    const int chunk = 16;
    int k = 0;
    bool done = resident;
    volatile OcDev* H = (volatile OcDev*)ctx->h_oc;
    // quad4: one launch per bisection step (k_oc_step); hex8: the candidate
    // and the filtered volume in two launches
    auto step = [&](int kk) {
        if (is2d(ctx)) {
            k_oc_step<<<g, kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->win, ctx->R, ctx->d_cg, kk, x, dfdx, dgdx,
                                                    prm->iota, prm->movelimit, prm->lambdaeps, prm->vf, prm->scale1,
                                                    prm->beta, ctx->red.partials, (int)g, xplus, S);
            return;
        }
        k_oc_xplus<<<g, kBlock, 0, ctx->stream>>>(ctx->ne, kk, x, dfdx, dgdx, prm->iota, prm->movelimit,
                                                 prm->lambdaeps, prm->scale1, ctx->red.partials, (int)g, xplus, S);
        k_oc_volume_h8<<<g, kBlock, 0, ctx->stream>>>(g3(ctx), ctx->win, ctx->R, ctx->d_cg, xplus, prm->vf,
                                                     prm->scale1, prm->beta, ctx->red.partials, S);
    };
    while (!done && k < max_steps) {
        int kend = std::min(max_steps, k + chunk);
        for (; k < kend; k++) step(k);
        PF_TRY(check_launch(ctx));
        PF_HIP(hipMemcpyAsync((void*)H, S, sizeof(OcDev), hipMemcpyDeviceToHost, ctx->stream));
        PF_TRY(sync(ctx));
        done = H->done != 0;
    }
    if (!done) {
        // the last step's decision has not been applied yet; apply it once more
        if (is2d(ctx))
            step(k);
        else
            k_oc_xplus<<<g, kBlock, 0, ctx->stream>>>(ctx->ne, k, x, dfdx, dgdx, prm->iota, prm->movelimit,
                                                     prm->lambdaeps, prm->scale1, ctx->red.partials, (int)g, xplus,
                                                     S);
        PF_HIP(hipMemcpyAsync((void*)H, S, sizeof(OcDev), hipMemcpyDeviceToHost, ctx->stream));
        PF_TRY(sync(ctx));
    }
    if (!H->done) {
        if (lambda_out) *lambda_out = H->lambda_last;
        if (steps_out) *steps_out = H->steps;
        ctx->err = "OC bisection did not reach lambdaeps within max_steps";
        return PF_NOT_CONVERGED;
    }
    if (lambda_out) *lambda_out = H->lambda_last;
    if (steps_out) *steps_out = H->steps;
    if (H->status == 1) {
        ctx->err = "OC bisection: the volume constraint is violated at every tested lambda; lambda reached "
                   "lambdamax (bracket too small)";
        return PF_NOT_CONVERGED;
    }
    if (H->status == 2) {
        ctx->err = "OC bisection: the volume constraint is satisfied at every tested lambda; lambda reached "
                   "lambdamin (bracket too large at its lower end)";
        return PF_NOT_CONVERGED;
    }
    return PF_OK;
}

int filter_device(pf_ctx* ctx, const double* in, double* out) {
    if (ctx->have_lists) {
        k_filter_lists<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->ne, ctx->d_fptr, ctx->d_fidx, ctx->d_fw, in,
                                                                  out);
        return check_launch(ctx);
    }
    PF_CHECK(ctx->have_filter, PF_ERR_STATE, "no filter: call pf_filter_setup or pf_filter_set_lists first");
    if (is2d(ctx))
        k_filter_q4<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->win, ctx->R, ctx->d_cg, in,
                                                               out);
    else
        k_filter_h8<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->win, ctx->R, ctx->d_cg, in, out);
    return check_launch(ctx);
}

int moduli_from_rho(pf_ctx* ctx) {
    k_E_from_rho<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->ne, ctx->d_rho, ctx->E1, ctx->E0, ctx->p, ctx->d_E,
                                                            ctx->d_Ef);
    PF_TRY(check_launch(ctx));
    ctx->have_E = true;
    return PF_OK;
}

// f = scale0 sum_e E_e u_e^T K0 u_e and dfdrho (device, nodal u).
int comp_sens_device(pf_ctx* ctx, const double* u, double scale0, double* dfdrho, double* f) {
    const double coef = ((-scale0) * ctx->p) * ((-ctx->E0) + ctx->E1);
    const unsigned g = gsize(ctx->ne);
    if (is2d(ctx))
        k_comp_sens_q4<false><<<g, kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, u, ctx->d_E, ctx->d_rho, ctx->d_K0, coef,
                                                     ctx->p - 1.0, dfdrho, ctx->red.partials);
    else
        k_comp_sens_h8<false><<<g, kBlock, 0, ctx->stream>>>(g3(ctx), u, ctx->d_E, ctx->d_rho, ctx->d_K0, coef, ctx->p - 1.0,
                                                     dfdrho, ctx->red.partials);
    PF_TRY(check_launch(ctx));
    int rc;
    *f = reduce_host(ctx, ctx->red.partials, (int)g, scale0, 0.0, &rc);
    return rc;
}

// ---------------------------------------------------------------- MMA -----
}  // namespace

struct MmaState {
    pf_mma_params prm{};
    bool conlin = false;  // CONLIN's approximation (same interior-point driver)
    int k = 0;
    double previousvalue = 0.0;
    long n = 0;
    double *xkm1 = nullptr, *xkm2 = nullptr, *L = nullptr, *U = nullptr, *alpha = nullptr, *beta = nullptr;
    double *p0 = nullptr, *q0 = nullptr, *p = nullptr, *q = nullptr, *x = nullptr, *gsi = nullptr, *ita = nullptr;
    double *G = nullptr, *Dx = nullptr, *dlx = nullptr, *dx = nullptr, *dgsi = nullptr, *dita = nullptr;
    double *xp = nullptr, *gp = nullptr, *ip = nullptr;
    std::vector<double> hpart;
    std::vector<double**> buffers() {
        return {&xkm1, &xkm2, &L, &U, &alpha, &beta, &p0, &q0, &p, &q, &x,
                &gsi, &ita, &G, &Dx, &dlx, &dx, &dgsi, &dita, &xp, &gp, &ip};
    }
};

namespace {

void mma_free(MmaState* M) {
    if (!M) return;
    for (double** b : M->buffers()) dfree(*b);
    delete M;
}

// Fixed-order host sum of K-wide workgroup partials.
int host_partials(pf_ctx* ctx, const double* part, int nparts, int K, double* out, bool is_max = false) {
    MmaState* M = ctx->mma;
    M->hpart.resize((size_t)nparts * K);
    PF_HIP(hipMemcpyAsync(M->hpart.data(), part, sizeof(double) * nparts * K, hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    for (int k = 0; k < K; k++) {
        double s = 0.0;
        for (int i = 0; i < nparts; i++) {
            double v = M->hpart[(size_t)i * K + k];
            if (is_max) s = (s < v) ? v : s;
            else s += v;
        }
        out[k] = s;
    }
    return PF_OK;
}

double max5(double a, double b, double c, double d, double e) {
    double r = a;
    if (r < b) r = b;
    if (r < c) r = c;
    if (r < d) r = d;
    if (r < e) r = e;
    return r;
}

// The update in one resident launch (k_mma_resident); *ran is false, and the
// state as it was, when the variables do not fit the registers of the chip or
// the launch cannot be made or stalled.
int mma_update_resident(pf_ctx* ctx, double* xk, const double* dfdx, double g, const double* dgdx, int* steps,
                        int* status, bool* ran) {
    MmaState* M = ctx->mma;
    const pf_mma_params& P = M->prm;
    *ran = false;
    const int max_newton = P.max_newton > 0 ? P.max_newton : 500;
    constexpr int NT = kMmaResThreads;
    const long most = (long)ctx->res_wgs * NT;
    if (!res_on(ctx) || M->n > 4 * most || max_newton > 100000) return PF_OK;
    // one variable per thread while the workgroups last, then two, then four
    const int S = M->n <= most ? 1 : M->n <= 2 * most ? 2 : 4;
    const void* kern = M->conlin ? (S == 1 ? (const void*)k_mma_resident<1, true>
                                    : S == 2 ? (const void*)k_mma_resident<2, true>
                                             : (const void*)k_mma_resident<4, true>)
                                 : (S == 1 ? (const void*)k_mma_resident<1, false>
                                    : S == 2 ? (const void*)k_mma_resident<2, false>
                                             : (const void*)k_mma_resident<4, false>);
    bool ok;
    PF_TRY(res_begin(ctx, 0, &ok));  // no buffer of its own
    MmaRes A{};
    A.n = M->n;
    A.early = M->k < 2;
    A.max_newton = max_newton;
    A.tag = ctx->res_tag;
    ctx->res_tag += 1 + 52u * (unsigned)max_newton;  // two exchanges and at most 50 trials a step
    A.a0 = P.a0; A.a = P.a; A.c = P.c; A.d = P.d;
    A.xmin = P.xmin; A.xmax = P.xmax; A.raa0 = P.raa0; A.albefa = P.albefa; A.move = P.move;
    A.asyinit = P.asyinit; A.asydecr = P.asydecr; A.asyincr = P.asyincr;
    A.g = g;
    A.xk = xk; A.xkm1 = M->xkm1; A.xkm2 = M->xkm2; A.L = M->L; A.U = M->U;
    A.dfdx = dfdx; A.dgdx = dgdx;
    A.xo = M->x; A.Lo = M->alpha; A.Uo = M->beta;
    A.slots = ctx->res_slots;
    A.R = ctx->d_res;
    res_force(ctx, 0);
    void* args[] = {&A};
    const unsigned wgs = (unsigned)((M->n + (long)NT * S - 1) / ((long)NT * S));
    if (!res_launch(ctx, kern, wgs, NT, args, 0)) return PF_OK;
    PF_HIP(hipMemcpyAsync(ctx->h_res, ctx->d_res, sizeof(ResDev), hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    if (res_gave_up(ctx)) return PF_OK;
    res_ended(ctx);
    *steps = (int)ctx->h_res->v[0];
    *status = (int)ctx->h_res->v[1];
    *ran = true;
    return PF_OK;
}

// The new variables (M->x) and the state for the next update.
int mma_accept(pf_ctx* ctx, double* xk, double f) {
    MmaState* M = ctx->mma;
    M->previousvalue = f;
    M->k++;
    const size_t eb = sizeof(double) * M->n;
    std::swap(M->xkm1, M->xkm2);
    PF_HIP(hipMemcpyAsync(M->xkm1, xk, eb, hipMemcpyDeviceToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(xk, M->x, eb, hipMemcpyDeviceToDevice, ctx->stream));
    return sync(ctx);
}

// MMA<T>::UpdateVariables (MMA.h:116-419) for m = 1 on device arrays.
int mma_update_device(pf_ctx* ctx, double* xk, double f, const double* dfdx, double g, const double* dgdx,
                      int* steps_out) {
    MmaState* M = ctx->mma;
    PF_CHECK(M, PF_ERR_STATE, "MMA not initialised: call pf_mma_init first");
    const long n = M->n;
    const pf_mma_params& P = M->prm;
    const double a = P.a, c = P.c, d = P.d, a0 = P.a0;
    {
        int steps = 0, status = 0;
        bool ran;
        res_enter(ctx);
        PF_TRY(mma_update_resident(ctx, xk, dfdx, g, dgdx, &steps, &status, &ran));
        if (ran) {
            if (steps_out) *steps_out = steps;
            if (status) {
                ctx->err = M->conlin ? "CONLIN interior-point loop reached max_newton"
                                     : "MMA interior-point loop reached max_newton";
                return PF_NOT_CONVERGED;
            }
            if (!M->conlin) {
                std::swap(M->L, M->alpha);
                std::swap(M->U, M->beta);
            }
            return mma_accept(ctx, xk, f);
        }
    }
    const unsigned gg = gsize(n);
    double* part = ctx->red.partials;
    if (M->conlin)
        k_conlin_prep<<<gg, kBlock, 0, ctx->stream>>>(n, xk, P.xmin, P.xmax, P.move, dfdx, dgdx, M->alpha, M->beta,
                                                     M->p0, M->q0, M->p, M->q, part);
    else
        k_mma_prep<<<gg, kBlock, 0, ctx->stream>>>(n, M->k < 2, xk, M->xkm1, M->xkm2, M->L, M->U, P.xmin, P.xmax,
                                                  P.asyinit, P.asydecr, P.asyincr, P.albefa, P.move, P.raa0, dfdx,
                                                  dgdx, M->alpha, M->beta, M->p0, M->q0, M->p, M->q, part);
    PF_TRY(check_launch(ctx));
    double Sb;
    PF_TRY(host_partials(ctx, part, (int)gg, 1, &Sb));
    const double b = -g + Sb;
    double eps = 1.0, y = 1.0, z = 1.0, zeta = 1.0, lam = 1.0, s = 1.0;
    double mu = (1.0 < 0.5 * c) ? 0.5 * c : 1.0;
    k_mma_start<<<gg, kBlock, 0, ctx->stream>>>(n, M->alpha, M->beta, M->x, M->gsi, M->ita);
    PF_TRY(check_launch(ctx));
    auto kkt = [&](double Ksum, double gsum, double yv, double zv, double lv, double mv, double zetav, double sv) {
        double norm = Ksum;
        double t;
        t = c + d * yv - lv - mv; norm += t * t;
        t = gsum - a * zv - yv + sv - b; norm += t * t;
        t = mv * yv - eps; norm += t * t;
        t = lv * sv - eps; norm += t * t;
        t = a0 - zetav - (0.0 + lv * a); norm += t * t;
        t = zetav * zv - eps; norm += t * t;
        return std::sqrt(norm);
    };
    int l = 0;
    const int max_newton = P.max_newton > 0 ? P.max_newton : 500;
    for (; eps > 1.0e-7; l++) {
        if (l >= max_newton) {
            ctx->err = M->conlin ? "CONLIN interior-point loop reached max_newton"
                                 : "MMA interior-point loop reached max_newton";
            if (steps_out) *steps_out = l;
            return PF_NOT_CONVERGED;
        }
        if (M->conlin)
            k_conlin_newton_a<<<gg, kBlock, 0, ctx->stream>>>(n, lam, eps, M->x, M->gsi, M->ita, M->alpha, M->beta,
                                                             M->p0, M->q0, M->p, M->q, M->G, M->Dx, M->dlx, part);
        else
            k_mma_newton_a<<<gg, kBlock, 0, ctx->stream>>>(n, lam, eps, M->x, M->gsi, M->ita, M->alpha, M->beta,
                                                          M->L, M->U, M->p0, M->q0, M->p, M->q, M->G, M->Dx, M->dlx,
                                                          part);
        PF_TRY(check_launch(ctx));
        double S[4];
        PF_TRY(host_partials(ctx, part, (int)gg, 4, S));
        double Dy = d + mu / y;
        double Dl = s / lam;
        double dly = c + d * y - lam - eps / y;
        double dlz = a0 - eps / z - (0.0 + lam * a);
        double dll = -a * z - y - b + eps / lam;
        dll += S[0];
        double Dlly = Dl + 1.0 / Dy;
        double dlly = dll + dly / Dy;
        double A00 = 0.0 + S[1];
        A00 += Dlly;
        double dlam, dz;
        mma_solve2(A00, a, a, -zeta / z, dlly - S[2], dlz, dlam, dz);
        k_mma_newton_b<<<gg, kBlock, 0, ctx->stream>>>(n, dlam, eps, M->x, M->gsi, M->ita, M->alpha, M->beta, M->G,
                                                      M->Dx, M->dlx, M->dx, M->dgsi, M->dita, part);
        PF_TRY(check_launch(ctx));
        double txmax;
        PF_TRY(host_partials(ctx, part, (int)gg, 1, &txmax, true));
        double dy = dlam / Dy - dly / Dy;
        double dmu = -mu * dy / y - mu + eps / y;
        double ds = -s * dlam / lam - s + eps / lam;
        double dzeta = -zeta * dz / z - zeta + eps / z;
        double tymax = 0.0;
        {
            double t = -1.01 * dy / y, t2 = -1.01 * dlam / lam, t3 = -1.01 * dmu / mu, t4 = -1.01 * ds / s;
            if (t < t2) t = t2;
            if (t < t3) t = t3;
            if (t < t4) t = t4;
            if (tymax < t) tymax = t;
        }
        double tau = 1.0 / max5(1.0, txmax, tymax, -1.01 * dz / z, -1.01 * dzeta / zeta);
        double deltawl = kkt(S[3], S[0], y, z, lam, mu, zeta, s);
        double yp = y, lp = lam, mp = mu, sp = s, zp = z, zetap = zeta, dw1 = 0.0;
        for (int ll = 0; ll < 50; ll++) {
            yp = y + tau * dy;
            lp = lam + tau * dlam;
            mp = mu + tau * dmu;
            sp = s + tau * ds;
            zp = z + tau * dz;
            zetap = zeta + tau * dzeta;
            if (M->conlin)
                k_conlin_trial<<<gg, kBlock, 0, ctx->stream>>>(n, tau, lp, eps, M->x, M->gsi, M->ita, M->dx,
                                                              M->dgsi, M->dita, M->alpha, M->beta, M->p0, M->q0,
                                                              M->p, M->q, M->xp, M->gp, M->ip, part);
            else
                k_mma_trial<<<gg, kBlock, 0, ctx->stream>>>(n, tau, lp, eps, M->x, M->gsi, M->ita, M->dx, M->dgsi,
                                                           M->dita, M->alpha, M->beta, M->L, M->U, M->p0, M->q0,
                                                           M->p, M->q, M->xp, M->gp, M->ip, part);
            PF_TRY(check_launch(ctx));
            double T[2];
            PF_TRY(host_partials(ctx, part, (int)gg, 2, T));
            dw1 = kkt(T[0], T[1], yp, zp, lp, mp, zetap, sp);
            if (dw1 < deltawl) break;
            tau *= 0.5;
        }
        std::swap(M->x, M->xp);
        std::swap(M->gsi, M->gp);
        std::swap(M->ita, M->ip);
        y = yp; z = zp; lam = lp; mu = mp; zeta = zetap; s = sp;
        if (dw1 < 0.9 * eps) eps *= 0.1;
        else eps *= 1.0;
    }
    if (steps_out) *steps_out = l;
    return mma_accept(ctx, xk, f);
}

int mma_init_device(pf_ctx* ctx, const pf_mma_params* prm, bool conlin = false) {
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_CHECK(prm && prm->m == 1, PF_ERR_UNSUPPORTED, "MMA on the device supports one constraint (m = 1)");
    PF_CHECK(prm->xmax > prm->xmin, PF_ERR_ARG, "MMA: xmax must exceed xmin");
    if (!ctx->mma || ctx->mma->n != ctx->ne) {
        mma_free(ctx->mma);
        ctx->mma = new MmaState();
        ctx->mma->n = ctx->ne;
        for (double** b : ctx->mma->buffers()) PF_TRY(dalloc(ctx, b, ctx->ne));
    }
    MmaState* M = ctx->mma;
    M->prm = *prm;
    M->conlin = conlin;
    M->k = 0;
    M->previousvalue = 0.0;
    const size_t eb = sizeof(double) * ctx->ne;
    PF_HIP(hipMemsetAsync(M->xkm1, 0, eb, ctx->stream));
    PF_HIP(hipMemsetAsync(M->xkm2, 0, eb, ctx->stream));
    PF_HIP(hipMemsetAsync(M->L, 0, eb, ctx->stream));
    PF_HIP(hipMemsetAsync(M->U, 0, eb, ctx->stream));
    return sync(ctx);
}

// ============================================== allocation-free scratch ==
// Device scratch of pf_compliance_sens_dev_noalloc: the per-workgroup
// partial sums of the compliance.  A file-scope device array, so that entry
// point needs no device allocation; every GPU the library runs on holds its
// own copy (8 KiB) until the process ends.  Host code never passes the
// array's name to a kernel: it is a host-side stand-in, and the device
// address is taken once per device with hipGetSymbolAddress
// (noalloc_scratch_init, called by pf_create with the device current).
constexpr int kNoAllocPartials = 1024;
static_assert(kNoAllocPartials >= grid_cap(), "a grid-stride launch must fit the static partials");
static __device__ __align__(256) double scratch[kNoAllocPartials];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

int noalloc_scratch_init(pf_ctx* ctx) {
    PF_CHECK(ctx->device < kMaxDevices, PF_ERR_UNSUPPORTED, "device index beyond the static scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[ctx->device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            ctx->err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return PF_ERR_HIP;
        }
        g_scratch_ptr[ctx->device] = (double*)p;
    }
    ctx->noalloc_scratch = g_scratch_ptr[ctx->device];
    return PF_OK;
}

}  // namespace

// =================================================================== ABI ==
extern "C" {

const char* pf_build_info(void) {
    return "pansfem2_amd: gfx950, hipcc -O3, FP64 kernels without contraction, packed-fp32 disabled";
}

int pf_create(pf_ctx** out, int device) {
    if (!out) return PF_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PF_ERR_HIP;
    if (device < 0 || device >= ndev) return PF_ERR_ARG;
    pf_ctx* ctx = new pf_ctx();
    ctx->device = device;
    int rc = set_device(ctx);
    if (rc == PF_OK && hipStreamCreate(&ctx->stream) != hipSuccess) rc = PF_ERR_HIP;
    // the partial sums, then the resident solves' slots and scalars
    constexpr long kResWords = 2L * 4 * kResMaxWg * 2;
    static_assert(sizeof(ResDev) % 8 == 0, "whole words");
    if (rc == PF_OK)
        rc = dalloc(ctx, &ctx->red.partials, 8L * kMaxPartials + kResWords + (long)sizeof(ResDev) / 8);
    if (rc == PF_OK) {
        ctx->res_slots = (u64*)(ctx->red.partials + 8L * kMaxPartials);
        ctx->d_res = (ResDev*)(ctx->res_slots + kResWords);
        if (hipMemset(ctx->res_slots, 0, kResWords * 8) != hipSuccess) rc = PF_ERR_HIP;  // tags start at 1
    }
    if (rc == PF_OK) rc = dalloc(ctx, &ctx->red.counter, 1);
    if (rc == PF_OK) rc = dalloc(ctx, &ctx->red.out, 16);
    if (rc == PF_OK && hipMalloc((void**)&ctx->d_pcg, sizeof(PcgDev)) != hipSuccess) rc = PF_ERR_NOMEM;
    if (rc == PF_OK && hipMalloc((void**)&ctx->d_oc, sizeof(OcDev)) != hipSuccess) rc = PF_ERR_NOMEM;
    if (rc == PF_OK && hipHostMalloc((void**)&ctx->h_pcg, sizeof(PcgDev)) != hipSuccess) rc = PF_ERR_NOMEM;
    if (rc == PF_OK && hipHostMalloc((void**)&ctx->h_oc, sizeof(OcDev)) != hipSuccess) rc = PF_ERR_NOMEM;
    if (rc == PF_OK && hipHostMalloc((void**)&ctx->h_red, sizeof(double) * 16 + sizeof(ResDev)) != hipSuccess)
        rc = PF_ERR_NOMEM;
    if (rc == PF_OK) ctx->h_res = (ResDev*)(ctx->h_red + 16);
    if (rc == PF_OK && hipMemset(ctx->d_pcg, 0, sizeof(PcgDev)) != hipSuccess) rc = PF_ERR_HIP;
    if (rc == PF_OK) rc = noalloc_scratch_init(ctx);
    if (rc == PF_OK) {
        int coop = 0, cus = 0;
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device);
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
        ctx->res_wgs = coop ? std::min(cus, kResMaxWg) : 0;
    }
    if (rc != PF_OK) {
        pf_destroy(ctx);
        return rc;
    }
    *out = ctx;
    return PF_OK;
}

int pf_destroy(pf_ctx* ctx) {
    if (!ctx) return PF_OK;
    hipSetDevice(ctx->device);
    if (ctx->stream) hipStreamSynchronize(ctx->stream);
    free_grid(ctx);
    release_net(ctx);
    mma_free(ctx->mma);
    ctx->mma = nullptr;
    dfree(ctx->d_K0);
    dfree(ctx->d_K0f);
    dfree(ctx->d_K0g);
    dfree(ctx->d_K0gf);
    dfree(ctx->d_K0m);
    dfree(ctx->d_K0mf);
    dfree(ctx->red.partials);
    dfree(ctx->red.counter);
    dfree(ctx->red.out);
    if (ctx->d_pcg) hipFree(ctx->d_pcg);
    if (ctx->d_oc) hipFree(ctx->d_oc);
    if (ctx->h_pcg) hipHostFree(ctx->h_pcg);
    if (ctx->h_oc) hipHostFree(ctx->h_oc);
    if (ctx->h_red) hipHostFree(ctx->h_red);
    if (ctx->stream) hipStreamDestroy(ctx->stream);
    delete ctx;
    return PF_OK;
}

const char* pf_last_error(pf_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int pf_grid2d(pf_ctx* ctx, int nx, int ny, double lx, double ly) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(nx >= 1 && ny >= 1 && lx > 0 && ly > 0, PF_ERR_ARG, "pf_grid2d: nx, ny >= 1 and lx, ly > 0 required");
    PF_CHECK((long)(nx + 1) * (ny + 1) * 2 < (1L << 31), PF_ERR_ARG, "pf_grid2d: grid exceeds int32 DOF numbering");
    PF_TRY(set_device(ctx));
    free_grid(ctx);
    ctx->dim = 2;
    ctx->nx = nx; ctx->ny = ny; ctx->nz = 0;
    ctx->lx = lx; ctx->ly = ly; ctx->lz = 0;
    ctx->nn = (long)(nx + 1) * (ny + 1);
    ctx->ne = (long)nx * ny;
    ctx->ndpn = 2;
    ctx->nd = 8;
    ctx->nv = ctx->nn * 2;
    PF_TRY(alloc_grid(ctx));
    k_centroids_q4<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(nx, ny, lx, ly, ctx->d_cg);
    PF_TRY(check_launch(ctx));
    return sync(ctx);
}

int pf_grid3d(pf_ctx* ctx, int nx, int ny, int nz, double lx, double ly, double lz) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(nx >= 1 && ny >= 1 && nz >= 1 && lx > 0 && ly > 0 && lz > 0, PF_ERR_ARG,
             "pf_grid3d: nx, ny, nz >= 1 and lx, ly, lz > 0 required");
    PF_CHECK((long)(nx + 1) * (ny + 1) * (nz + 1) * 3 < (1L << 31), PF_ERR_ARG,
             "pf_grid3d: grid exceeds int32 DOF numbering");
    PF_TRY(set_device(ctx));
    free_grid(ctx);
    ctx->dim = 3;
    ctx->nx = nx; ctx->ny = ny; ctx->nz = nz;
    ctx->lx = lx; ctx->ly = ly; ctx->lz = lz;
    ctx->nn = (long)(nx + 1) * (ny + 1) * (nz + 1);
    ctx->ne = (long)nx * ny * nz;
    ctx->ndpn = 3;
    ctx->nd = 24;
    ctx->nv = ctx->nn * 3;
    PF_TRY(alloc_grid(ctx));
    k_centroids_h8<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(g3(ctx), lx, ly, lz, ctx->d_cg);
    PF_TRY(check_launch(ctx));
    return sync(ctx);
}

int pf_set_dirichlet(pf_ctx* ctx, const int32_t* node, const int32_t* dof, int nfixed, int32_t* n_free) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_CHECK(nfixed == 0 || (node && dof), PF_ERR_ARG, "null fixed list");
    std::vector<uint8_t> fix(ctx->nn, 0);
    for (int k = 0; k < nfixed; k++) {
        PF_CHECK(node[k] >= 0 && node[k] < ctx->nn && dof[k] >= 0 && dof[k] < ctx->ndpn, PF_ERR_ARG,
                 "pf_set_dirichlet: node/dof out of range");
        fix[node[k]] |= (uint8_t)(1u << dof[k]);
    }
    PF_TRY(set_device(ctx));
    PF_TRY(upload_dofmap(ctx, fix));
    if (n_free) *n_free = ctx->N;
    return PF_OK;
}

int pf_get_dofmap(pf_ctx* ctx, int32_t* n2g) {
    if (!ctx || !n2g) return PF_ERR_ARG;
    PF_CHECK(!ctx->h_n2g.empty(), PF_ERR_STATE, "no DOF map");
    std::memcpy(n2g, ctx->h_n2g.data(), sizeof(int32_t) * ctx->h_n2g.size());
    return PF_OK;
}

int pf_set_point_loads(pf_ctx* ctx, const int32_t* node, const int32_t* dof, const double* value, int n) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->N > 0, PF_ERR_STATE, "no DOF map");
    std::vector<double> F(ctx->nv, 0.0);
    for (int k = 0; k < n; k++) {
        PF_CHECK(node[k] >= 0 && node[k] < ctx->nn && dof[k] >= 0 && dof[k] < ctx->ndpn, PF_ERR_ARG,
                 "pf_set_point_loads: node/dof out of range");
        long idx = (long)node[k] * ctx->ndpn + dof[k];
        if (ctx->h_n2g[idx] != -1) F[idx] += value[k];  // Assembling.h:151-158
    }
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_load, F.data(), sizeof(double) * ctx->nv, hipMemcpyHostToDevice, ctx->stream));
    return sync(ctx);
}

int pf_get_load(pf_ctx* ctx, double* F_free) {
    if (!ctx || !F_free) return PF_ERR_ARG;
    PF_CHECK(ctx->N > 0, PF_ERR_STATE, "no DOF map");
    PF_TRY(set_device(ctx));
    PF_TRY(to_free(ctx, ctx->d_load, ctx->d_t0));
    PF_HIP(hipMemcpyAsync(F_free, ctx->d_t0, sizeof(double) * ctx->N, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_set_element_matrix(pf_ctx* ctx, const double* K0, int nd) {
    if (!ctx || !K0) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_CHECK(nd == ctx->nd, PF_ERR_ARG, "pf_set_element_matrix: nd does not match the grid's element");
    PF_TRY(set_device(ctx));
    ctx->h_K0.assign(K0, K0 + nd * nd);
    std::vector<float> k32(nd * nd);
    for (int i = 0; i < nd * nd; i++) k32[i] = (float)K0[i];
    PF_TRY(dalloc(ctx, &ctx->d_K0, nd * nd));
    PF_TRY(dalloc(ctx, &ctx->d_K0f, nd * nd));
    PF_HIP(hipMemcpyAsync(ctx->d_K0, K0, sizeof(double) * nd * nd, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_K0f, k32.data(), sizeof(float) * nd * nd, hipMemcpyHostToDevice, ctx->stream));
    if (nd == 24) {
        std::vector<double> g64(nd * nd);
        std::vector<float> g32(nd * nd);
        h8_pack_k0(K0, g64.data());
        h8_pack_k0(K0, g32.data());
        PF_TRY(dalloc(ctx, &ctx->d_K0g, nd * nd));
        PF_TRY(dalloc(ctx, &ctx->d_K0gf, nd * nd));
        PF_HIP(hipMemcpyAsync(ctx->d_K0g, g64.data(), sizeof(double) * nd * nd, hipMemcpyHostToDevice, ctx->stream));
        PF_HIP(hipMemcpyAsync(ctx->d_K0gf, g32.data(), sizeof(float) * nd * nd, hipMemcpyHostToDevice, ctx->stream));
        // the MFMA operator's A fragments, then the parity blocks
        std::vector<double> m64(768 + kH8ParityCoefs, 0.0);
        std::vector<float> m32(768 + kH8ParityCoefs, 0.f);
        h8m_pack_k0(K0, m64.data());
        h8m_pack_k0(K0, m32.data());
        const bool parity = h8_parity_pack(K0, m64.data() + 768);
        for (int i = 0; i < kH8ParityCoefs; i++) m32[768 + i] = (float)m64[768 + i];
        const long nm = (long)m64.size();
        ctx->d_K0p = nullptr;  // inside d_K0m and d_K0mf, which the next lines free
        ctx->d_K0pf = nullptr;
        PF_TRY(dalloc(ctx, &ctx->d_K0m, nm));
        PF_TRY(dalloc(ctx, &ctx->d_K0mf, nm));
        PF_HIP(hipMemcpyAsync(ctx->d_K0m, m64.data(), sizeof(double) * nm, hipMemcpyHostToDevice, ctx->stream));
        PF_HIP(hipMemcpyAsync(ctx->d_K0mf, m32.data(), sizeof(float) * nm, hipMemcpyHostToDevice, ctx->stream));
        ctx->d_K0p = parity ? ctx->d_K0m + 768 : nullptr;
        ctx->d_K0pf = parity ? ctx->d_K0mf + 768 : nullptr;
    }
    return sync(ctx);
}

int pf_element_stiffness(pf_ctx* ctx, int e, double E, double nu, double t, double* Ke) {
    if (!ctx || !Ke) return PF_ERR_ARG;
    PF_CHECK(ctx->dim == 2 || ctx->dim == 3, PF_ERR_STATE, "no grid");
    PF_CHECK(e >= 0 && e < ctx->ne, PF_ERR_ARG, "element id out of range");
    PF_TRY(set_device(ctx));
    const int nd2 = ctx->nd * ctx->nd;
    double* dK;
    PF_HIP(hipMalloc((void**)&dK, sizeof(double) * nd2));
    // compute only element e: one workgroup, one active thread
    if (is2d(ctx))
        k_ke_one_q4<<<1, 64, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->lx, ctx->ly, e, E, nu, t, dK);
    else
        k_ke_one_h8<<<1, 64, 0, ctx->stream>>>(g3(ctx), ctx->lx, ctx->ly, ctx->lz, e, E, nu, dK);
    hipError_t le = hipGetLastError();
    hipError_t ce = hipMemcpyAsync(Ke, dK, sizeof(double) * nd2, hipMemcpyDeviceToHost, ctx->stream);
    hipError_t se = hipStreamSynchronize(ctx->stream);
    hipFree(dK);
    PF_HIP(le);
    PF_HIP(ce);
    PF_HIP(se);
    return PF_OK;
}

int pf_set_material(pf_ctx* ctx, double E1, double E0, double p, double nu, double t) {
    if (!ctx) return PF_ERR_ARG;
    ctx->E1 = E1; ctx->E0 = E0; ctx->p = p; ctx->nu = nu; ctx->t = t;
    return PF_OK;
}

int pf_set_density(pf_ctx* ctx, const double* rho) {
    if (!ctx || !rho) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    for (long e = 0; e < ctx->ne; e++)
        PF_CHECK(std::isfinite(rho[e]), PF_ERR_NUMERIC, "pf_set_density: non-finite density");
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_rho, rho, sizeof(double) * ctx->ne, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(moduli_from_rho(ctx));
    ctx->nnz = ctx->nnz >= 0 ? -2 : ctx->nnz;  // values out of date
    return sync(ctx);
}

int pf_set_moduli(pf_ctx* ctx, const double* E) {
    if (!ctx || !E) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    for (long e = 0; e < ctx->ne; e++)
        PF_CHECK(std::isfinite(E[e]), PF_ERR_NUMERIC, "pf_set_moduli: non-finite modulus");
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_E, E, sizeof(double) * ctx->ne, hipMemcpyHostToDevice, ctx->stream));
    k_convert<double, float><<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->ne, ctx->d_E, ctx->d_Ef);
    PF_TRY(check_launch(ctx));
    ctx->have_E = true;
    return sync(ctx);
}

// CSR structure in closed form on the grid, values gathered per row from
// the element matrices in ascending element id (Assembling.h:46-66 summed
// from 0.0, then CSR(LILCSR&) sorted by column, CSR.h:92-105).  ke_host:
// caller-given element matrices (ne x nd x nd); NULL: computed on the device
// in the reference's arithmetic from the current moduli.
int assemble_csr(pf_ctx* ctx, const double* ke_host, int64_t* nnz) {
    const int N = ctx->N;
    dfree(ctx->d_indptr); dfree(ctx->d_indices); dfree(ctx->d_data);
    ctx->nnz = -1;
    PF_TRY(dalloc(ctx, &ctx->d_indptr, N + 1));
    int32_t* rowlen = nullptr;
    PF_TRY(dalloc(ctx, &rowlen, N));
    if (is2d(ctx))
        k_csr_count_q4<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->d_n2g, ctx->d_fix, rowlen);
    else
        k_csr_count_h8<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->d_n2g, ctx->d_fix, rowlen);
    k_scan<<<1, 1024, 0, ctx->stream>>>(rowlen, ctx->d_indptr, N);
    int32_t total = 0;
    hipError_t e1 = hipGetLastError();
    hipError_t e2 = hipMemcpyAsync(&total, ctx->d_indptr + N, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream);
    hipError_t e3 = hipStreamSynchronize(ctx->stream);
    hipFree(rowlen);
    PF_HIP(e1);
    PF_HIP(e2);
    PF_HIP(e3);
    PF_TRY(dalloc(ctx, &ctx->d_indices, std::max<long>(total, 1)));
    PF_TRY(dalloc(ctx, &ctx->d_data, std::max<long>(total, 1)));
    const long kesz = ctx->ne * (long)ctx->nd * ctx->nd;
    PF_TRY(dalloc(ctx, &ctx->d_ke_all, kesz));
    if (ke_host) {
        PF_HIP(hipMemcpyAsync(ctx->d_ke_all, ke_host, sizeof(double) * kesz, hipMemcpyHostToDevice, ctx->stream));
    } else if (is2d(ctx)) {
        k_ke_all_q4<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->lx, ctx->ly, ctx->d_E, ctx->nu,
                                                               ctx->t, ctx->d_ke_all);
    } else {
        k_ke_all_h8<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->lx, ctx->ly, ctx->lz, ctx->d_E, ctx->nu,
                                                               ctx->d_ke_all);
    }
    if (is2d(ctx))
        k_csr_fill_q4<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->d_n2g, ctx->d_indptr,
                                                                 ctx->d_ke_all, ctx->d_indices, ctx->d_data);
    else
        k_csr_fill_h8<<<gsize(ctx->nn), kBlock, 0, ctx->stream>>>(g3(ctx), ctx->d_n2g, ctx->d_indptr, ctx->d_ke_all,
                                                                 ctx->d_indices, ctx->d_data);
    PF_TRY(check_launch(ctx));
    PF_TRY(sync(ctx));
    dfree(ctx->d_ke_all);
    ctx->nnz = total;
    if (nnz) *nnz = total;
    return PF_OK;
}

int pf_assemble_csr(pf_ctx* ctx, int64_t* nnz) {
    if (!ctx) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_TRY(set_device(ctx));
    return assemble_csr(ctx, nullptr, nnz);
}

int pf_assemble_csr_elements(pf_ctx* ctx, const double* ke_all, int64_t* nnz) {
    if (!ctx || !ke_all) return PF_ERR_ARG;
    PF_CHECK(ctx->dim == 2 || ctx->dim == 3, PF_ERR_STATE, "no grid: call pf_grid2d/pf_grid3d first");
    PF_CHECK(ctx->N > 0, PF_ERR_STATE, "no DOF map: call pf_set_dirichlet first");
    PF_TRY(set_device(ctx));
    return assemble_csr(ctx, ke_all, nnz);
}

int pf_get_csr(pf_ctx* ctx, int32_t* indptr, int32_t* indices, double* data) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->nnz >= 0, PF_ERR_STATE, "no assembled CSR");
    PF_TRY(set_device(ctx));
    if (indptr)
        PF_HIP(hipMemcpyAsync(indptr, ctx->d_indptr, sizeof(int32_t) * (ctx->N + 1), hipMemcpyDeviceToHost, ctx->stream));
    if (indices)
        PF_HIP(hipMemcpyAsync(indices, ctx->d_indices, sizeof(int32_t) * ctx->nnz, hipMemcpyDeviceToHost, ctx->stream));
    if (data) PF_HIP(hipMemcpyAsync(data, ctx->d_data, sizeof(double) * ctx->nnz, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_apply_K(pf_ctx* ctx, int op, const double* x_free, double* y_free) {
    if (!ctx || !x_free || !y_free) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, op != PF_OP_CSR64));
    PF_TRY(set_device(ctx));
    const int N = ctx->N;
    PF_HIP(hipMemcpyAsync(ctx->d_t1, x_free, sizeof(double) * N, hipMemcpyHostToDevice, ctx->stream));
    if (op == PF_OP_CSR64) {
        PF_CHECK(ctx->nnz >= 0, PF_ERR_STATE, "no assembled CSR: call pf_assemble_csr first");
        k_csr_spmv<<<gsize(N), kBlock, 0, ctx->stream>>>(N, ctx->d_indptr, ctx->d_indices, ctx->d_data, ctx->d_t1,
                                                        ctx->d_t0);
        PF_TRY(check_launch(ctx));
    } else if (op == PF_OP_EBE64) {
        PF_TRY(to_nodal(ctx, ctx->d_t1, ctx->d_x));
        PF_TRY(apply_nodal(ctx, false, ctx->d_x, ctx->d_q, true));
        PF_TRY(to_free(ctx, ctx->d_q, ctx->d_t0));
    } else if (op == PF_OP_EBE32) {
        PF_TRY(to_nodal(ctx, ctx->d_t1, ctx->d_x));
        k_convert<double, float><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->d_x, ctx->f_x);
        PF_TRY(apply_nodal(ctx, true, ctx->f_x, ctx->f_q, true));
        k_convert<float, double><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->f_q, ctx->d_q);
        PF_TRY(to_free(ctx, ctx->d_q, ctx->d_t0));
    } else {
        ctx->err = "unknown operator";
        return PF_ERR_ARG;
    }
    PF_HIP(hipMemcpyAsync(y_free, ctx->d_t0, sizeof(double) * N, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_pcg_dev(pf_ctx* ctx, int op, const double* b_free_dev, double* x_free_dev, double eps, int itrmax,
               pf_solve_stats* st) {
    if (!ctx || !b_free_dev || !x_free_dev) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, op != PF_OP_CSR64));
    PF_CHECK(itrmax >= 0 && eps >= 0, PF_ERR_ARG, "pf_pcg: itrmax and eps must be non-negative");
    PF_TRY(set_device(ctx));
    PF_TRY(to_nodal(ctx, b_free_dev, ctx->d_b));
    int rc = solve_nodal(ctx, op, ctx->d_b, ctx->d_x, eps, itrmax, 1e-5, st);
    if (rc < 0) return rc;
    PF_TRY(to_free(ctx, ctx->d_x, x_free_dev));
    PF_TRY(sync(ctx));
    return rc;
}

int pf_mg_setup(pf_ctx* ctx, int nu, double omega) {
    if (!ctx) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, false));
    PF_TRY(set_device(ctx));
    if (nu == 0) {
        mg_free(ctx);
        return PF_OK;
    }
    PF_CHECK(nu >= 1 && nu <= 8, PF_ERR_ARG, "pf_mg_setup: nu must be 1..8 (0 to switch off)");
    // damped Jacobi smooths only for omega < 2 / lambda_max(D^-1 K): about 0.67
    // for quad4 and 0.48 for hex8 (lambda_max about 3 and 4.2)
    if (omega <= 0.0) omega = is2d(ctx) ? 0.6 : 0.4;
    PF_CHECK(omega <= 1.0, PF_ERR_ARG, "pf_mg_setup: omega must be at most 1 (or <= 0 for the default)");
    const int rc = mg_plan(ctx, nu, (float)omega, ctx->mg_prolong);
    if (rc < 0) mg_free(ctx);
    return rc;
}

int pf_mg_set_prolongation(pf_ctx* ctx, int mode) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(mode == PF_MG_PROLONG_BILINEAR || mode == PF_MG_PROLONG_STIFFNESS, PF_ERR_ARG,
             "pf_mg_set_prolongation: PF_MG_PROLONG_BILINEAR or PF_MG_PROLONG_STIFFNESS");
    ctx->mg_prolong = mode;
    if (ctx->mg && ctx->mg->prolong != mode) {
        PF_TRY(set_device(ctx));
        const int nu = ctx->mg->nu;
        const float omega = ctx->mg->omega;
        const int rc = mg_plan(ctx, nu, omega, mode);
        if (rc < 0) mg_free(ctx);
        return rc;
    }
    return PF_OK;
}

int pf_mg_set_residual_form(pf_ctx* ctx, int form) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(form == PF_MG_RESIDUAL_AUTO || form == PF_MG_RESIDUAL_NODE || form == PF_MG_RESIDUAL_ELEMENT, PF_ERR_ARG,
             "pf_mg_set_residual_form: PF_MG_RESIDUAL_AUTO, PF_MG_RESIDUAL_NODE or PF_MG_RESIDUAL_ELEMENT");
    const bool change = ctx->mg_resid != form;
    ctx->mg_resid = form;
    if (ctx->mg && change) {  // the element form's buffers are planned with the hierarchy
        PF_TRY(set_device(ctx));
        const int nu = ctx->mg->nu;
        const float omega = ctx->mg->omega;
        const int rc = mg_plan(ctx, nu, omega, ctx->mg->prolong);
        if (rc < 0) mg_free(ctx);
        return rc;
    }
    return PF_OK;
}

int pf_mg_build(pf_ctx* ctx) {
    if (!ctx) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_TRY(set_device(ctx));
    return mg_build(ctx);
}

int pf_mg_apply(pf_ctx* ctx, const double* r_free, double* z_free) {
    if (!ctx || !r_free || !z_free) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_TRY(set_device(ctx));
    PF_TRY(mg_build(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_t1, r_free, sizeof(double) * ctx->N, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(to_nodal(ctx, ctx->d_t1, ctx->d_r));
    PF_TRY(mg_apply(ctx, ctx->d_r, ctx->d_z));
    PF_TRY(to_free(ctx, ctx->d_z, ctx->d_t0));
    PF_HIP(hipMemcpyAsync(z_free, ctx->d_t0, sizeof(double) * ctx->N, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_mg_level(pf_ctx* ctx, int level, int* levels, int* nx, int* ny, int* nz, double* Ke, float* D,
                uint8_t* fix) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->mg, PF_ERR_STATE, "multigrid not set up: call pf_mg_setup first");
    PF_TRY(set_device(ctx));
    MgState* S = ctx->mg;
    if (levels) *levels = (int)S->L.size();
    PF_CHECK(level >= 0 && level < (int)S->L.size(), PF_ERR_ARG, "pf_mg_level: no such level");
    const MgLevel& a = S->L[level];
    if (nx) *nx = a.nx;
    if (ny) *ny = a.ny;
    if (nz) *nz = a.nz;
    if (Ke) {
        PF_CHECK(level >= 1, PF_ERR_ARG, "pf_mg_level: level 0's element matrices are E_e K0");
        const long kes = a.nz > 0 ? 576 : 64;
        PF_HIP(hipMemcpyAsync(Ke, a.Ke64, sizeof(double) * a.ne * kes, hipMemcpyDeviceToHost, ctx->stream));
    }
    if (D) PF_HIP(hipMemcpyAsync(D, a.D, sizeof(float) * a.nv, hipMemcpyDeviceToHost, ctx->stream));
    if (fix)
        PF_HIP(hipMemcpyAsync(fix, level == 0 ? ctx->d_fix : a.fix, a.nn, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_set_pcg_form(pf_ctx* ctx, int form) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(form >= PF_PCG_SCALINGCG && form <= PF_PCG_SINGLE_REDUCTION_RECOMPUTED, PF_ERR_ARG, "pf_set_pcg_form: unknown form");
    ctx->pcg_form = form;
    return PF_OK;
}

int pf_set_resident(pf_ctx* ctx, int mode, int after) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(mode >= PF_RESIDENT_AUTO && mode <= PF_RESIDENT_REFUSED && after >= 0, PF_ERR_ARG,
             "pf_set_resident: unknown mode");
    ctx->res_mode = mode;
    ctx->res_after = after;
    return PF_OK;
}

int pf_resident_runs(pf_ctx* ctx, int64_t* done, int64_t* gave_way) {
    if (!ctx) return PF_ERR_ARG;
    if (done) *done = ctx->res_done;
    if (gave_way) *gave_way = ctx->res_gave;
    return PF_OK;
}

int pf_set_h8_operator(pf_ctx* ctx, int kind) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(kind == PF_H8_OP_AUTO || kind == PF_H8_OP_VALU || kind == PF_H8_OP_MFMA, PF_ERR_ARG,
             "pf_set_h8_operator: unknown kind");
    ctx->h8_op = kind;
    return PF_OK;
}

int pf_pcg(pf_ctx* ctx, int op, const double* b_free, double* x_free, double eps, int itrmax, pf_solve_stats* st) {
    if (!ctx || !b_free || !x_free) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, op != PF_OP_CSR64));
    for (int i = 0; i < ctx->N; i++) PF_CHECK(std::isfinite(b_free[i]), PF_ERR_NUMERIC, "pf_pcg: non-finite b");
    PF_TRY(set_device(ctx));
    double *bd = nullptr, *xd = nullptr;
    PF_HIP(hipMalloc((void**)&bd, sizeof(double) * ctx->N));
    PF_HIP(hipMalloc((void**)&xd, sizeof(double) * ctx->N));
    int rc = PF_OK;
    if (hipMemcpyAsync(bd, b_free, sizeof(double) * ctx->N, hipMemcpyHostToDevice, ctx->stream) != hipSuccess)
        rc = PF_ERR_HIP;
    if (rc == PF_OK) rc = pf_pcg_dev(ctx, op, bd, xd, eps, itrmax, st);
    if (rc >= 0 && hipMemcpyAsync(x_free, xd, sizeof(double) * ctx->N, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
        rc = PF_ERR_HIP;
    hipStreamSynchronize(ctx->stream);
    hipFree(bd);
    hipFree(xd);
    return rc;
}

int pf_compliance_sens(pf_ctx* ctx, const double* u_free, double scale0, double* f, double* dfdrho) {
    if (!ctx || !u_free || !f || !dfdrho) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_t1, u_free, sizeof(double) * ctx->N, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(to_nodal(ctx, ctx->d_t1, ctx->d_x));
    PF_TRY(comp_sens_device(ctx, ctx->d_x, scale0, ctx->d_e0, f));
    PF_HIP(hipMemcpyAsync(dfdrho, ctx->d_e0, sizeof(double) * ctx->ne, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_compliance_sens_dev_noalloc(pf_ctx* ctx, const double* u_free_dev, double scale0, double* f_dev,
                                   double* dfdrho_dev) {
    if (!ctx || !u_free_dev || !f_dev || !dfdrho_dev) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_CHECK(ctx->noalloc_scratch, PF_ERR_STATE, "no static scratch address for this device");
    PF_TRY(set_device(ctx));
    const unsigned g = gsize(ctx->ne);
    PF_CHECK(g <= (unsigned)kNoAllocPartials, PF_ERR_ARG,
             "pf_compliance_sens_dev_noalloc: the launch needs more partial sums than the static scratch holds");
    const double coef = ((-scale0) * ctx->p) * ((-ctx->E0) + ctx->E1);
    // every workgroup writes its own partial, so nothing in the scratch
    // needs clearing; the sum reads only this launch's g entries
    double* part = ctx->noalloc_scratch;
    if (is2d(ctx))
        k_comp_sens_q4<true><<<g, kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, u_free_dev, ctx->d_E, ctx->d_rho,
                                                            ctx->d_K0, coef, ctx->p - 1.0, dfdrho_dev, part,
                                                            ctx->d_n2g);
    else
        k_comp_sens_h8<true><<<g, kBlock, 0, ctx->stream>>>(g3(ctx), u_free_dev, ctx->d_E, ctx->d_rho, ctx->d_K0,
                                                            coef, ctx->p - 1.0, dfdrho_dev, part, ctx->d_n2g);
    PF_TRY(check_launch(ctx));
    k_reduce_final<<<1, kBlock, 0, ctx->stream>>>(part, (int)g, 1, scale0, 0.0, f_dev);
    PF_TRY(check_launch(ctx));
    return sync(ctx);
}

int pf_filter_setup(pf_ctx* ctx, double R) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_CHECK(R > 0 && std::isfinite(R), PF_ERR_ARG, "pf_filter_setup: R must be positive");
    double h = std::min(ctx->lx / ctx->nx, ctx->ly / ctx->ny);
    if (ctx->dim == 3) h = std::min(h, ctx->lz / ctx->nz);
    ctx->R = R;
    // offsets beyond floor(R/h) elements are farther than R (centroid spacing
    // is h up to rounding of the node coordinates)
    ctx->win = (int)std::floor(R / h * (1.0 + 1e-9));
    ctx->have_filter = true;
    ctx->have_lists = false;
    ctx->have_fcol = false;
    return PF_OK;
}

int pf_sensitivity_filter(pf_ctx* ctx, int scheme, const double* s, const double* dfds, double* out) {
    if (!ctx || !s || !dfds || !out) return PF_ERR_ARG;
    PF_CHECK(scheme == 1 || scheme == 2, PF_ERR_ARG, "pf_sensitivity_filter: scheme 1 or 2");
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_CHECK(ctx->have_lists || (ctx->have_filter && is2d(ctx)), PF_ERR_STATE,
             "pf_sensitivity_filter: needs neighbour lists (pf_filter_set_lists) or the quad4 grid rule");
    PF_TRY(set_device(ctx));
    const long ne = ctx->ne;
    const size_t eb = sizeof(double) * ne;
    PF_HIP(hipMemcpyAsync(ctx->d_e0, s, eb, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e1, dfds, eb, hipMemcpyHostToDevice, ctx->stream));
    if (ctx->have_lists)
        k_sensfilter_lists<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, ctx->d_fptr, ctx->d_fidx, ctx->d_fw, ctx->d_e0,
                                                                 ctx->d_e1, scheme, ctx->d_e2);
    else
        k_sensfilter_q4<<<gsize(ne), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->win, ctx->R, ctx->d_cg,
                                                              ctx->d_e0, ctx->d_e1, scheme, ctx->d_e2);
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(out, ctx->d_e2, eb, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_filter_set_lists(pf_ctx* ctx, const int32_t* ptr, const int32_t* idx, const double* w) {
    if (!ctx || !ptr || !idx || !w) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    const long ne = ctx->ne;
    PF_CHECK(ptr[0] == 0, PF_ERR_ARG, "pf_filter_set_lists: ptr[0] must be 0");
    for (long e = 0; e < ne; e++)
        PF_CHECK(ptr[e + 1] > ptr[e], PF_ERR_ARG, "pf_filter_set_lists: every element needs at least one neighbour");
    const long total = ptr[ne];
    double wmin = 0.0;
    for (long k = 0; k < total; k++) {
        PF_CHECK(idx[k] >= 0 && idx[k] < ne, PF_ERR_ARG, "pf_filter_set_lists: neighbour index out of range");
        PF_CHECK(std::isfinite(w[k]), PF_ERR_ARG, "pf_filter_set_lists: non-finite weight");
        wmin = std::min(wmin, w[k]);
    }
    PF_TRY(set_device(ctx));
    dfree(ctx->d_fptr); dfree(ctx->d_fidx); dfree(ctx->d_fw);
    PF_TRY(dalloc(ctx, &ctx->d_fptr, ne + 1));
    PF_TRY(dalloc(ctx, &ctx->d_fidx, total));
    PF_TRY(dalloc(ctx, &ctx->d_fw, total));
    PF_HIP(hipMemcpyAsync(ctx->d_fptr, ptr, sizeof(int32_t) * (ne + 1), hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_fidx, idx, sizeof(int32_t) * total, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_fw, w, sizeof(double) * total, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(sync(ctx));
    ctx->have_lists = true;
    return PF_OK;
}

int pf_filter(pf_ctx* ctx, int mode, const double* in, double* out) {
    if (!ctx || !in || !out) return PF_ERR_ARG;
    PF_CHECK(mode == PF_FILTER_VARIABLES || mode == PF_FILTER_SENSITIVITIES, PF_ERR_ARG, "pf_filter: bad mode");
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_e0, in, sizeof(double) * ctx->ne, hipMemcpyHostToDevice, ctx->stream));
    // both modes are the same row-normalised stencil (DensityFilter.h:45-71)
    PF_TRY(filter_device(ctx, ctx->d_e0, ctx->d_e1));
    PF_HIP(hipMemcpyAsync(out, ctx->d_e1, sizeof(double) * ctx->ne, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_oc_update(pf_ctx* ctx, double* x, const double* dfdx, const double* dgdx, const pf_oc_params* prm,
                 double* lambda_out, int* steps_out) {
    if (!ctx || !x || !dfdx || !dgdx || !prm) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_TRY(set_device(ctx));
    size_t bytes = sizeof(double) * ctx->ne;
    PF_HIP(hipMemcpyAsync(ctx->d_e0, x, bytes, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e1, dfdx, bytes, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e2, dgdx, bytes, hipMemcpyHostToDevice, ctx->stream));
    int rc = oc_device(ctx, prm, ctx->d_e0, ctx->d_e1, ctx->d_e2, ctx->d_e3, lambda_out, steps_out);
    if (rc < 0) return rc;
    PF_HIP(hipMemcpyAsync(x, ctx->d_e3, bytes, hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    return rc;
}

int pf_oc_candidate(pf_ctx* ctx, const double* x, const double* dfdx, const double* dgdx, double lambda,
                    double iota, double movelimit, double* xplus) {
    if (!ctx || !x || !dfdx || !dgdx || !xplus) return PF_ERR_ARG;
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_TRY(set_device(ctx));
    const long ne = ctx->ne;
    PF_HIP(hipMemcpyAsync(ctx->d_e0, x, sizeof(double) * ne, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e1, dfdx, sizeof(double) * ne, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e2, dgdx, sizeof(double) * ne, hipMemcpyHostToDevice, ctx->stream));
    k_oc_candidate<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, ctx->d_e0, ctx->d_e1, ctx->d_e2, lambda, iota, movelimit,
                                                         ctx->d_e4);
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(xplus, ctx->d_e4, sizeof(double) * ne, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_mma_init(pf_ctx* ctx, const pf_mma_params* prm) {
    if (!ctx || !prm) return PF_ERR_ARG;
    PF_TRY(set_device(ctx));
    return mma_init_device(ctx, prm);
}

int pf_conlin_init(pf_ctx* ctx, const pf_mma_params* prm) {
    if (!ctx || !prm) return PF_ERR_ARG;
    PF_TRY(set_device(ctx));
    return mma_init_device(ctx, prm, true);
}

int pf_conlin_update(pf_ctx* ctx, double* x, double f, const double* dfdx, double g, const double* dgdx,
                     int* newton_steps) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->mma && ctx->mma->conlin, PF_ERR_STATE, "CONLIN not initialised: call pf_conlin_init first");
    return pf_mma_update(ctx, x, f, dfdx, g, dgdx, newton_steps);
}

int pf_mma_get_state(pf_ctx* ctx, int* k, double* previousvalue, double* xkm1, double* xkm2, double* L, double* U) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->mma, PF_ERR_STATE, "MMA/CONLIN not initialised: call pf_mma_init or pf_conlin_init first");
    PF_TRY(set_device(ctx));
    MmaState* M = ctx->mma;
    const size_t eb = sizeof(double) * M->n;
    if (k) *k = M->k;
    if (previousvalue) *previousvalue = M->previousvalue;
    if (xkm1) PF_HIP(hipMemcpyAsync(xkm1, M->xkm1, eb, hipMemcpyDeviceToHost, ctx->stream));
    if (xkm2) PF_HIP(hipMemcpyAsync(xkm2, M->xkm2, eb, hipMemcpyDeviceToHost, ctx->stream));
    if (L) PF_HIP(hipMemcpyAsync(L, M->L, eb, hipMemcpyDeviceToHost, ctx->stream));
    if (U) PF_HIP(hipMemcpyAsync(U, M->U, eb, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_mma_set_state(pf_ctx* ctx, int k, double previousvalue, const double* xkm1, const double* xkm2,
                     const double* L, const double* U) {
    if (!ctx || !xkm1 || !xkm2 || !L || !U) return PF_ERR_ARG;
    PF_CHECK(ctx->mma, PF_ERR_STATE, "MMA/CONLIN not initialised: call pf_mma_init or pf_conlin_init first");
    PF_CHECK(k >= 0, PF_ERR_ARG, "pf_mma_set_state: k must be non-negative");
    MmaState* M = ctx->mma;
    for (long i = 0; i < M->n; i++)
        PF_CHECK(std::isfinite(xkm1[i]) && std::isfinite(xkm2[i]) && std::isfinite(L[i]) && std::isfinite(U[i]),
                 PF_ERR_NUMERIC, "pf_mma_set_state: non-finite state");
    PF_TRY(set_device(ctx));
    const size_t eb = sizeof(double) * M->n;
    PF_HIP(hipMemcpyAsync(M->xkm1, xkm1, eb, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(M->xkm2, xkm2, eb, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(M->L, L, eb, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(M->U, U, eb, hipMemcpyHostToDevice, ctx->stream));
    M->k = k;
    M->previousvalue = previousvalue;
    return sync(ctx);
}

int pf_mma_update(pf_ctx* ctx, double* x, double f, const double* dfdx, double g, const double* dgdx,
                  int* newton_steps) {
    if (!ctx || !x || !dfdx || !dgdx) return PF_ERR_ARG;
    PF_CHECK(ctx->mma, PF_ERR_STATE, "MMA not initialised: call pf_mma_init first");
    PF_TRY(set_device(ctx));
    size_t bytes = sizeof(double) * ctx->ne;
    PF_HIP(hipMemcpyAsync(ctx->d_e0, x, bytes, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e1, dfdx, bytes, hipMemcpyHostToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(ctx->d_e2, dgdx, bytes, hipMemcpyHostToDevice, ctx->stream));
    int rc = mma_update_device(ctx, ctx->d_e0, f, ctx->d_e1, g, ctx->d_e2, newton_steps);
    if (rc < 0) return rc;
    PF_HIP(hipMemcpyAsync(x, ctx->d_e0, bytes, hipMemcpyDeviceToHost, ctx->stream));
    PF_TRY(sync(ctx));
    return rc;
}

void pf_simp_default_params(pf_simp_params* p) {
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->E1 = 1.0; p->E0 = 1e-9; p->nu = 0.3; p->t = 1.0; p->p = 3.0;
    p->vf = 0.5; p->R = 1.5; p->scale0 = 1.0; p->scale1 = 1.0;
    p->cg_eps = 1e-10; p->cg_itrmax = 100000;
    p->use_mma = 0; p->solver = PF_OP_EBE64; p->mixed = 0; p->inner_eps = 1e-5; p->learned = 0;
    p->stop_on_convergence = 0;
    p->oc.iota = 0.5; p->oc.lambdamin = 0.0; p->oc.lambdamax = 1e9; p->oc.lambdaeps = 1e-3; p->oc.movelimit = 0.2;
    p->oc.vf = 0.5; p->oc.scale1 = 1.0; p->oc.max_steps = 200;
    p->mma.m = 1; p->mma.a0 = 1.0; p->mma.a = 0.0; p->mma.c = 1e4; p->mma.d = 0.0;
    p->mma.xmin = 0.01; p->mma.xmax = 1.0; p->mma.raa0 = 1e-5; p->mma.albefa = 0.1; p->mma.move = 0.2;
    p->mma.asyinit = 0.5; p->mma.asydecr = 0.7; p->mma.asyincr = 1.2; p->mma.epsvalue = 1e-6; p->mma.max_newton = 500;
    p->oc.beta = 0.0;
    p->heaviside = 0; p->beta0 = 0.5; p->beta_factor = 2.0; p->beta_every = 40; p->iter_offset = 0;
}

int pf_simp_run(pf_ctx* ctx, const pf_simp_params* prm, int iters, double* s, double* rho_out, pf_simp_history* hist) {
    if (!ctx || !prm || !s) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, false));
    PF_CHECK(iters >= 0, PF_ERR_ARG, "iters must be non-negative");
    for (long e = 0; e < ctx->ne; e++)
        PF_CHECK(std::isfinite(s[e]), PF_ERR_NUMERIC, "pf_simp_run: non-finite design variable");
    PF_CHECK(!prm->learned || (ctx->net && ctx->net->trained), PF_ERR_STATE,
             "learned solves need a trained preconditioner (pf_precond_init, collect, train)");
    PF_CHECK(prm->collect <= 0 || ctx->net, PF_ERR_STATE, "collecting pairs needs pf_precond_init first");
    PF_TRY(set_device(ctx));
    ctx->E1 = prm->E1; ctx->E0 = prm->E0; ctx->p = prm->p; ctx->nu = prm->nu; ctx->t = prm->t;
    if (!ctx->have_filter || ctx->R != prm->R) PF_TRY(pf_filter_setup(ctx, prm->R));
    const long ne = ctx->ne;
    const size_t eb = sizeof(double) * ne;
    double *d_s = ctx->d_e0, *d_dfdrho = ctx->d_e1, *d_dfds = ctx->d_e2, *d_dgds = ctx->d_e3, *d_xplus = ctx->d_e4;
    double* d_tmp = ctx->d_e5;
    double* d_dr = ctx->d_e6;
    const bool hv = prm->heaviside != 0;
    PF_CHECK(!hv || (prm->beta0 > 0 && prm->beta_factor > 0 && prm->beta_every > 0), PF_ERR_ARG,
             "Heaviside continuation needs beta0, beta_factor and beta_every > 0");
    PF_HIP(hipMemcpyAsync(d_s, s, eb, hipMemcpyHostToDevice, ctx->stream));
    // dgdrho is the constant scale1/(vf ne) (sample...oc.cpp:103); with the
    // density filter its filtered form is fixed
    const double dgdrho = prm->scale1 / (prm->vf * (double)ne);
    if (!hv) {
        k_fill<double><<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, d_tmp, dgdrho);
        PF_TRY(filter_device(ctx, d_tmp, d_dgds));
    }
    pf_oc_params oc = prm->oc;
    oc.vf = prm->vf;
    oc.scale1 = prm->scale1;
    oc.beta = 0.0;
    double beta = 0.0;
    PF_CHECK(prm->use_mma >= 0 && prm->use_mma <= 2, PF_ERR_ARG, "use_mma: 0 OC, 1 MMA, 2 CONLIN");
    if (prm->use_mma && !(prm->resume_optimizer && ctx->mma && ctx->mma->n == ctx->ne &&
                          ctx->mma->conlin == (prm->use_mma == 2)))
        PF_TRY(mma_init_device(ctx, &prm->mma, prm->use_mma == 2));
    double prev_f = 0.0;
    // a solve that stops at itrmax, an OC bisection that ends at its cap or
    // at an end of its bracket: the loop goes on with the valid last result
    // (as the reference does) and the call returns PF_NOT_CONVERGED with the
    // first such message; an MMA/CONLIN interior-point loop that reaches
    // max_newton ends the loop there
    int warn = PF_OK;
    std::string warn_msg;
    bool stop = false;
    int it = 0;
    for (; it < iters && !stop; it++) {
        auto t0 = std::chrono::steady_clock::now();
        const unsigned ge = gsize(ne);
        if (hv) {
            // beta continuation (sample_optimize_density_oc.cpp:89-93): beta0
            // multiplied by beta_factor at every beta_every-th iteration from 0
            const int K = prm->iter_offset + it;
            beta = prm->beta0;
            for (int q = 0; q <= K / prm->beta_every; q++) beta *= prm->beta_factor;
            oc.beta = beta;
            // rho = H(filter(s)), dr = H'(filter(s)) (HeavisideFilter.h:62-99)
            PF_TRY(filter_device(ctx, d_s, d_tmp));
            k_heaviside<<<ge, kBlock, 0, ctx->stream>>>(ne, d_tmp, beta, ctx->d_rho, d_dr);
        } else {
            // rho = filter(s)
            PF_TRY(filter_device(ctx, d_s, ctx->d_rho));
        }
        // g = volume(rho)
        k_volume_partials<<<ge, kBlock, 0, ctx->stream>>>(ne, ctx->d_rho, prm->vf, prm->scale1, ctx->red.partials);
        int rc;
        double g = reduce_host(ctx, ctx->red.partials, (int)ge, 1.0, 1.0 * prm->scale1, &rc);
        PF_TRY(rc);
        PF_TRY(moduli_from_rho(ctx));
        // solve K u = F
        pf_solve_stats st{};
        int op = prm->learned ? PF_OP_LEARNED : (prm->mixed ? PF_OP_EBE32 : prm->solver);
        if (op == PF_OP_CSR64) PF_TRY(pf_assemble_csr(ctx, nullptr));
        if (prm->collect > 0 && op == PF_OP_EBE64) {
            PcgRun run;
            int cnt;
            PF_TRY(net_collect(ctx, ctx->d_load, prm->collect, prm->collect_max > 0 ? prm->collect_max : 16, &cnt,
                               &run));
            st.iterations = run.iterations;
            st.status = run.status;
            st.true_residual = run.bnorm > 0 ? run.rnorm / run.bnorm : 0.0;
        } else {
            int src = solve_nodal(ctx, op, ctx->d_load, ctx->d_x, prm->cg_eps, prm->cg_itrmax, prm->inner_eps, &st);
            if (src < 0) return src;
            if (src != PF_OK && warn == PF_OK) {
                warn = PF_NOT_CONVERGED;
                warn_msg = "iteration " + std::to_string(prm->iter_offset + it) +
                           ": the solve stopped before eps (itrmax reached)";
            }
        }
        // compliance, sensitivities, filtered sensitivities
        double f;
        PF_TRY(comp_sens_device(ctx, ctx->d_x, prm->scale0, d_dfdrho, &f));
        if (hv) {
            // sum_j dfdrho_j dr_j w_ij / sum_j w_ij, and the same for dgdrho
            k_mul_d<<<ge, kBlock, 0, ctx->stream>>>(ne, d_dfdrho, d_dr, d_tmp);
            PF_TRY(filter_device(ctx, d_tmp, d_dfds));
            k_cmul_d<<<ge, kBlock, 0, ctx->stream>>>(ne, dgdrho, d_dr, d_tmp);
            PF_TRY(filter_device(ctx, d_tmp, d_dgds));
        } else {
            PF_TRY(filter_device(ctx, d_dfdrho, d_dfds));
        }
        // IsConvergence of OC (OC.h:67-73, eps 1e-5) / MMA (MMA.h:107-113, epsvalue)
        const double ceps = prm->use_mma ? prm->mma.epsvalue : 1.0e-5;
        bool conv = std::fabs(f - prev_f) / (f + prev_f) < ceps;
        double lam = 0.0;
        int steps = 0;
        if (!(prm->stop_on_convergence && conv)) {
            if (prm->use_mma) {
                int mrc = mma_update_device(ctx, d_s, f, d_dfds, g, d_dgds, &steps);
                if (mrc < 0) return mrc;
                if (mrc != PF_OK) {
                    if (warn == PF_OK) {
                        warn = PF_NOT_CONVERGED;
                        warn_msg = "iteration " + std::to_string(prm->iter_offset + it) + ": " + ctx->err +
                                   " (loop stopped, design left at this iteration's input)";
                    }
                    stop = true;
                }
            } else {
                int orc = oc_device(ctx, &oc, d_s, d_dfds, d_dgds, d_xplus, &lam, &steps);
                if (orc < 0) return orc;
                if (orc != PF_OK && warn == PF_OK) {
                    warn = PF_NOT_CONVERGED;
                    warn_msg = "iteration " + std::to_string(prm->iter_offset + it) + ": " + ctx->err;
                }
                PF_HIP(hipMemcpyAsync(d_s, d_xplus, eb, hipMemcpyDeviceToDevice, ctx->stream));
            }
        }
        PF_TRY(sync(ctx));
        double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        if (hist) {
            if (hist->f) hist->f[it] = f;
            if (hist->g) hist->g[it] = g;
            if (hist->lambda) hist->lambda[it] = lam;
            if (hist->cg_iters) hist->cg_iters[it] = st.iterations;
            if (hist->bisect) hist->bisect[it] = steps;
            if (hist->seconds) hist->seconds[it] = secs;
            if (hist->residual) hist->residual[it] = st.true_residual;
            if (hist->fallbacks) hist->fallbacks[it] = st.fallbacks;
        }
        prev_f = f;
        if (prm->stop_on_convergence && conv) {
            it++;
            break;
        }
    }
    if (hist) hist->iterations = it;
    PF_HIP(hipMemcpyAsync(s, d_s, eb, hipMemcpyDeviceToHost, ctx->stream));
    if (rho_out) {
        PF_TRY(filter_device(ctx, d_s, hv ? d_tmp : ctx->d_rho));
        if (hv) k_heaviside<<<gsize(ne), kBlock, 0, ctx->stream>>>(ne, d_tmp, beta, ctx->d_rho, nullptr);
        PF_HIP(hipMemcpyAsync(rho_out, ctx->d_rho, eb, hipMemcpyDeviceToHost, ctx->stream));
    }
    PF_TRY(sync(ctx));
    if (warn != PF_OK) ctx->err = warn_msg;
    return warn;
}

int pf_heaviside(pf_ctx* ctx, double beta, int mode, const double* s, const double* dfdrho, double* out) {
    if (!ctx || !s || !out || (mode == 1 && !dfdrho)) return PF_ERR_ARG;
    PF_CHECK(mode == 0 || mode == 1, PF_ERR_ARG, "pf_heaviside: mode 0 (variables) or 1 (sensitivities)");
    PF_CHECK(beta > 0 && std::isfinite(beta), PF_ERR_ARG, "pf_heaviside: beta must be positive");
    PF_CHECK(ctx->dim > 0, PF_ERR_STATE, "no grid");
    PF_TRY(set_device(ctx));
    const long ne = ctx->ne;
    const size_t eb = sizeof(double) * ne;
    const unsigned ge = gsize(ne);
    PF_HIP(hipMemcpyAsync(ctx->d_e0, s, eb, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(filter_device(ctx, ctx->d_e0, ctx->d_e1));  // s~
    if (mode == 0) {
        k_heaviside<<<ge, kBlock, 0, ctx->stream>>>(ne, ctx->d_e1, beta, ctx->d_e2, nullptr);
    } else {
        k_heaviside<<<ge, kBlock, 0, ctx->stream>>>(ne, ctx->d_e1, beta, ctx->d_e3, ctx->d_e6);
        PF_HIP(hipMemcpyAsync(ctx->d_e4, dfdrho, eb, hipMemcpyHostToDevice, ctx->stream));
        k_mul_d<<<ge, kBlock, 0, ctx->stream>>>(ne, ctx->d_e4, ctx->d_e6, ctx->d_e5);
        PF_TRY(filter_device(ctx, ctx->d_e5, ctx->d_e2));
    }
    PF_TRY(check_launch(ctx));
    PF_HIP(hipMemcpyAsync(out, ctx->d_e2, eb, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_profile_kernels(pf_ctx* ctx, int op, int reps, double* ms) {
    if (!ctx || !ms || reps < 1) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_CHECK(op == PF_OP_EBE64 || op == PF_OP_EBE32, PF_ERR_ARG, "pf_profile_kernels: EbE operators only");
    PF_CHECK(is2d(ctx), PF_ERR_UNSUPPORTED, "pf_profile_kernels: quad4 grids only in this build");
    PF_TRY(set_device(ctx));
    const bool f32 = op == PF_OP_EBE32;
    PcgDev* S = (PcgDev*)ctx->d_pcg;
    double* partA = ctx->red.partials;
    double* partB = ctx->red.partials + 2 * kMaxPartials;
    const K1Shape sh = k1_shape(ctx->nx, ctx->ny);
    const unsigned g1 = sh.grid;
    const unsigned g2 = std::min<unsigned>(gsize(ctx->nv), (unsigned)k2_cap());
    PF_CHECK(g1 <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
    // a defined state: b = load, x = 0, z = b/D, p = 0; launches use k = 0 (no
    // convergence test) so every repetition does the full work
    PF_TRY(diag_nodal(ctx, f32));
    if (f32) {
        k_convert<double, float><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->d_load, ctx->f_b);
        k_pcg_init<float><<<g2, kBlock, 0, ctx->stream>>>(ctx->nv, ctx->f_b, ctx->f_D, ctx->f_x, ctx->f_r, ctx->f_z,
                                                         ctx->f_p0, partB, S);
    } else {
        k_pcg_init<double><<<g2, kBlock, 0, ctx->stream>>>(ctx->nv, ctx->d_load, ctx->d_D, ctx->d_x, ctx->d_r,
                                                          ctx->d_z, ctx->d_p0, partB, S);
    }
    PF_TRY(check_launch(ctx));
    hipEvent_t e0, e1;
    PF_HIP(hipEventCreate(&e0));
    PF_HIP(hipEventCreate(&e1));
    auto timed = [&](auto&& launch) -> double {
        launch();  // warm
        hipEventRecord(e0, ctx->stream);
        for (int i = 0; i < reps; i++) launch();
        hipEventRecord(e1, ctx->stream);
        hipEventSynchronize(e1);
        float t = 0.f;
        hipEventElapsedTime(&t, e0, e1);
        return (double)t / reps;
    };
    if (f32) {
        ms[0] = timed([&] {
            k_pcg_k1_q4_tile<float, kTileI, kTileJ><<<g1, kBlock, 0, ctx->stream>>>(
                ctx->nx, ctx->ny, sh.tilesJ, sh.ntiles, 0, ctx->f_p0, ctx->f_z, ctx->f_p1, ctx->f_q, ctx->d_Ef, ctx->d_K0f, ctx->d_fix,
                partB, (int)g2, partA, S, 0.0);
        });
        ms[1] = timed([&] {
            k_pcg_k2<float><<<g2, kBlock, 0, ctx->stream>>>(ctx->nv, 0, ctx->f_x, ctx->f_r, ctx->f_z, ctx->f_p1,
                                                          ctx->f_q, ctx->f_D, partA, (int)g1, partB, S);
        });
    } else {
        ms[0] = timed([&] {
            k_pcg_k1_q4_tile<double, kTileI, kTileJ><<<g1, kBlock, 0, ctx->stream>>>(
                ctx->nx, ctx->ny, sh.tilesJ, sh.ntiles, 0, ctx->d_p0, ctx->d_z, ctx->d_p1, ctx->d_q, ctx->d_E, ctx->d_K0, ctx->d_fix,
                partB, (int)g2, partA, S, 0.0);
        });
        ms[1] = timed([&] {
            k_pcg_k2<double><<<g2, kBlock, 0, ctx->stream>>>(ctx->nv, 0, ctx->d_x, ctx->d_r, ctx->d_z, ctx->d_p1,
                                                           ctx->d_q, ctx->d_D, partA, (int)g1, partB, S);
        });
    }
    ms[4] = 0.0;
    if (!f32) {
        // the single-reduction kernel: launch 0 from r = b, then launches 1
        // and 2 (no convergence test) repeated in turn
        unsigned gc;
        const Cg1Tiles G = cg1_tiles(ctx, &gc);
        PF_CHECK(gc <= (unsigned)kMaxPartials, PF_ERR_ARG, "grid too large for the reduction scratch");
        double* pc0 = ctx->red.partials;
        double* pc1 = ctx->red.partials + 3 * kMaxPartials;
        k_cg1_start<<<1, 1, 0, ctx->stream>>>(S);
        k_recip<double><<<gsize(ctx->nv), kBlock, 0, ctx->stream>>>(ctx->nv, ctx->d_D, ctx->d_Dinv);
        Cg1Vecs<double> V0{ctx->d_load, ctx->d_p1, ctx->d_s1, ctx->d_r, ctx->d_p1, ctx->d_s0, ctx->d_p0, ctx->d_x,
                           ctx->d_Dinv};
        k_cg1_q4_tile<double, kCg1TI, kCg1TJ, true><<<gc, kBlock, 0, ctx->stream>>>(
            ctx->nx, ctx->ny, G, 0, V0, ctx->d_E, ctx->d_K0, ctx->d_fix, pc1, (int)gc, pc0, S, 0.0);
        Cg1Vecs<double> V1{ctx->d_r, ctx->d_p1, ctx->d_s0, ctx->d_z, ctx->d_q, ctx->d_s1, ctx->d_p0, ctx->d_x,
                           ctx->d_Dinv};
        Cg1Vecs<double> V2{ctx->d_z, ctx->d_q, ctx->d_s1, ctx->d_r, ctx->d_p1, ctx->d_s0, ctx->d_p0, ctx->d_x,
                           ctx->d_Dinv};
        // an odd launch (x untouched) and an even one (x updated): the mean of the pair
        ms[4] = 0.5 * timed([&] {
            k_cg1_q4_tile<double, kCg1TI, kCg1TJ, false><<<gc, kBlock, 0, ctx->stream>>>(
                ctx->nx, ctx->ny, G, 1, V1, ctx->d_E, ctx->d_K0, ctx->d_fix, pc0, (int)gc, pc1, S, 0.0);
            k_cg1_q4_tile<double, kCg1TI, kCg1TJ, true><<<gc, kBlock, 0, ctx->stream>>>(
                ctx->nx, ctx->ny, G, 2, V2, ctx->d_E, ctx->d_K0, ctx->d_fix, pc1, (int)gc, pc0, S, 0.0);
        });
    }
    ms[2] = ms[3] = 0.0;
    if (ctx->have_filter) {
        ms[2] = timed([&] {
            k_filter_q4<<<gsize(ctx->ne), kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->win, ctx->R, ctx->d_cg,
                                                                   ctx->d_rho, ctx->d_e5);
        });
        OcDev init{};
        init.l0i = 0.0;
        init.l1i = 1e9;
        hipMemcpyAsync(ctx->d_oc, &init, sizeof(OcDev), hipMemcpyHostToDevice, ctx->stream);
        const unsigned ge = gsize(ctx->ne);
        k_fill<double><<<ge, kBlock, 0, ctx->stream>>>(ctx->ne, ctx->d_e1, -1.0);
        k_fill<double><<<ge, kBlock, 0, ctx->stream>>>(ctx->ne, ctx->d_e2, 1.0);
        // step 0 of a bisection (no decision to read), the one-launch form
        ms[3] = timed([&] {
            k_oc_step<<<ge, kBlock, 0, ctx->stream>>>(ctx->nx, ctx->ny, ctx->win, ctx->R, ctx->d_cg, 0, ctx->d_rho,
                                                     ctx->d_e1, ctx->d_e2, 0.5, 0.2, 1e-3, 0.5, 1.0, 0.0,
                                                     ctx->red.partials, (int)ge, ctx->d_e4, (OcDev*)ctx->d_oc);
        });
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    PF_TRY(check_launch(ctx));
    return sync(ctx);
}

int pf_precond_init(pf_ctx* ctx, int channels, uint64_t seed) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(channels == 0 || channels == 16, PF_ERR_ARG, "pf_precond_init: base width 16 (pass 0 or 16)");
    PF_TRY(require_ready(ctx, false));
    PF_TRY(set_device(ctx));
    return net_build(ctx, seed);
}

int pf_precond_num_params(pf_ctx* ctx, int64_t* count) {
    if (!ctx || !count) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    int64_t n = 0;
    for (NetLayer& l : ctx->net->L) n += l.size();
    *count = n;
    return PF_OK;
}

int pf_precond_save(pf_ctx* ctx, float* params, int64_t* count) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    int64_t off = 0;
    for (NetLayer& l : ctx->net->L) {
        if (params) PF_HIP(hipMemcpyAsync(params + off, l.W, sizeof(float) * l.size(), hipMemcpyDeviceToHost, ctx->stream));
        off += l.size();
    }
    if (count) *count = off;
    return sync(ctx);
}

int pf_precond_load(pf_ctx* ctx, const float* params, int64_t count) {
    if (!ctx || !params) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    int64_t n;
    PF_TRY(pf_precond_num_params(ctx, &n));
    PF_CHECK(n == count, PF_ERR_ARG, "pf_precond_load: parameter count mismatch");
    for (int64_t q = 0; q < count; q++) PF_CHECK(std::isfinite(params[q]), PF_ERR_NUMERIC, "non-finite parameter");
    PF_TRY(set_device(ctx));
    int64_t off = 0;
    for (NetLayer& l : ctx->net->L) {
        PF_HIP(hipMemcpyAsync(l.W, params + off, sizeof(float) * l.size(), hipMemcpyHostToDevice, ctx->stream));
        off += l.size();
    }
    PF_TRY(net_refresh_bf16(ctx, ctx->net));
    ctx->net->trained = true;
    return sync(ctx);
}

int pf_precond_collect(pf_ctx* ctx, int every, int max_pairs, int* count) {
    if (!ctx) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    return net_collect(ctx, ctx->d_load, every, max_pairs, count);
}

int pf_precond_collect_random(pf_ctx* ctx, int count, uint64_t seed, int* total) {
    if (!ctx || count < 0) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    PF_TRY(net_dataset_alloc(ctx));
    return net_collect_random(ctx, count, seed, total);
}

int pf_precond_train(pf_ctx* ctx, int steps, double lr, uint64_t seed, double* loss_first, double* loss_last) {
    if (!ctx) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_CHECK(ctx->net->nsamp > 0, PF_ERR_STATE, "no training pairs: call pf_precond_collect first");
    PF_CHECK(steps >= 0 && lr > 0, PF_ERR_ARG, "pf_precond_train: steps >= 0, lr > 0");
    PF_TRY(set_device(ctx));
    LearnedNet* N = ctx->net;
    // Each step loads its pair's densities into the context (moduli,
    // diagonal, multigrid hierarchy); the caller's densities and moduli are
    // kept aside and put back on every return path, and the assembled CSR
    // values are marked out of date while they are away.
    const long ne = ctx->ne;
    if (!N->keep_rho) {
        PF_TRY(net_alloc(ctx, N, &N->keep_rho, ne));
        PF_TRY(net_alloc(ctx, N, &N->keep_E, ne));
        PF_TRY(net_alloc(ctx, N, &N->keep_Ef, ne));
    }
    PF_HIP(hipMemcpyAsync(N->keep_rho, ctx->d_rho, sizeof(double) * ne, hipMemcpyDeviceToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(N->keep_E, ctx->d_E, sizeof(double) * ne, hipMemcpyDeviceToDevice, ctx->stream));
    PF_HIP(hipMemcpyAsync(N->keep_Ef, ctx->d_Ef, sizeof(float) * ne, hipMemcpyDeviceToDevice, ctx->stream));
    const long nnz_kept = ctx->nnz;
    const bool had_E = ctx->have_E;
    ctx->nnz = ctx->nnz >= 0 ? -2 : ctx->nnz;
    auto restore = [&]() -> int {
        PF_HIP(hipMemcpyAsync(ctx->d_rho, N->keep_rho, sizeof(double) * ne, hipMemcpyDeviceToDevice, ctx->stream));
        PF_HIP(hipMemcpyAsync(ctx->d_E, N->keep_E, sizeof(double) * ne, hipMemcpyDeviceToDevice, ctx->stream));
        PF_HIP(hipMemcpyAsync(ctx->d_Ef, N->keep_Ef, sizeof(float) * ne, hipMemcpyDeviceToDevice, ctx->stream));
        ctx->have_E = had_E;
        ctx->nnz = nnz_kept;
        if (had_E) PF_TRY(diag_nodal(ctx, false));
        return sync(ctx);
    };
    uint64_t rs = seed ? seed : 7ull;
    double first = 0, last = 0;
    int nf = 0, nl = 0, nfinite = 0;
    const int win = std::max(1, std::min(20, steps / 4));
    for (int it = 0; it < steps; it++) {
        int smp = (int)(splitmix(rs) % (uint64_t)N->nsamp);
        double loss;
        const int rc = net_train_step(ctx, smp, (float)lr, &loss);
        if (rc < 0) {
            const std::string msg = ctx->err;
            restore();
            ctx->err = msg;
            return rc;
        }
        if (!std::isfinite(loss)) continue;
        nfinite++;
        if (it < win) { first += loss; nf++; }
        if (it >= steps - win) { last += loss; nl++; }
    }
    PF_TRY(restore());
    if (loss_first) *loss_first = nf ? first / nf : NAN;
    if (loss_last) *loss_last = nl ? last / nl : NAN;
    if (steps > 0 && nfinite == 0) {
        ctx->err = "pf_precond_train: no step produced a finite loss (network left untrained)";
        return PF_ERR_NUMERIC;
    }
    N->trained = true;
    return PF_OK;
}

int pf_precond_apply(pf_ctx* ctx, const double* r_free, double* d_free) {
    if (!ctx || !r_free || !d_free) return PF_ERR_ARG;
    PF_TRY(require_ready(ctx, true));
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    PF_HIP(hipMemcpyAsync(ctx->d_t1, r_free, sizeof(double) * ctx->N, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(to_nodal(ctx, ctx->d_t1, ctx->d_r));
    PF_TRY(diag_nodal(ctx, false));
    PF_TRY(net_apply(ctx, ctx->d_rho, ctx->d_r, ctx->d_z, nullptr));
    PF_TRY(to_free(ctx, ctx->d_z, ctx->d_t0));
    PF_HIP(hipMemcpyAsync(d_free, ctx->d_t0, sizeof(double) * ctx->N, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

// x0 (FP32, rounded to BF16) into the network's input tensor
int net_load_input(pf_ctx* ctx, const float* x0) {
    LearnedNet* N = ctx->net;
    const long n = lvl_px(N, 0) * 16;
    std::vector<bf16> h(n);
    for (long q = 0; q < n; q++) h[q] = f2bf(x0[q]);
    PF_HIP(hipMemcpyAsync(N->x0, h.data(), sizeof(bf16) * n, hipMemcpyHostToDevice, ctx->stream));
    return sync(ctx);  // h is freed on return
}

int pf_precond_forward_raw(pf_ctx* ctx, const float* x0, float* y) {
    if (!ctx || !x0 || !y) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    LearnedNet* N = ctx->net;
    PF_TRY(net_load_input(ctx, x0));
    PF_TRY(net_forward(ctx, false));
    PF_HIP(hipMemcpyAsync(y, N->y, sizeof(float) * lvl_px(N, 0) * 16, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_precond_forward_nodal(pf_ctx* ctx, const float* x0, double* y_nodal) {
    if (!ctx || !x0 || !y_nodal) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    LearnedNet* N = ctx->net;
    PF_TRY(net_load_input(ctx, x0));
    PF_TRY(net_forward(ctx, true));
    PF_HIP(hipMemcpyAsync(y_nodal, N->w, sizeof(double) * ctx->nn * ctx->ndpn, hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int pf_conv_raw(pf_ctx* ctx, int mode, int cin, int cout, int H, int W, int Dp, const float* x, const float* w_or_dz,
                float* out) {
    if (!ctx || !x || !w_or_dz || !out) return PF_ERR_ARG;
    PF_CHECK(mode == 0 || mode == 1, PF_ERR_ARG, "pf_conv_raw: mode 0 (forward) or 1 (weight gradient)");
    PF_CHECK(H > 0 && W > 0 && Dp >= 0, PF_ERR_ARG, "pf_conv_raw: H, W > 0, Dp >= 0");
    PF_CHECK((cin == 16 || cin == 32 || cin == 64) && (cout == 16 || cout == 32 || cout == 64), PF_ERR_ARG,
             "pf_conv_raw: channel counts 16, 32 or 64");
    PF_TRY(set_device(ctx));
    const bool d3 = Dp > 0;
    const long npx = (long)H * W * (d3 ? Dp : 1);
    const long ntap = d3 ? 27 : 9;
    const long nw = ntap * cin * cout;
    const long nx_ = npx * cin, nz_ = npx * cout;
    std::vector<bf16> hx(nx_), hw(mode == 0 ? nw : nz_);
    for (long q = 0; q < nx_; q++) hx[q] = f2bf(x[q]);
    for (long q = 0; q < (long)hw.size(); q++) hw[q] = f2bf(w_or_dz[q]);
    bf16 *dx = nullptr, *dw = nullptr;
    float *dout = nullptr, *wpart = nullptr;
    const long nb = (npx + kWgradPixels - 1) / kWgradPixels;
    const long nout = mode == 0 ? nz_ : nw;
    int rc = PF_OK;
    auto fail = [&](hipError_t e, const char* what) {
        if (e != hipSuccess && rc == PF_OK) {
            ctx->err = std::string("pf_conv_raw: ") + what + ": " + hipGetErrorString(e);
            rc = PF_ERR_HIP;
        }
    };
    fail(hipMalloc((void**)&dx, sizeof(bf16) * nx_), "hipMalloc");
    fail(hipMalloc((void**)&dw, sizeof(bf16) * hw.size()), "hipMalloc");
    fail(hipMalloc((void**)&dout, sizeof(float) * nout), "hipMalloc");
    if (mode == 1) fail(hipMalloc((void**)&wpart, sizeof(float) * nb * nw), "hipMalloc");
    if (rc == PF_OK) {
        fail(hipMemcpyAsync(dx, hx.data(), sizeof(bf16) * nx_, hipMemcpyHostToDevice, ctx->stream), "copy");
        fail(hipMemcpyAsync(dw, hw.data(), sizeof(bf16) * hw.size(), hipMemcpyHostToDevice, ctx->stream), "copy");
    }
    if (rc == PF_OK) {
        if (mode == 0)
            rc = d3 ? conv3_fwd(ctx, cin, cout, H, W, Dp, dx, dw, nullptr, dout, 0)
                    : conv_fwd(ctx, cin, cout, H, W, dx, dw, nullptr, dout, 0);
        else
            rc = d3 ? conv3_wgrad(ctx, cin, cout, H, W, Dp, dx, dw, dout, wpart)
                    : conv_wgrad(ctx, cin, cout, H, W, dx, dw, dout, wpart);
    }
    if (rc == PF_OK) fail(hipMemcpyAsync(out, dout, sizeof(float) * nout, hipMemcpyDeviceToHost, ctx->stream), "copy");
    fail(hipStreamSynchronize(ctx->stream), "sync");
    hipFree(dx);
    hipFree(dw);
    hipFree(dout);
    if (wpart) hipFree(wpart);
    return rc;
}

int pf_precond_backward_raw(pf_ctx* ctx, const float* dy, float* grad) {
    if (!ctx || !dy || !grad) return PF_ERR_ARG;
    PF_CHECK(ctx->net, PF_ERR_STATE, "learned preconditioner not initialised");
    PF_TRY(set_device(ctx));
    LearnedNet* N = ctx->net;
    const long n = lvl_px(N, 0) * 16;
    std::vector<bf16> h(n);
    for (long q = 0; q < n; q++) h[q] = f2bf(dy[q]);
    PF_HIP(hipMemcpyAsync(N->gy, h.data(), sizeof(bf16) * n, hipMemcpyHostToDevice, ctx->stream));
    PF_TRY(net_backward(ctx));
    int64_t off = 0;
    for (NetLayer& l : N->L) {
        PF_HIP(hipMemcpyAsync(grad + off, l.g, sizeof(float) * l.size(), hipMemcpyDeviceToHost, ctx->stream));
        off += l.size();
    }
    return sync(ctx);
}

}  // extern "C"
