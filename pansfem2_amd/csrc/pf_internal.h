// Internal declarations shared by the HIP translation units of libpansfem2_amd.
//
// Data layout in HBM (structured grids only):
//   * nodes are numbered as SquareMesh does (src/PrePost/Mesher/SquareMesh.h:60-70):
//     2D node (i,j) -> (ny+1)*i + j, element (i,j) -> ny*i + j;
//     3D node (i,j,k) -> ((ny+1)*(nz+1))*i + (nz+1)*j + k, element -> ny*nz*i + nz*j + k.
//   * every solver vector is "nodal": ndpn consecutive values per node, fixed DOFs
//     held at zero, so the EbE operator and all vector kernels index without
//     indirection.  Free-DOF (reference-numbered) vectors exist only at the
//     boundary and are converted with g2n / n2g.
//   * per-node fixity is one byte, bit d set when DOF d is fixed.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/pansfem2_amd.h"

namespace pf {

constexpr int kBlock = 256;        // threads per workgroup for the 1D kernels
constexpr int kMaxPartials = 8192;  // upper bound on workgroups of a reducing launch

// Device-resident scalars of a PCG solve (defined with the kernels that
// write them, pf_kernels.hip) and of the OC bisection.
struct PcgDev;
struct OcDev;
struct ResDev;

// Reduction scratch: per-workgroup partials and the arrival counter of the
// "last workgroup reduces" pattern.  One set per context; launches that reduce
// are serialised on the context's stream.
struct ReduceScratch {
    double* partials;    // kMaxPartials * 8 doubles, then the resident solves' slots and scalars
    unsigned* counter;   // one counter, returned to zero by the last workgroup
    double* out;         // 16 doubles of results
};

}  // namespace pf

struct pf_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;

    // grid
    int dim = 0;
    int nx = 0, ny = 0, nz = 0;
    long nn = 0, ne = 0;
    int ndpn = 0, nd = 0;
    double lx = 0, ly = 0, lz = 0;

    // DOF map
    int N = 0;
    std::vector<int32_t> h_n2g;
    int32_t* d_n2g = nullptr;   // nn*ndpn, -1 for fixed
    int32_t* d_g2n = nullptr;   // N, nodal index of each free DOF
    uint8_t* d_fix = nullptr;   // nn, fixity bits

    // shared unit element matrix (E = 1)
    std::vector<double> h_K0;
    double* d_K0 = nullptr;
    float* d_K0f = nullptr;
    double* d_K0g = nullptr;  // hex8: K0 packed in the operator kernel's order (h8_pack_k0)
    float* d_K0gf = nullptr;
    double* d_K0m = nullptr;  // hex8: K0 as the MFMA operator's A fragments (h8m_pack_k0)
    float* d_K0mf = nullptr;
    double* d_K0p = nullptr;  // hex8: K0's parity blocks (h8_parity_pack), behind d_K0m; null when it has none
    float* d_K0pf = nullptr;

    // material / design
    double E1 = 1.0, E0 = 1e-9, p = 3.0, nu = 0.3, t = 1.0;
    double* d_rho = nullptr;
    double* d_E = nullptr;
    float* d_Ef = nullptr;
    bool have_E = false;

    // nodal work vectors (nv = nn*ndpn)
    long nv = 0;
    double *d_x = nullptr, *d_r = nullptr, *d_z = nullptr, *d_q = nullptr, *d_p0 = nullptr, *d_p1 = nullptr;
    double *d_D = nullptr, *d_b = nullptr, *d_t0 = nullptr, *d_t1 = nullptr;
    float *f_x = nullptr, *f_r = nullptr, *f_z = nullptr, *f_q = nullptr, *f_p0 = nullptr, *f_p1 = nullptr;
    int pcg_form = 0;  // PF_PCG_SCALINGCG or PF_PCG_SINGLE_REDUCTION (quad4 matrix-free solves)
    // second buffers of the single-reduction solver's s = K p
    double *d_s0 = nullptr, *d_s1 = nullptr;
    float *f_s0 = nullptr, *f_s1 = nullptr;
    double* d_Dinv = nullptr;  // 1 / D of the single-reduction solves
    float *f_D = nullptr, *f_b = nullptr;

    // element work vectors (ne)
    double *d_e0 = nullptr, *d_e1 = nullptr, *d_e2 = nullptr, *d_e3 = nullptr, *d_e4 = nullptr, *d_e5 = nullptr;
    double* d_e6 = nullptr;     // projection derivative of the Heaviside filter
    double* d_cg = nullptr;     // element centroids (ne*dim)

    // point loads (nodal)
    double* d_load = nullptr;

    // assembled CSR (free-DOF numbering)
    long nnz = -1;
    int32_t *d_indptr = nullptr, *d_indices = nullptr;
    double* d_data = nullptr;
    double* d_ke_all = nullptr;  // ne*nd*nd element matrices in reference arithmetic

    // filter: the grid rule (pf_filter_setup) or caller-given neighbour
    // lists (pf_filter_set_lists, CSR-like ptr/idx/w over elements)
    double R = 0.0;
    int win = 0;
    bool have_filter = false;
    bool have_lists = false;
    double* d_fcol = nullptr;  // column sums of the grid rule's normalised weights, formed when an OC update needs them
    bool have_fcol = false;
    long fcol_n = 0;           // its size
    int32_t *d_fptr = nullptr, *d_fidx = nullptr;
    double* d_fw = nullptr;

    // device scalars
    pf::PcgDev* d_pcg = nullptr;
    pf::OcDev* d_oc = nullptr;
    pf::ReduceScratch red{};
    pf::PcgDev* h_pcg = nullptr;  // pinned mirror
    pf::OcDev* h_oc = nullptr;    // pinned mirror
    double* h_red = nullptr;          // pinned mirror of red.out

    // resident solves (pf_resident.hip): exchange buffers and scalars between
    // launches (slots, d_res and h_res are parts of red.partials and h_red),
    // the next unused exchange tag and the workgroups that run at once (0: none)
    unsigned long long *res_slots = nullptr, *res_halo = nullptr;
    double* res_loc = nullptr;              // hex8: the workgroups' own x
    long res_halo_n = 0, res_loc_n = 0;     // their sizes
    pf::ResDev *d_res = nullptr, *h_res = nullptr;
    unsigned res_tag = 1;
    int res_wgs = 0;
    // calls still to be launched after a stall or a refused launch, and the last
    // stall's number of them (res_gave_up, res_launch)
    int res_pause = 0, res_backoff = 0;
    int res_mode = PF_RESIDENT_AUTO, res_after = 0;  // pf_set_resident
    int64_t res_done = 0, res_gave = 0;              // pf_resident_runs

    // MMA state
    struct MmaState* mma = nullptr;
    // learned preconditioner
    struct LearnedNet* net = nullptr;

    // multigrid base preconditioner of the flexible CG (pf_mg_setup) and the
    // prolongation its next setup takes (pf_mg_set_prolongation)
    struct MgState* mg = nullptr;
    int mg_prolong = PF_MG_PROLONG_STIFFNESS;
    int mg_resid = PF_MG_RESIDUAL_AUTO;  // hex8 coarse-level residual form
    int h8_op = PF_H8_OP_AUTO;  // hex8 matrix-free operator of the Jacobi-PCG (pf_set_h8_operator)

    // device address of the library's static scratch array on this
    // context's device (pf_compliance_sens_dev_noalloc)
    double* noalloc_scratch = nullptr;
};

// ---------------------------------------------------------------- errors ----
#define PF_HIP(call)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess) {                                                               \
            ctx->err = std::string(#call) + ": " + hipGetErrorString(e_);                     \
            return PF_ERR_HIP;                                                                \
        }                                                                                     \
    } while (0)

#define PF_CHECK(cond, code, msg)                                                             \
    do {                                                                                      \
        if (!(cond)) {                                                                        \
            ctx->err = (msg);                                                                 \
            return (code);                                                                    \
        }                                                                                     \
    } while (0)

#define PF_TRY(call)                                                                          \
    do {                                                                                      \
        int rc_ = (call);                                                                     \
        if (rc_ < 0) return rc_;                                                              \
    } while (0)

namespace pf {
inline unsigned nblocks(long n, int bs = kBlock) { return (unsigned)((n + bs - 1) / bs); }
}  // namespace pf
