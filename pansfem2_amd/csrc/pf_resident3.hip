// Hex8 counterpart of pf_resident.hip: Jacobi-PCG in ScalingCG's order with
// the solve resident on the chip, and the operator in the element matrix's
// parity basis.
//
// Operator.  A box element of a material that the three mirror planes of the
// box leave as it is (checked on the matrix itself, h8_parity_pack) has a
// stiffness matrix that is block diagonal after a Hadamard transform over the
// eight corners of each displacement component: sum_corner (-1)^(s.corner)
// u_c(corner), s in {0,1}^3.  A mirror along axis a multiplies the pair (s, c)
// by (-1)^(s_a + [a = c]), so pairs couple only within one of eight classes
// eps = s xor e_c of three pairs each: with symmetry and the translations
// (s = 0, which the matrix annihilates) left out, 39 numbers in scalar
// registers instead of 576, and about 190 FP64 operations per element instead
// of 576 multiply-adds.  The transform splits over the axes, so a thread that
// marches along i transforms each face once for the two elements that share it.
//
// Decomposition.  Workgroup (I, J, K) owns a box of elements (at most 16 along
// j and k) and holds r, p and q of all its nodes; nodes on a shared face are
// held by both sides.  After the operator the sums of the shared nodes are
// completed axis by axis: each side sends its sum and adds the other's, and as
// a + b = b + a every holder of a node has the same bits.  Each global node is
// counted and written by one holder.  p and q live in LDS, r and the diagonal in
// registers; x is read and written once an iteration, in the order of the
// workgroup's own values, through the L2 that holds it.  FP64 with 16 values per
// thread is the exception: beside the operator's four faces r, d and z do not
// fit, 64 of its vector registers (244 bytes a lane) go to scratch, and all
// variants keep about 200 scalars in lanes of vector registers.
//
// Measured per iteration (launched kernels before, resident now): 128x64x64
// FP64 68 us, 32 us; 100x50x50 56, 32; 100x40x40 49, 26; 80x40x40 49, 25;
// 60x30x30 FP64 35, 13, FP32 28, 10; 16x8x8 31, 8.  Of the 32 us at 128x64x64 (by
// the clock in workgroup 0) the operator takes 9.6 (its FP64 issue bounds it at
// 3.5; one or two waves a SIMD leave the rest to latency), the three face
// exchanges 9.5, p and p.Kp 1.8, the update of r and x and the new z 4.5, the two
// sums' waits 5.8; of the 13.5 us at 60x30x30 3.2, 4.8, 0.6, 1.5 and 3.0.
#pragma once

namespace pf {

constexpr int kH8ParityCoefs = 39;

// Members of class eps: pairs (s, c) with s = eps xor (4 >> c); f(c, s) for
// those with s != 0.
__host__ __device__ constexpr int h8_parity_s(int eps, int c) { return eps ^ (4 >> c); }

// K0's blocks in the order in which the kernel reads them: per class the upper
// triangle of its members' block.  False when K0 is not symmetric, couples
// different classes or translations by more than rounding (64 eps of its
// largest entry): the general operator then applies it.
inline bool h8_parity_pack(const double* K0, double* out) {
    double Kc[24][24], H[8][8], T[24][24];
    double big = 0.0;
    for (int a = 0; a < 8; a++)
        for (int s = 0; s < 8; s++) H[s][a] = (__builtin_popcount(s & a) & 1) ? -1.0 : 1.0;
    // corners 4 di + 2 dj + dk
    auto ref = [](int a) {
        const int di = a >> 2, dj = (a >> 1) & 1, dk = a & 1;
        return 4 * dk + (dj == 0 ? di : 3 - di);
    };
    for (int a = 0; a < 8; a++)
        for (int b = 0; b < 8; b++)
            for (int c = 0; c < 3; c++)
                for (int d = 0; d < 3; d++) {
                    Kc[3 * a + c][3 * b + d] = K0[(3 * ref(a) + c) * 24 + 3 * ref(b) + d];
                    big = std::max(big, std::fabs(Kc[3 * a + c][3 * b + d]));
                }
    // T = (H x I) Kc (H x I)^T / 64
    for (int s = 0; s < 8; s++)
        for (int u = 0; u < 8; u++)
            for (int c = 0; c < 3; c++)
                for (int d = 0; d < 3; d++) {
                    double v = 0.0;
                    for (int a = 0; a < 8; a++)
                        for (int b = 0; b < 8; b++) v += H[s][a] * H[u][b] * Kc[3 * a + c][3 * b + d];
                    T[3 * s + c][3 * u + d] = v / 64.0;
                }
    const double tol = 64.0 * 2.220446049250313e-16 * big;
    if (!(big > 0.0) || !std::isfinite(big)) return false;
    for (int s = 0; s < 8; s++)
        for (int u = 0; u < 8; u++)
            for (int c = 0; c < 3; c++)
                for (int d = 0; d < 3; d++) {
                    const double v = T[3 * s + c][3 * u + d];
                    if (!(std::fabs(v - T[3 * u + d][3 * s + c]) <= tol)) return false;
                    const bool same = (s ^ (4 >> c)) == (u ^ (4 >> d));
                    if ((!same || s == 0 || u == 0) && !(std::fabs(v) <= tol)) return false;
                }
    int pos = 0;
    for (int eps = 0; eps < 8; eps++)
        for (int c = 0; c < 3; c++)
            for (int d = c; d < 3; d++) {
                const int s = h8_parity_s(eps, c), u = h8_parity_s(eps, d);
                if (s == 0 || u == 0) continue;
                out[pos++] = 0.5 * (T[3 * s + c][3 * u + d] + T[3 * u + d][3 * s + c]);
            }
    return pos == kH8ParityCoefs;
}

// The four values of a face's corners (index 2 dj + dk) to their sums and
// differences (index 2 s_j + s_k); its own inverse but for a factor 4, which
// the packed blocks carry.
template <class T>
__device__ inline void h8_face_transform(T (&v)[4]) {
    const T a0 = v[0] + v[1], a1 = v[0] - v[1], b0 = v[2] + v[3], b1 = v[2] - v[3];
    v[0] = a0 + b0;
    v[1] = a1 + b1;
    v[2] = a0 - b0;
    v[3] = a1 - b1;
}

// One element: the transformed faces lo (i) and up (i + 1) to their transformed
// results times E, lower added to clo, upper in cup.  kp: the packed blocks.
// One class at a time, each pinned by an empty asm: 24 inputs and 24 results
// at once, beside the four faces, would not fit the registers.
template <class T>
__device__ inline void h8_parity_element(const T (&kp)[kH8ParityCoefs], T E, const T (&lo)[3][4], const T (&up)[3][4], T (&clo)[3][4],
                                         T (&cup)[3][4]) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int f = 0; f < 4; f++) cup[c][f] = 0;
    int pos = 0;
#pragma unroll
    for (int eps = 0; eps < 8; eps++) {
        T u[3], o[3] = {0, 0, 0};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int s = h8_parity_s(eps, c), f = s & 3;
            u[c] = E * (s >> 2 ? lo[c][f] - up[c][f] : lo[c][f] + up[c][f]);
        }
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int d = c; d < 3; d++) {
                if (h8_parity_s(eps, c) == 0 || h8_parity_s(eps, d) == 0) continue;
                const T k = kp[pos++];
                o[c] += k * u[d];
                if (d != c) o[d] += k * u[c];
            }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int s = h8_parity_s(eps, c), f = s & 3;
            if (s == 0) continue;
            clo[c][f] += o[c];
            cup[c][f] = s >> 2 ? cup[c][f] - o[c] : cup[c][f] + o[c];
            asm volatile("" : "+v"(clo[c][f]), "+v"(cup[c][f]));
        }
    }
}

// the value of the next lower lane of the row of 16 (0 for lane 0 of a row)
__device__ inline double res_row_up(double v) {
    const u64 b = (u64)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x111, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x111, 0xf, 0xf, true);
    return res_join(lo, hi);
}
__device__ inline float res_row_up(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));
}

// The two words of a double in one 16-byte store (each word is read by itself).
// A store of more than 8 bytes must be two wait states ahead of the next write
// of its data registers; the compiler does not see the store in the asm, so the
// s_nop is in it too.
__device__ inline void res_put2(u64* p, unsigned tag, double v) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 w = {res_half(v, 0), tag, res_half(v, 1), tag};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(w) : "memory");
}

constexpr int kRes3Threads = 512;
constexpr int kRes3Slots = 16;   // node values per thread, at most
constexpr int kRes3Items = 4;    // values of two opposite faces per thread, at most

template <class T>
struct Res3Args {
    int nx, ny, nz, gi, gj, gk;
    int m0, m1, last;
    unsigned tag;
    int box, fb[3];          // exchange words per workgroup and buffer, first word per axis
    const T *b, *D, *E, *Kp;
    T *x, *r, *p;            // r, p: state between launches
    T* loc;                  // x of every workgroup's values: [workgroups][threads x slots]
    const uint8_t* fix;
    u64 *slots, *edge;       // edge: [2][workgroups][box]
    PcgDev* S;
    ResDev* R;
    double eps;
};

// face values (both sides, three components) of a box of di x dj x dk nodes, per axis
__host__ __device__ inline int res3_face(int ax, int di, int dj, int dk) {
    return 3 * (ax == 0 ? dj * dk : ax == 1 ? di * dk : di * dj);
}

// Thread t of half-workgroup t / 256 marches over its half of the box's element
// layers: element column (j, k) = (4 wave + lane / 16, lane % 16).
template <class T, int SL>
__global__ void __launch_bounds__(kRes3Threads) k_pcg_h8_resident(Res3Args<T> A) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    extern __shared__ __align__(16) unsigned char res_lds_raw[];
    __shared__ ResLds L;
    constexpr int NT = kRes3Threads, NW = (int)sizeof(T) / 4;
    typedef const __attribute__((address_space(4))) T* KPtr;
    const int t = threadIdx.x, wg = blockIdx.x;
    const int K = wg % A.gk, J = wg / A.gk % A.gj, I = wg / (A.gk * A.gj);
    const int e0i = (int)((long)I * A.nx / A.gi), ei = (int)((long)(I + 1) * A.nx / A.gi) - e0i;
    const int e0j = (int)((long)J * A.ny / A.gj), ej = (int)((long)(J + 1) * A.ny / A.gj) - e0j;
    const int e0k = (int)((long)K * A.nz / A.gk), ek = (int)((long)(K + 1) * A.nz / A.gk) - e0k;
    const int dj = ej + 1, dk = ek + 1, di = ei + 1;
    const int PL = dj * dk, NN = di * PL, NV = 3 * NN;
    T* sp = (T*)res_lds_raw;  // p: [component][node]
    T* sq = sp + NT * SL;     // q likewise

    if (t == 0) L.bad = 0;
    if (A.R->stall) return;  // S->done is not tested: see k_pcg_q4_resident

    // this thread's node values v = t + NT s (component-major); own: counted
    // and written here, fixm: fixed.  Values beyond NV are zeros that take part
    // in everything.
    auto gindex = [&](int v, bool& mine) {
        const int c = v / NN, ln = v - c * NN;
        const int a = ln / PL, b = (ln - a * PL) / dk, k = ln - a * PL - b * dk;
        mine = (a > 0 || I == 0) && (b > 0 || J == 0) && (k > 0 || K == 0);
        return 3 * (((A.ny + 1) * (e0i + a) + e0j + b) * (A.nz + 1) + e0k + k) + c;
    };
    T* locx = A.loc + (size_t)wg * NT * SL + t;
    unsigned own = 0, fixm = 0;
    T r[SL], d[SL];
#pragma unroll
    for (int s = 0; s < SL; s++) {
        const int v = t + NT * s;
        T pv = 0;
        r[s] = 0;
        d[s] = 1;
        if (v < NV) {
            bool mine;
            const int x = gindex(v, mine);
            if (mine) own |= 1u << s;
            if ((A.fix[x / 3] >> (x % 3)) & 1) fixm |= 1u << s;
            r[s] = (A.m0 ? A.r : A.b)[x];
            d[s] = A.D[x];
            if (A.m0) pv = A.p[x];
        }
        sp[v] = pv;
        sq[v] = 0;
        if (!A.m0) locx[NT * s] = 0;
    }
    // per-value tests are made where they are used: hoisted out of the loop
    // their masks would take the scalar registers of the element's blocks
    auto bit = [](unsigned& m, int s) {
        asm volatile("" : "+v"(m));
        return ((m >> s) & 1) != 0;
    };
    // element column and moduli
    const int g = __builtin_amdgcn_readfirstlane(t >> 8), cj = ((t >> 6) & 3) * 4 + ((t & 63) >> 4), ck = t & 15;
    const bool act = cj < ej && ck < ek;
    const int hl = (ei + 1) / 2;                       // layers of the first half
    const int a0 = g ? hl : 0, nl = g ? ei - hl : hl;  // first plane, layers
    const T* Ecol = A.E + ((long)A.ny * (e0i + a0) + e0j + (act ? cj : 0)) * A.nz + e0k + (act ? ck : 0);
    const long Estep = (long)A.ny * A.nz;

    // faces: axis ax, item h = side F + (the rest): LDS position, -1: no neighbour there
    int fq[3][kRes3Items];
    const int gdim[3] = {A.gi, A.gj, A.gk}, at[3] = {I, J, K}, step[3] = {A.gj * A.gk, A.gk, 1};
    {
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const int F = res3_face(ax, di, dj, dk);  // the same on both sides of a face
#pragma unroll
            for (int m = 0; m < kRes3Items; m++) {
                const int h = t + NT * m, side = h >= F;
                fq[ax][m] = -1;
                if (h >= 2 * F || (side ? at[ax] == gdim[ax] - 1 : at[ax] == 0)) continue;
                const int f = h - side * F, c = f / (F / 3), q = f - c * (F / 3);
                int a, b, k;
                if (ax == 0) { a = side ? ei : 0; b = q / dk; k = q - b * dk; }
                else if (ax == 1) { a = q / dk; b = side ? ej : 0; k = q - a * dk; }
                else { a = q / dj; b = q - a * dj; k = side ? ek : 0; }
                fq[ax][m] = c * NN + a * PL + b * dk + k;
            }
        }
    }
    __syncthreads();

    // sq = this box's part of K p
    auto apply = [&]() {
        T lo[3][4], up[3][4], acc[3][4], nxt[3][4];
#pragma unroll
        for (int c = 0; c < 3; c++) {
#pragma unroll
            for (int f = 0; f < 4; f++) acc[c][f] = 0;
            const T* q = sp + c * NN + a0 * PL + (act ? cj * dk + ck : 0);
            lo[c][0] = q[0];
            lo[c][1] = q[1];
            lo[c][2] = q[dk];
            lo[c][3] = q[dk + 1];
            h8_face_transform(lo[c]);
        }
        for (int st = 0; st <= hl; st++) {
            if (st == hl) __syncthreads();  // the shared plane's first sums are complete
            const int a = a0 + st;
            const bool layer = st < nl, plane = nl > 0 && st <= nl;
            int col = act ? cj * dk + ck : 0;
            asm volatile("" : "+v"(col));  // addresses formed here, not kept
            if (layer) {
                // the blocks' scalar loads, in flight with the face's reads;
                // all of them arrive before the element's classes (loaded
                // where they are used, each class would wait for its own) and
                // are dropped after it (kept, they push the rest of the loop's
                // scalars into vector lanes)
                unsigned long long ka = (unsigned long long)A.Kp;
                asm volatile("" : "+s"(ka));
                T kp[kH8ParityCoefs];
#pragma unroll
                for (int e = 0; e < kH8ParityCoefs; e++) kp[e] = ((KPtr)ka)[e];
                const T E = act ? Ecol[Estep * st] : (T)0;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const T* q = sp + c * NN + (a + 1) * PL + col;
                    up[c][0] = q[0];
                    up[c][1] = q[1];
                    up[c][2] = q[dk];
                    up[c][3] = q[dk + 1];
                    h8_face_transform(up[c]);
                }
#pragma unroll
                for (int e = 0; e < kH8ParityCoefs; e++) asm volatile("" : "+s"(kp[e]));
                h8_parity_element<T>(kp, E, lo, up, acc, nxt);
            } else {
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int f = 0; f < 4; f++) nxt[c][f] = 0;
            }
            T nd[2][3], nl1[2][3];  // node ck and (last lane) node ek of rows cj, cj + 1
#pragma unroll
            for (int c = 0; c < 3; c++) {
                h8_face_transform(acc[c]);  // corners 2 dj + dk
                nd[0][c] = acc[c][0] + res_row_up(acc[c][1]);
                nd[1][c] = acc[c][2] + res_row_up(acc[c][3]);
                nl1[0][c] = acc[c][1];
                nl1[1][c] = acc[c][3];
            }
            // row cj, then (after the barrier) row cj + 1 added; the last row
            // has no first writer; the first half adds to the plane that both
            // halves share
            const bool add = !g && st == hl && ei > hl;
            if (act && plane) {
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    T* q = sq + c * NN + a * PL + col;
                    q[0] = add ? q[0] + nd[0][c] : nd[0][c];
                    if (ck == ek - 1) q[1] = add ? q[1] + nl1[0][c] : nl1[0][c];
                }
            }
            __syncthreads();
            if (act && plane) {
                const bool add2 = add || cj < ej - 1;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    T* q = sq + c * NN + a * PL + dk + col;
                    q[0] = add2 ? q[0] + nd[1][c] : nd[1][c];
                    if (ck == ek - 1) q[1] = add2 ? q[1] + nl1[1][c] : nl1[1][c];
                }
            }
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    lo[c][f] = up[c][f];
                    acc[c][f] = nxt[c][f];
                }
        }
        __syncthreads();
    };
    // the sums of the shared nodes completed along one axis
    auto exchange = [&](int ax, const int (&q)[kRes3Items], unsigned tag, int par) {
        // addresses are formed here each time: kept across the iteration, those
        // of three axes take 50 registers
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int F = res3_face(ax, di, dj, dk);
        u64* out = A.edge + ((size_t)par * gridDim.x + wg) * A.box + A.fb[ax];
#pragma unroll
        for (int m = 0; m < kRes3Items; m++)
            if (q[m] >= 0) {
                const T v = sq[q[m]];
                u64* o = out + (t + NT * m) * NW;
                if constexpr (NW == 2) {
                    res_put2(o, tag, v);
                } else {
                    res_put(o, tag, __float_as_uint(v));
                }
            }
        __builtin_amdgcn_s_sleep(8);
        unsigned w[kRes3Items * NW];
        long long t0 = 0;
        for (int n = 0;; n++) {
            u64 in[kRes3Items * NW];
            bool ok = true;
#pragma unroll
            for (int m = 0; m < kRes3Items; m++)
                if (q[m] >= 0) {
                    const int h = t + NT * m, side = h >= F;
                    const u64* src = A.edge + ((size_t)par * gridDim.x + wg + (side ? step[ax] : -step[ax])) * A.box +
                                     A.fb[ax] + (side ? h - F : h + F) * NW;
#pragma unroll
                    for (int e = 0; e < NW; e++) in[m * NW + e] = res_get(src + e);
                }
#pragma unroll
            for (int m = 0; m < kRes3Items; m++)
#pragma unroll
                for (int e = 0; e < NW; e++) {
                    w[m * NW + e] = (unsigned)in[m * NW + e];
                    ok = ok && (q[m] < 0 || (unsigned)(in[m * NW + e] >> 32) == tag);
                }
            if (ok) break;
            if ((n & 63) == 63) {
                const long long c = wall_clock64();
                if (!t0) t0 = c;
                if (c - t0 > kResWaitTicks) {
                    L.bad = 1;
                    break;
                }
            }
        }
#pragma unroll
        for (int m = 0; m < kRes3Items; m++)
            if (q[m] >= 0) {
                T v;
                if constexpr (NW == 2) v = (T)res_join(w[2 * m], w[2 * m + 1]);
                else v = (T)__uint_as_float(w[m]);
                sq[q[m]] += v;
            }
        __syncthreads();
    };
    const bool w0 = t == 0 && wg == 0;
    auto finish = [&](double rnorm, int iterations, int status) {
        for (int s = 0; s < SL; s++) {
            const int v = t + NT * s;
            bool mine = false;
            const int x = v < NV ? gindex(v, mine) : 0;
            if (mine) A.x[x] = locx[NT * s];
        }
        if (w0) {
            A.S->rnorm = rnorm;
            A.S->iterations = iterations;
            A.S->status = status;
            A.S->done = 1;
        }
    };

    unsigned tag = A.tag;
    double zrprev = A.R->v[0], rr = A.R->v[1], zr = A.R->g, bnorm = A.R->bnorm;
    auto near_stop = [&](double q) { return q < (A.eps * bnorm) * (A.eps * bnorm) * 1.0001 || q < 1e-290; };
    T z[SL];
    // z = r ./ D (CG.h:412) and the sums z.r, r.r of the counted nodes
    auto scale = [&](double (&v2)[2]) {
        v2[0] = v2[1] = 0.0;
#pragma unroll
        for (int s = 0; s < SL; s++) {
            z[s] = r[s] / d[s];
            const double w = bit(own, s) ? (double)r[s] : 0.0;
            v2[0] += (double)z[s] * w;
            v2[1] += (double)r[s] * w;
        }
    };
    double v2[2];
    scale(v2);
    if (A.m0 == 0) {
        res_publish<2, NT>(v2, L, A.slots, tag);
        res_pause<false>();
        if (!res_collect<2, NT>(v2, L, A.slots, tag)) {
            if (t == 0) A.R->stall = 1;
            return;
        }
        tag++;
        zr = v2[0];
        rr = v2[1];
        bnorm = sqrt(rr);
        if (w0) A.S->bnorm = bnorm;
    }
    for (int k = A.m0; k < A.m1; k++) {
        double beta = 0.0;
        if (k > 0) {  // pcg_head_sums
            if (near_stop(rr)) {
                const double rnorm = sqrt(rr);
                if (rnorm < A.eps * bnorm) {
                    finish(rnorm, k, 1);
                    return;
                }
            }
            beta = wave_uniform(zr / zrprev);
        }
        const T tb = (T)beta;
#pragma unroll
        for (int s = 0; s < SL; s++)
            sp[t + NT * s] = tb * sp[t + NT * s] + z[s];  // xeaxpy (CG.h:42-49)
        __syncthreads();
        apply();
        double acc[1] = {0.0};  // p.Kp from the boxes' parts
#pragma unroll
        for (int s = 0; s < SL; s++)
            acc[0] += (double)sp[t + NT * s] * (double)sq[t + NT * s];
        res_publish<1, NT>(acc, L, A.slots, tag);
        if (A.gi > 1) exchange(0, fq[0], tag, k & 1);
        if (A.gj > 1) exchange(1, fq[1], tag, k & 1);
        if (A.gk > 1) exchange(2, fq[2], tag, k & 1);
        if (!res_collect<1, NT>(acc, L, A.slots, tag)) {
            if (t == 0) A.R->stall = 1;
            return;
        }
        tag++;
        const double alpha = wave_uniform(zr / acc[0]);  // CG.h:433
        const T ta = (T)alpha, tma = (T)(-alpha);
#pragma unroll
        for (int s = 0; s < SL; s++)
            r[s] = r[s] + tma * (bit(fixm, s) ? (T)0 : sq[t + NT * s]);
        scale(v2);
        res_publish<2, NT>(v2, L, A.slots, tag);
        {  // while the sums travel
            T x[SL];
#pragma unroll
            for (int s = 0; s < SL; s++) x[s] = locx[NT * s];
#pragma unroll
            for (int s = 0; s < SL; s++) locx[NT * s] = x[s] + ta * sp[t + NT * s];
        }
        if (!res_collect<2, NT>(v2, L, A.slots, tag)) {
            if (t == 0) A.R->stall = 1;
            return;
        }
        tag++;
        zrprev = zr;
        zr = v2[0];
        rr = v2[1];
    }
    if (A.last) {  // k_pcg_final
        const double rnorm = sqrt(rr);
        finish(rnorm, A.m1, (A.m1 > 0 && rnorm < A.eps * bnorm) ? 1 : 2);
        return;
    }
    // the state of the next launch
#pragma unroll
    for (int s = 0; s < SL; s++)
        if (t + NT * s < NV) {
            bool mine;
            const int x = gindex(t + NT * s, mine);
            if (mine) {
                A.r[x] = r[s];
                A.p[x] = sp[t + NT * s];
            }
        }
    if (w0) {
        A.R->v[0] = zrprev;
        A.R->v[1] = rr;
        A.R->g = zr;
        A.R->bnorm = bnorm;
    }
}

// ------------------------------------------------------ OC bisection -----
// Sums of the density filter's normalised weights over the filtered elements:
// with winv null out_j = 1 / sum_e w_je, else out_j = sum_e w_ej winv_e.
__global__ void __launch_bounds__(256) k_filter_colsum(G3 g, int dim, int win, double R, const double* __restrict__ cg,
                                                       const double* __restrict__ winv, double* __restrict__ out) {
    const int nz = dim == 3 ? g.nz : 1;
    const long ne = (long)g.nx * g.ny * nz;
    const BlockRange xr = xcd_block_range(ne);
    for (long e = xr.begin + threadIdx.x; e < xr.end; e += blockDim.x) {
        const int i = (int)(e / ((long)g.ny * nz)), r = (int)(e - (long)i * g.ny * nz), j = r / nz, k = r - j * nz;
        double s = 0.0;
        for (int ii = max(i - win, 0); ii <= min(i + win, g.nx - 1); ii++)
            for (int jj = max(j - win, 0); jj <= min(j + win, g.ny - 1); jj++)
                for (int kk = max(k - win, 0); kk <= min(k + win, nz - 1); kk++) {
                    const long m = ((long)ii * g.ny + jj) * nz + kk;
                    double q = 0.0;
                    for (int d = 0; d < dim; d++) {
                        const double v = cg[dim * e + d] - cg[dim * m + d];
                        q += v * v;
                    }
                    const double dist = sqrt(q);
                    if (dist <= R) s += (R - dist) / R * (winv ? winv[m] : 1.0);
                }
        out[e] = winv ? s : 1.0 / s;
    }
}

// The whole bisection of an OC update with the density filter (no projection) in
// one cooperative launch: x, the derivatives and the filter's column sums of S
// elements per thread stay in registers (of sixteen, 170 go to scratch).  The
// filter is linear, so the filtered volume is the column sums' product with x+,
// the same sum in another order, and a step is S candidates and one exchanged
// sum, whose latency bounds it on small grids.  The launched form filters x+ in
// every step.  A launch takes 72 us at 120x40 (2.3 per step; launched 8.6) and
// 102 at 128x64x64 (launched 36 per step); a whole update with host vectors,
// launched and resident: 120x40 0.38, 0.20 ms; 1024x512 (four per thread) 1.31,
// 0.78; 1024x1000 (eight) 2.46, 1.50; 2048x1024 (sixteen) 5.32, 3.69.
struct OcRes {
    long n;
    int max_steps;
    unsigned tag;
    double iota, move, leps, vf, scale1, l0, l1;
    const double *x, *dfdx, *dgdx, *col;
    double* xplus;
    u64* slots;
    ResDev* R;
    OcDev* O;  // lambda_last, steps, done, status
};
constexpr int kOcResThreads = 512;

template <int S>
__global__ void __launch_bounds__(kOcResThreads) k_oc_resident(OcRes A) {
    __shared__ ResLds lds;
    constexpr int NT = kOcResThreads;
    if (threadIdx.x == 0) lds.bad = 0;
    __syncthreads();
    auto index = [&](int s) { return ((long)blockIdx.x * S + s) * NT + threadIdx.x; };
    double x[S], df[S], dg[S], col[S], xp[S];
    const double den = A.vf * (double)A.n;
#pragma unroll
    for (int s = 0; s < S; s++) {
        const long j = index(s);
        const bool on = j < A.n;
        x[s] = on ? A.x[j] : 0.0;
        df[s] = on ? A.dfdx[j] : -1.0;
        dg[s] = on ? A.dgdx[j] : 1.0;
        col[s] = on ? A.col[j] : 0.0;
        xp[s] = 0.0;  // xkp1 starts as zeros (OC.h:81)
    }
    double l0 = A.l0, l1 = A.l1, lambda = 0.0;
    unsigned tag = A.tag;
    int k = 0, steps = 0, done = 0, status = 0;
    for (;; k++) {
        if (!((l1 - l0) / (l1 + l0) > A.leps)) {
            steps = k;
            done = 1;
            status = (k > 0 && l1 == A.l1) ? 1 : (k > 0 && l0 == A.l0 && l0 > 0.0) ? 2 : 0;
            break;
        }
        lambda = 0.5 * (l1 + l0);
        steps = k + 1;
        double v[1] = {0.0};
#pragma unroll
        for (int s = 0; s < S; s++) {
            xp[s] = oc_candidate(x[s], df[s], dg[s], lambda, A.iota, A.move);
            if (index(s) < A.n) v[0] += A.scale1 * (col[s] * xp[s]) / den;
        }
        if (k == A.max_steps) break;  // the cap: the last decision's candidate
        res_publish<1, NT>(v, lds, A.slots, tag);
        res_pause<false>();
        if (!res_collect<1, NT>(v, lds, A.slots, tag)) {
            if (threadIdx.x == 0) A.R->stall = 1;
            return;
        }
        tag++;
        if (v[0] - 1.0 * A.scale1 > 0.0) l0 = lambda;
        else l1 = lambda;
    }
#pragma unroll
    for (int s = 0; s < S; s++)
        if (index(s) < A.n) A.xplus[index(s)] = xp[s];
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        A.O->lambda_last = lambda;
        A.O->steps = steps;
        A.O->done = done;
        A.O->status = status;
    }
}

}  // namespace pf
