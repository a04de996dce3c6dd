// Jacobi-PCG on quad4 grids with the whole solve resident on the chip.
//
// One workgroup per CU (at most 256, launched cooperatively, so all of them
// run at once) owns a tile of nodes for the whole solve: r, p, x, the Jacobi
// diagonal and the carried products stay in registers, the operator's input
// (with a one-node halo) and the moduli in LDS.  Per iteration a workgroup
// exchanges with the others only the operator's result on its tile's edge and
// its partial sums, so no vector passes through memory: at 1024x512 the
// launched kernels move 80-105 MB per iteration, this one about 1 MB.
//
// Exchange: every 32-bit half of a value is stored as one 8-byte word beside
// a 32-bit tag that grows with every exchange; a reader polls a word until it
// carries the tag it waits for.  Each word is a relaxed agent-scope atomic, so
// value and tag arrive together and no fence or separate barrier is needed: an
// exchange costs one store and one load through memory.  A workgroup stores
// the next exchange's words only after it has read all of the previous one's,
// so two buffers in turn are enough.  Every wait is bounded by the wall clock
// (kResWaitTicks): a workgroup that waits too long sets `stall` and ends, the
// others follow, and the host solves the system with the launched kernels.
//
// Every workgroup adds all partial sums in one order, so all of them take the
// same decisions and the result does not depend on timing.
//
// Measured per iteration (launched kernels before, resident now): single-
// reduction form 1024x512 18.4, 5.9 us, 601x333 10.9, 4.0, 301x149 8.8, 3.3,
// 120x40 8.5, 2.9; ScalingCG's order 1024x512 26.5, 7.4, 601x333 16.0, 5.4,
// 301x149 11.8, 4.5, 120x40 11.4, 4.0.  About 2.5 us (single-reduction) or 3.5
// us of it are the exchanges, whose latency bounds the small grids; at 1024x512
// the rest is the operator's FP64 issue and LDS reads on every CU.
#pragma once

namespace pf {

typedef unsigned long long u64;

constexpr int kResMaxWg = 256;               // slots of the partial sums
constexpr long long kResWaitTicks = 200000000;  // 2 s of the 100 MHz clock

// scalars of a resident solve between two launches of it
struct ResDev {
    double v[3];        // the last exchange's sums
    double g, a;        // single-reduction: gamma and alpha before; ScalingCG: z.r, -
    double bnorm;
    int stall, pad;
};

template <class T>
struct ResArgs {
    int nx, ny, gi, gj;   // element counts, tiles along i and j
    int m0, m1, last;     // iterations of this launch, last: m1 is the iteration limit
    unsigned tag;         // tag of this launch's first exchange
    const T *b, *D, *E, *K0;  // D: the diagonal (ScalingCG's order) or its inverse
    T *x, *r, *s, *p, *w;     // state between launches (s, w: single-reduction form)
    const uint8_t* fix;
    u64 *slots, *halo;    // partial sums [2][4][kResMaxWg][2]; edge values [2][nn][words of a node]
    PcgDev* S;
    ResDev* R;
    double eps;
};

__device__ inline void res_put(u64* p, unsigned tag, unsigned v) {
    __hip_atomic_store(p, ((u64)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline u64 res_get(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// G groups of NW consecutive words, `stride` words apart, polled until all
// carry `tag`; false after kResWaitTicks
template <int NW, int G = 1, int STRIDE = 0>
__device__ inline bool res_wait(const u64* p, unsigned tag, unsigned (&v)[NW * G]) {
    long long t0 = 0;
    for (int n = 0;; n++) {
        u64 q[NW * G];
#pragma unroll
        for (int k = 0; k < NW * G; k++) q[k] = res_get(p + k / NW * STRIDE + k % NW);
        bool ok = true;
#pragma unroll
        for (int k = 0; k < NW * G; k++) {
            ok = ok && (unsigned)(q[k] >> 32) == tag;
            v[k] = (unsigned)q[k];
        }
        if (ok) return true;
        if ((n & 63) == 63) {
            const long long t = wall_clock64();
            if (!t0) t0 = t;
            if (t - t0 > kResWaitTicks) return false;
        }
    }
}
__device__ inline double res_join(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((u64)hi << 32) | lo));
}
__device__ inline unsigned res_half(double v, int h) {
    const u64 b = (u64)__double_as_longlong(v);
    return h ? (unsigned)(b >> 32) : (unsigned)b;
}

// One node's pair as tagged words and back.
__device__ inline void res_put_pair(u64* p, unsigned tag, Vec2<double> v) {
    res_put(p, tag, res_half(v.x, 0));
    res_put(p + 1, tag, res_half(v.x, 1));
    res_put(p + 2, tag, res_half(v.y, 0));
    res_put(p + 3, tag, res_half(v.y, 1));
}
__device__ inline void res_put_pair(u64* p, unsigned tag, Vec2<float> v) {
    res_put(p, tag, __float_as_uint(v.x));
    res_put(p + 1, tag, __float_as_uint(v.y));
}
__device__ inline bool res_wait_pair(const u64* p, unsigned tag, Vec2<double>& v) {
    unsigned q[4];
    const bool ok = res_wait<4>(p, tag, q);
    v.x = res_join(q[0], q[1]);
    v.y = res_join(q[2], q[3]);
    return ok;
}
__device__ inline bool res_wait_pair(const u64* p, unsigned tag, Vec2<float>& v) {
    unsigned q[2];
    const bool ok = res_wait<2>(p, tag, q);
    v.x = __uint_as_float(q[0]);
    v.y = __uint_as_float(q[1]);
    return ok;
}

// Wavefront sum, complete in lane 63 only: row shifts and row broadcasts (DPP)
// instead of a butterfly through the LDS crossbar, a fixed order of additions.
// MAX: the maximum of non-negative values instead.
template <bool MAX>
__device__ inline double res_op(double a, double b) {
    if constexpr (MAX) return (a < b) ? b : a;
    else return a + b;
}
template <bool MAX, int CTRL, int ROWS>
__device__ inline double res_dpp_op(double v) {
    const u64 b = (u64)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xf, false);
    return res_op<MAX>(v, res_join(lo, hi));
}
template <bool MAX = false>
__device__ inline double res_wave_sum(double v) {
    v = res_dpp_op<MAX, 0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of a row has its sum
    v = res_dpp_op<MAX, 0x112, 0xf>(v);
    v = res_dpp_op<MAX, 0x114, 0xf>(v);
    v = res_dpp_op<MAX, 0x118, 0xf>(v);
    v = res_dpp_op<MAX, 0x142, 0xa>(v);  // lane 15 of rows 0, 2 to rows 1, 3
    v = res_dpp_op<MAX, 0x143, 0xc>(v);  // lane 31 to rows 2, 3
    return v;
}

struct ResLds {
    double part[4 * 16];  // this workgroup's sums per wave
    double sum[4 * 4];    // all workgroups' sums per group of 64 slots
    int bad;
};

// the two words of sum k of workgroup wg: one sum's words of consecutive
// workgroups are contiguous, so that a wave polls whole lines
__device__ inline u64* res_slot(u64* slots, unsigned tag, int k, int wg) {
    return slots + (((tag & 1) * 4 + k) * kResMaxWg + wg) * 2;
}
__device__ inline const u64* res_slot(const u64* slots, unsigned tag, int k, int wg) {
    return res_slot(const_cast<u64*>(slots), tag, k, wg);
}
// Between an exchange's stores and its first poll: polls of words that are
// still on their way delay the stores.  1024x512, 256 workgroups, ScalingCG's
// order: 11.0 us per iteration without the pause, 8.5 with half, 7.6 with
// this one, 7.8 with 1.5 times it; single-reduction form 6.4, 6.1, 6.1, 6.1.
// Few workgroups poll little: 120x40, 32 of them, ScalingCG's order 4.2, 4.1,
// 4.2, 4.6; single-reduction (which has the update of x here) 3.0, 3.1, 3.4, 3.6
// (64 of them without a pause 3.0, 80 of them 3.6).
template <bool SR>
__device__ inline void res_pause() {
    if (gridDim.x > 64) __builtin_amdgcn_s_sleep(16);
    else if (!SR && gridDim.x > 1) __builtin_amdgcn_s_sleep(8);
}

// This workgroup's sums of v, published under `tag` by K*2 threads.  The
// barrier inside also ends the phase that filled v.
template <int K, int NT, bool MAX = false>
__device__ inline void res_publish(double (&v)[K], ResLds& L, u64* slots, unsigned tag) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = res_wave_sum<MAX>(v[k]);
    if (lane == 63) {
#pragma unroll
        for (int k = 0; k < K; k++) L.part[k * 16 + w] = v[k];
    }
    __syncthreads();
    if (t < 2 * K) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NT / 64; i++) s = res_op<MAX>(s, L.part[(t >> 1) * 16 + i]);
        res_put(res_slot(slots, tag, t >> 1, blockIdx.x) + (t & 1), tag, res_half(s, t & 1));
    }
}
// All workgroups' sums into v (the same bits in every thread); false: stalled.
// Threads [NT / 2, NT / 2 + 256) (NT = 256: all) each read one workgroup's slot.
template <int K, int NT, bool MAX = false>
__device__ inline bool res_collect(double (&v)[K], ResLds& L, const u64* slots, unsigned tag) {
    if (gridDim.x == 1) {  // nobody to wait for
#pragma unroll
        for (int k = 0; k < K; k++) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < NT / 64; i++) s = res_op<MAX>(s, L.part[k * 16 + i]);
            v[k] = wave_uniform(s);
        }
        __syncthreads();
        return true;
    }
    constexpr int base = NT >= 512 ? 256 : 0;
    const int t = (int)threadIdx.x - base, lane = threadIdx.x & 63;
    if (t >= 0 && t < kResMaxWg) {
        double s[K];
#pragma unroll
        for (int k = 0; k < K; k++) s[k] = 0.0;
        if (t < (int)gridDim.x) {
            unsigned q[2 * K];
            if (!res_wait<2, K, 2 * kResMaxWg>(res_slot(slots, tag, 0, t), tag, q)) L.bad = 1;
#pragma unroll
            for (int k = 0; k < K; k++) s[k] = res_join(q[2 * k], q[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < K; k++) s[k] = res_wave_sum<MAX>(s[k]);
        if (lane == 63) {
#pragma unroll
            for (int k = 0; k < K; k++) L.sum[k * 4 + (t >> 6)] = s[k];
        }
    }
    __syncthreads();
    if (L.bad) return false;
#pragma unroll
    for (int k = 0; k < K; k++)
        v[k] = wave_uniform(res_op<MAX>(
            res_op<MAX>(res_op<MAX>(L.sum[k * 4], L.sum[k * 4 + 1]), L.sum[k * 4 + 2]), L.sum[k * 4 + 3]));
    return true;
}

// LDS of a tile of at most ti x tj nodes, S rows per thread: the operator's
// input with its halo, x and the diagonal of every thread's nodes, three values
// of every halo node, then the moduli.
template <class T>
constexpr size_t res_lds_bytes(int ti, int tj, int S, int nt) {
    const int rows = (ti + S - 1) / S * S;
    return sizeof(T) * (2 * (size_t)(rows + 2) * (tj + 2) + 4 * (size_t)S * nt + 12 * (size_t)(ti + tj + 2) +
                        (size_t)(rows + 1) * (tj + 1));
}

// Thread t owns column t mod tj and the S node rows from S (t / tj) on of its
// workgroup's tile (ti x tj nodes, tile sizes differ by at most one), and one
// halo node (t < 2 (tj + 2) + 2 ti).  SR: the single-reduction recurrences of
// k_cg1_q4_tile, one exchange per iteration; else ScalingCG's order, two.
template <class T, int S, int NT, bool SR>
__global__ void __launch_bounds__(NT) k_pcg_q4_resident(ResArgs<T> A) {
#pragma clang fp contract(fast)  // not a check-path kernel: FMA allowed
    extern __shared__ __align__(16) unsigned char res_lds_raw[];
    __shared__ ResLds L;
    constexpr int NWD = (int)sizeof(T) / 2;  // tagged words of a node
    const int t = threadIdx.x;
    const int I = blockIdx.x / A.gj, J = blockIdx.x - I * A.gj;
    const int nx = A.nx, ny = A.ny;
    const int i0 = (int)((long)I * (nx + 1) / A.gi), i1 = (int)((long)(I + 1) * (nx + 1) / A.gi);
    const int j0 = (int)((long)J * (ny + 1) / A.gj), j1 = (int)((long)(J + 1) * (ny + 1) / A.gj);
    const int ti = i1 - i0, tj = j1 - j0, ss = tj + 2, es = tj + 1;
    const int rows = (ti + S - 1) / S * S;
    Vec2<T>* su = (Vec2<T>*)res_lds_raw;      // (rows + 2) x ss, node (i0 - 1 + a, j0 - 1 + b)
    // x and the diagonal, read or written once an iteration, leave the registers
    // to the operator's window
    Vec2<T>* sx = su + (rows + 2) * ss + t;
    Vec2<T>* sd = sx + S * NT;
    const int nh = 2 * (tj + 2) + 2 * ti;
    Vec2<T>* sh = sd + S * NT;                // halo node t: r, s (ScalingCG's order: p), A.D at 0, nh, 2 nh
    T* se = (T*)(sh - t + 3 * nh);            // (rows + 1) x es, element (i0 - 1 + a, j0 - 1 + b)
    const unsigned nn = (unsigned)(nx + 1) * (ny + 1);

    if (t == 0) L.bad = 0;
    // a workgroup that starts after another has given up; S->done is no reason
    // to leave (the host launches no more once it is set): workgroup 0 sets it
    // without an exchange when a launch finds its first iterate converged, and
    // the workgroups that start later have their part of x still to write
    if (A.R->stall) return;
    for (int h = t; h < (rows + 2) * ss; h += NT) su[h] = Vec2<T>{0, 0};
    for (int h = t; h < (rows + 1) * es; h += NT) {
        const int a = h / es, ei = i0 - 1 + a, ej = j0 - 1 + (h - a * es);
        se[h] = (a <= ti && ei >= 0 && ei < nx && ej >= 0 && ej < ny) ? A.E[(long)ny * ei + ej] : (T)0;
    }

    // own nodes
    const int g = t / tj, c = t - g * tj;
    const int row0 = g * S < rows ? g * S : 0;  // LDS rows of idle threads: any valid ones
    // four bits per own node: 0, 1: DOF free; 2: another workgroup reads the
    // node; 3: the node exists
    unsigned fl = 0;
    static_assert(4 * S <= 32, "flags of the own nodes");
    Vec2<T> r[S], s[S], p[S], w[S];  // ScalingCG's order: s holds z, w holds q
    const int n0 = (ny + 1) * (i0 + row0) + j0 + c;
    auto flag = [&](int o, unsigned bit) { return (fl & (bit << (4 * o))) != 0; };
#pragma unroll
    for (int o = 0; o < S; o++) {
        const int a = row0 + o;
        r[o] = s[o] = p[o] = w[o] = Vec2<T>{0, 0};
        Vec2<T> x{0, 0}, d{1, 1};
        if (g * S < rows && a < ti) {
            const int n = n0 + (ny + 1) * o;
            const unsigned f = A.fix[n];
            fl |= (8u | (~f & 3u)) << (4 * o);
            if ((a == 0 && i0 > 0) || (a == ti - 1 && i1 <= nx) || (c == 0 && j0 > 0) || (c == tj - 1 && j1 <= ny))
                fl |= 4u << (4 * o);
            d = load2(A.D, n);
            r[o] = load2(A.m0 ? A.r : A.b, n);
            if (A.m0) {
                p[o] = load2(A.p, n);
                x = load2(A.x, n);
                if (SR) {
                    s[o] = load2(A.s, n);
                    w[o] = load2(A.w, n);
                }
            }
        }
        sx[o * NT] = x;
        sd[o * NT] = d;
    }
    // this thread's halo node: LDS position hq, node hn (hq < 0: none)
    int hq = -1;
    int hn = 0;
    {
        int a = -1, b = 0, h = t;
        bool in = true;
        if (h < tj + 2) { a = -1; b = h - 1; }
        else if ((h -= tj + 2) < tj + 2) { a = ti; b = h - 1; }
        else if ((h -= tj + 2) < ti) { a = h; b = -1; }
        else if ((h -= ti) < ti) { a = h; b = tj; }
        else in = false;
        const int ii = i0 + a, jj = j0 + b;
        if (in && ii >= 0 && ii <= nx && jj >= 0 && jj <= ny) {
            hq = (a + 1) * ss + b + 1;
            hn = (ny + 1) * ii + jj;
        }
    }
    Vec2<T> hw{0, 0};
    if (hq >= 0) {
        sh[0] = load2(A.m0 ? A.r : A.b, hn);
        sh[nh] = A.m0 ? load2(SR ? A.s : A.p, hn) : Vec2<T>{0, 0};
        sh[2 * nh] = load2(A.D, hn);
        if (SR && A.m0) hw = load2(A.w, hn);
    }
    __syncthreads();

    // w = K u at the own nodes from su and se (0 outside the grid), 0 at fixed
    // DOFs, dot += u.w; values that other workgroups read are published.  Columns c, c + 1
    // of the window serve the elements left of the node, c + 1, c + 2 those
    // right of it; each group of K0's rows is loaded once for the S nodes
    // (the pointer passes through an empty asm in every call, or the compiler
    // keeps all of K0 live across the loop and spills it).
    typedef const __attribute__((address_space(4))) T* KPtr;  // scalar loads: K0 does not change here
    auto apply = [&](unsigned tag, int par, double& dot) {
        const Vec2<T>* u0 = su + row0 * ss + c;
        const T* e0 = se + row0 * es + c;
        Vec2<T> vl[S + 2], vr[S + 2];
        T em[S + 1];
#pragma unroll
        for (int a = 0; a < S + 2; a++) vr[a] = u0[a * ss];
#pragma unroll
        for (int o = 0; o < S; o++) w[o] = Vec2<T>{0, 0};
#pragma unroll
        for (int side = 0; side < 2; side++) {
#pragma unroll
            for (int a = 0; a < S + 2; a++) {
                vl[a] = vr[a];
                vr[a] = u0[a * ss + side + 1];
            }
#pragma unroll
            for (int a = 0; a < S + 1; a++) em[a] = e0[a * es + side];
#pragma unroll
            for (int h = 0; h < 2; h++) {  // elements above (TR, BR) and below (TL, BL) the node
                const int loc = side ? (h ? 0 : 1) : (h ? 3 : 2);
                unsigned long long kp = (unsigned long long)A.K0;
                asm volatile("" : "+s"(kp));
#pragma unroll
                for (int o = 0; o < S; o++) {
                    T ex, ey;
                    elem_rows_q4<T>((KPtr)kp, loc, vl[o + h], vl[o + h + 1], vr[o + h + 1], vr[o + h], ex, ey);
                    w[o].x += em[o + h] * ex;
                    w[o].y += em[o + h] * ey;
                }
                // the sums are formed here and not next to their use behind the
                // branches below, where K0's rows would have to be kept
#pragma unroll
                for (int o = 0; o < S; o++) asm volatile("" : "+v"(w[o].x), "+v"(w[o].y));
            }
        }
#pragma unroll
        for (int o = 0; o < S; o++) {
            w[o].x = flag(o, 1u) ? w[o].x : (T)0;
            w[o].y = flag(o, 2u) ? w[o].y : (T)0;
            dot += (double)vl[o + 1].x * (double)w[o].x;
            dot += (double)vl[o + 1].y * (double)w[o].y;
            if (flag(o, 4u)) res_put_pair(A.halo + (par * nn + (unsigned)(n0 + (ny + 1) * o)) * NWD, tag, w[o]);
        }
    };
    const bool w0 = t == 0 && blockIdx.x == 0;
    auto store_x = [&]() {
#pragma unroll
        for (int o = 0; o < S; o++)
            if (flag(o, 8u)) store2(A.x, n0 + (ny + 1) * o, sx[o * NT]);
    };
    auto finish = [&](double rnorm, int iterations, int status) {
        store_x();
        if (w0) {
            A.S->rnorm = rnorm;
            A.S->iterations = iterations;
            A.S->status = status;
            A.S->done = 1;
        }
    };

    unsigned tag = A.tag;
    double v3[3] = {A.R->v[0], A.R->v[1], A.R->v[2]};
    double gprev = A.R->g, aprev = A.R->a, bnorm = A.R->bnorm;
    // whether sqrt(rr) < eps bnorm is possible at all: saves the root, a long
    // dependent chain, on the other iterations
    auto near_stop = [&](double rr) { return rr < (A.eps * bnorm) * (A.eps * bnorm) * 1.0001 || rr < 1e-290; };
    if constexpr (SR) {
        for (int m = A.m0; m < A.m1; m++, tag++) {
            double alpha = 0.0, beta = 0.0;
            if (m > 0) {  // cg1_head
                if (m == 1) {
                    const double rnorm = sqrt(v3[2]);
                    bnorm = rnorm;
                    alpha = v3[0] / v3[1];
                    if (w0) A.S->bnorm = rnorm;
                    if (!(v3[0] > 0.0)) {  // b = 0: x = 0 is the solution
                        finish(rnorm, 0, 1);
                        return;
                    }
                } else {
                    if (near_stop(v3[2])) {
                        const double rnorm = sqrt(v3[2]);
                        if (rnorm < A.eps * bnorm) {  // CG.h:445-449
                            finish(rnorm, m - 1, 1);
                            return;
                        }
                    }
                    beta = v3[0] / gprev;
                    alpha = v3[0] / (v3[1] - beta * v3[0] / aprev);
                }
                alpha = wave_uniform(alpha);
                beta = wave_uniform(beta);
                gprev = v3[0];
                aprev = alpha;
            }
            const T ta = (T)alpha, tb = (T)beta;
            double acc[3] = {0.0, 0.0, 0.0};  // r.u, u.w, r.r of iterate m
#pragma unroll
            for (int o = 0; o < S; o++) {
                // m = 0: alpha = beta = 0 and w = s = 0 leave r and x as they
                // are; p = u then takes no part in step 1, whose beta is 0
                const Vec2<T> d = sd[o * NT];
                p[o].x = r[o].x * d.x + tb * p[o].x;  // p = u + beta p
                p[o].y = r[o].y * d.y + tb * p[o].y;
                asm volatile("" : "+v"(p[o].x), "+v"(p[o].y));  // here, not later beside a second copy of r
                s[o].x = w[o].x + tb * s[o].x;  // s = w + beta s
                s[o].y = w[o].y + tb * s[o].y;
                r[o].x = r[o].x - ta * s[o].x;
                r[o].y = r[o].y - ta * s[o].y;
                const Vec2<T> u{r[o].x * d.x, r[o].y * d.y};  // Scaling (CG.h:412), by 1/D
                if (flag(o, 8u)) su[(row0 + o + 1) * ss + c + 1] = u;
                acc[0] += (double)r[o].x * (double)u.x;
                acc[0] += (double)r[o].y * (double)u.y;
                acc[2] += (double)r[o].x * (double)r[o].x;
                acc[2] += (double)r[o].y * (double)r[o].y;
            }
            if (hq >= 0) {
                Vec2<T> hr = sh[0], hs = sh[nh];
                const Vec2<T> hd = sh[2 * nh];
                hs.x = hw.x + tb * hs.x;
                hs.y = hw.y + tb * hs.y;
                hr.x = hr.x - ta * hs.x;
                hr.y = hr.y - ta * hs.y;
                su[hq] = Vec2<T>{hr.x * hd.x, hr.y * hd.y};
                sh[0] = hr;
                sh[nh] = hs;
            }
            __syncthreads();
            apply(tag, m & 1, acc[1]);
            res_publish<3, NT>(acc, L, A.slots, tag);
#pragma unroll
            for (int o = 0; o < S; o++) {  // while the sums travel (alpha = 0 at m = 0)
                Vec2<T> x = sx[o * NT];
                x.x = x.x + ta * p[o].x;
                x.y = x.y + ta * p[o].y;
                sx[o * NT] = x;
            }
            res_pause<SR>();
            if (hq >= 0 && !res_wait_pair(A.halo + ((m & 1) * nn + (unsigned)hn) * NWD, tag, hw)) L.bad = 1;
            if (!res_collect<3, NT>(v3, L, A.slots, tag)) {
                if (t == 0) A.R->stall = 1;
                return;
            }
        }
        if (A.last) {  // k_cg1_final
            const double rnorm = sqrt(v3[2]);
            finish(rnorm, A.m1 - 1, (A.m1 > 1 && rnorm < A.eps * bnorm) ? 1 : 2);
            return;
        }
    } else {
        double zr = gprev, rr = v3[1];  // of the iterate that iteration m starts from
        auto sums2 = [&](double (&v2)[2]) {  // z.r, r.r of the own nodes
            v2[0] = v2[1] = 0.0;
#pragma unroll
            for (int o = 0; o < S; o++) {
                if (!flag(o, 8u)) continue;
                v2[0] += (double)s[o].x * (double)r[o].x;
                v2[0] += (double)s[o].y * (double)r[o].y;
                v2[1] += (double)r[o].x * (double)r[o].x;
                v2[1] += (double)r[o].y * (double)r[o].y;
            }
        };
        auto scale = [&]() {  // z = r ./ D (CG.h:412)
#pragma unroll
            for (int o = 0; o < S; o++) {
                const Vec2<T> d = sd[o * NT];
                s[o].x = r[o].x / d.x;
                s[o].y = r[o].y / d.y;
            }
        };
        double v2[2];
        scale();
        double zrprev = v3[0];
        if (A.m0 == 0) {
            sums2(v2);
            res_publish<2, NT>(v2, L, A.slots, tag);
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
            for (int o = 0; o < S; o++) {
                p[o].x = tb * p[o].x + s[o].x;  // xeaxpy: p = beta p + z (CG.h:42-49)
                p[o].y = tb * p[o].y + s[o].y;
                if (flag(o, 8u)) su[(row0 + o + 1) * ss + c + 1] = p[o];
            }
            if (hq >= 0) {
                Vec2<T> hs = sh[nh];
                const Vec2<T> hr = sh[0], hd = sh[2 * nh];
                hs.x = tb * hs.x + hr.x / hd.x;
                hs.y = tb * hs.y + hr.y / hd.y;
                su[hq] = hs;
                sh[nh] = hs;
            }
            __syncthreads();
            double acc[1] = {0.0};
            apply(tag, k & 1, acc[0]);
            res_publish<1, NT>(acc, L, A.slots, tag);
            res_pause<SR>();
            if (hq >= 0 && !res_wait_pair(A.halo + ((k & 1) * nn + (unsigned)hn) * NWD, tag, hw)) L.bad = 1;
            if (!res_collect<1, NT>(acc, L, A.slots, tag)) {
                if (t == 0) A.R->stall = 1;
                return;
            }
            tag++;
            const double alpha = wave_uniform(zr / acc[0]);  // CG.h:433
            const T ta = (T)alpha, tma = (T)(-alpha);
#pragma unroll
            for (int o = 0; o < S; o++) {
                r[o].x = r[o].x + tma * w[o].x;
                r[o].y = r[o].y + tma * w[o].y;
            }
            if (hq >= 0) {
                Vec2<T> hr = sh[0];
                hr.x = hr.x + tma * hw.x;
                hr.y = hr.y + tma * hw.y;
                sh[0] = hr;
            }
            scale();
            sums2(v2);
            res_publish<2, NT>(v2, L, A.slots, tag);
#pragma unroll
            for (int o = 0; o < S; o++) {  // while the sums travel
                Vec2<T> x = sx[o * NT];
                x.x = x.x + ta * p[o].x;
                x.y = x.y + ta * p[o].y;
                sx[o * NT] = x;
            }
            res_pause<SR>();
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
        v3[0] = zrprev;
        v3[1] = rr;
        gprev = zr;
    }
    // the state of the next launch
    store_x();
#pragma unroll
    for (int o = 0; o < S; o++)
        if (flag(o, 8u)) {
            const int n = n0 + (ny + 1) * o;
            store2(A.r, n, r[o]);
            store2(A.p, n, p[o]);
            if (SR) {
                store2(A.s, n, s[o]);
                store2(A.w, n, w[o]);
            }
        }
    if (w0) {
        A.R->v[0] = v3[0];
        A.R->v[1] = v3[1];
        A.R->v[2] = v3[2];
        A.R->g = gprev;
        A.R->a = aprev;
        A.R->bnorm = bnorm;
    }
}

__global__ void k_res_start(PcgDev* __restrict__ S, ResDev* __restrict__ R) {
    S->done = 0;
    S->status = 0;
    S->iterations = 0;
    *R = ResDev{};
}

// What a workgroup that has waited too long does, before a launch of its own:
// that launch's workgroups leave at once or as after any solve, and the host
// goes on with the launched kernels.
__global__ void k_res_stall(ResDev* __restrict__ R) { R->stall = 1; }

}  // namespace pf
