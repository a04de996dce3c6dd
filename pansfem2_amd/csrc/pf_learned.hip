// Learned preconditioner: a 4-level convolutional network on the nodal grid
// of a quad4 problem, BF16 weights and activations with FP32 accumulation on
// the MFMA units (v_mfma_f32_16x16x16_bf16), trained on the device with its
// own forward / data-gradient / weight-gradient kernels and Adam.  No
// counterpart in the reference.  Included by pf_capi.hip.
//
// Tensors are H x W x C, channels fastest, C a multiple of 16; H = nx + 1 and
// W = ny + 1 at the finest level (node (i, j) is pixel (i, j)).
//
// MFMA operand layout (16x16x16, one wavefront; checked on gfx950):
//   A (16 x 16, M x K): lane l holds A[l % 16][4 (l / 16) + t], t = 0..3
//   B (16 x 16, K x N): lane l holds B[4 (l / 16) + t][l % 16]
//   D (16 x 16, M x N): lane l holds D[4 (l / 16) + t][l % 16]
// A convolution is O^T (Cout x pixels) = W (Cout x 9 Cin) . X_col (9 Cin x pixels):
// W is stored [tap][Cout][Cin] so A fragments are 8-byte loads, X fragments
// are 8-byte loads of 4 channels of one pixel, D fragments 8-byte stores.
#pragma once

namespace pf {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

union F32Bits {
    float f;
    uint32_t u;
};

__device__ __host__ inline bf16 f2bf(float f) {
    // round to nearest even (no NaN inputs occur here)
    F32Bits b;
    b.f = f;
    uint32_t u = b.u;
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16)(u >> 16);
}

__device__ __host__ inline float bf2f(bf16 h) {
    F32Bits b;
    b.u = (uint32_t)h << 16;
    return b.f;
}

__device__ inline bf16x4 ld4(const bf16* p) { return *reinterpret_cast<const bf16x4*>(p); }

// ------------------------------------------------------------- forward ---
// Tiles of 4 RPW image rows x 64 pixels, each workgroup taking tiles b,
// b + G, ... (G workgroups).  The layer's weights are staged in LDS
// once per workgroup; a tile's input and its one-pixel halo (4 RPW + 2 rows
// of 66 pixels) are staged in LDS, the next tile's being loaded into
// registers while the current one is computed.  Wave w computes rows w,
// w + 4, ... (RPW of them) of the tile as four 16-pixel groups each, so each
// weight fragment (tap, output block, input block) feeds 4 RPW MFMAs.  Per
// output the sum runs over taps, then input blocks of 16 channels.
// relu: 0 linear, 1 ReLU.  OUT: kConvOutBf16 writes the BF16 result to Y,
// kConvOutF32 the FP32 one to Yf, kConvOutNodal channels 0 and 1 of each
// pixel (node) as FP64 to Yn[2 n], Yn[2 n + 1], 0 where bit 0 / bit 1 of
// fix[n] marks the DOF fixed (the network's output field, in the layout of
// the solver's nodal vectors).  With 64 channels in or out the LDS copies
// take 62-88 KB (one or two workgroups per CU): those layers are the
// coarsest (129 x 65 pixels at 1024 x 512 elements), a few dozen tiles.
//
// LDS layout: both copies hold chunks of 8 channels outermost ([chunk][pixel]
// [8] and [tap][chunk][Cout][8]), so that each half-wave of an operand read
// (lanes (g, pl), g = 2h, 2h + 1: channels 4g.. of pixel or output channel
// pl) covers 256 contiguous bytes, every bank once.  With the channels of a
// pixel contiguous (the global layout) a half-wave's 16 pixels spread over
// 512 or 1024 bytes, two or four lanes to a bank.  The input chunks are
// NPXP >= NPX pixels apart, NPXP = 16 / CH mod 16, so that the staging writes
// (consecutive lanes: the chunks of one pixel) start the chunks in different
// banks.
//
// Memory accesses are buffer loads and stores, with out-of-range offsets for
// pixels outside the image (loads return zeros, stores are dropped), so that
// no branch skips one: every iteration then issues the same loads and
// stores, and the wait for the next tile's loads lets this tile's stores stay
// in flight.
constexpr int kConvTW = 64;
constexpr uint32_t kBufOut = 0x80000000u;  // an offset past every buffer's range
enum { kConvOutBf16, kConvOutF32, kConvOutNodal };
__device__ inline __amdgpu_buffer_rsrc_t conv_buf(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
template <int CIN, int COUT, int RPW, int OUT>
__global__ void __launch_bounds__(256) k_conv_fwd(int H, int W, const bf16* __restrict__ X, const bf16* __restrict__ Wt,
                                                  bf16* __restrict__ Y, float* __restrict__ Yf, int relu,
                                                  const uint8_t* __restrict__ fix, double* __restrict__ Yn) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4v __attribute__((ext_vector_type(4)));
    constexpr int TR = 4 * RPW, SW = kConvTW + 2, SR = TR + 2, CH = CIN / 8;  // 16-byte chunks per pixel
    constexpr int CT = COUT / 16, KT = CIN / 16;
    constexpr int NW = 9 * COUT * CIN;                      // the layer's weights
    constexpr int NPX = SR * SW;                            // pixels of a staged tile
    constexpr int NPXP = NPX + ((16 / CH - NPX) % 16 + 16) % 16;
    constexpr int NE = NPX * CH;                            // 16-byte chunks of a staged tile
    constexpr int PF = (NE + 255) / 256;                    // of them per thread
    static_assert(NPXP % 16 == (16 / CH) % 16, "chunk stride");
    static_assert(OUT != kConvOutNodal || (RPW == 1 && COUT == 16), "nodal output: one 4 x 64 tile, 16 channels");
    __shared__ __align__(16) bf16 sx[CH * NPXP * 8];
    __shared__ __align__(16) bf16 sw[NW];
    __shared__ uint8_t sfix[OUT == kConvOutNodal ? 256 : 1];  // fixity bits of the tile's own pixels
    const uint32_t npix = (uint32_t)H * (uint32_t)W;
    const __amdgpu_buffer_rsrc_t rx = conv_buf(X, npix * CIN * 2);
    const __amdgpu_buffer_rsrc_t ry = OUT == kConvOutNodal ? conv_buf(Yn, npix * 16)
                                      : OUT == kConvOutF32 ? conv_buf(Yf, npix * COUT * 4)
                                                           : conv_buf(Y, npix * COUT * 2);
    const __amdgpu_buffer_rsrc_t rf = conv_buf(fix, OUT == kConvOutNodal ? npix : 0);
    const int tilesJ = (W + kConvTW - 1) / kConvTW, ntiles = ((H + TR - 1) / TR) * tilesJ;
    u32x4 pre[PF];
    uint8_t fpre = 0;
    // tile t's input chunks (zeros outside the image and for t >= ntiles)
    // and, for the nodal output, the fixity bits of its own pixels
    auto fetch = [&](int t) {
        const int i0 = (t / tilesJ) * TR, j0 = (t % tilesJ) * kConvTW;
        if constexpr (OUT == kConvOutNodal) {
            const int i = i0 + (threadIdx.x >> 6), j = j0 + (threadIdx.x & 63);
            fpre = __builtin_amdgcn_raw_buffer_load_b8(rf, i < H && j < W ? (uint32_t)(i * W + j) : kBufOut, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + 256 * u;
            const int pix = e / CH, ch = e - pix * CH;
            const int r = pix / SW, cc = pix - r * SW;
            const int ii = i0 - 1 + r, jj = j0 - 1 + cc;
            const bool in = e < NE && ii >= 0 && ii < H && jj >= 0 && jj < W;
            const uint32_t off = in ? ((uint32_t)(ii * W + jj) * CIN + ch * 8) * 2 : kBufOut;
            pre[u] = __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0);
        }
    };
    auto stage = [&] {
        if constexpr (OUT == kConvOutNodal) sfix[threadIdx.x] = fpre;
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + 256 * u;
            if (NE % 256 == 0 || e < NE) {
                const int pix = e / CH, ch = e - pix * CH;
                *reinterpret_cast<u32x4*>(sx + (ch * NPXP + pix) * 8) = pre[u];
            }
        }
    };
    fetch(blockIdx.x);
    for (int e = threadIdx.x; e < NW / 8; e += 256) {
        // global [tap][co][ci] -> LDS [tap][ci / 8][co][8]
        const int ci = (8 * e) % CIN, co = ((8 * e) / CIN) % COUT, tap = (8 * e) / (CIN * COUT);
        *reinterpret_cast<uint4*>(sw + ((tap * CH + ci / 8) * COUT + co) * 8) =
            *reinterpret_cast<const uint4*>(Wt + 8 * e);
    }
    stage();
    __syncthreads();
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int g = l >> 4, pl = l & 15;
    const int hw = g >> 1, lo = (g & 1) * 4;  // the lane's chunk within a 16-channel block, and its 4 channels
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        fetch(t + gridDim.x);  // in flight during this tile
        const int i0 = (t / tilesJ) * TR, j0 = (t % tilesJ) * kConvTW;
        f32x4 acc[RPW][4][CT];
#pragma unroll
        for (int h = 0; h < RPW; h++)
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int c = 0; c < CT; c++) acc[h][q][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int dr = tap / 3, dc = tap % 3;
#pragma unroll
            for (int kc = 0; kc < KT; kc++) {
                const int ch = 2 * kc + hw;
                bf16x4 b[RPW][4];
#pragma unroll
                for (int h = 0; h < RPW; h++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        b[h][q] = *reinterpret_cast<const bf16x4*>(
                            sx + (ch * NPXP + (wave + 4 * h + dr) * SW + q * 16 + pl + dc) * 8 + lo);
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    const int co = c * 16 + pl;
                    const bf16x4 a = *reinterpret_cast<const bf16x4*>(sw + ((tap * CH + ch) * COUT + co) * 8 + lo);
#pragma unroll
                    for (int h = 0; h < RPW; h++)
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            acc[h][q][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[h][q], acc[h][q][c], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int h = 0; h < RPW; h++) {
            const int i = i0 + wave + 4 * h;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int px = j0 + q * 16 + pl;
                const bool in = i < H && px < W;
                const uint32_t o = (uint32_t)(i * W + px) * COUT;
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    float v[4];
#pragma unroll
                    for (int tt = 0; tt < 4; tt++) {
                        v[tt] = acc[h][q][c][tt];
                        if (relu && v[tt] < 0.f) v[tt] = 0.f;
                    }
                    const uint32_t co = c * 16 + 4 * g;
                    if constexpr (OUT == kConvOutNodal) {
                        // lanes g = 0 hold channels 0..3 of their pixel
                        const uint8_t fx = sfix[wave * 64 + q * 16 + pl];
                        const double v0 = (fx & 1) ? 0.0 : (double)v[0], v1 = (fx & 2) ? 0.0 : (double)v[1];
                        typedef double f64x2 __attribute__((ext_vector_type(2)));
                        const f64x2 pk = {v0, v1};
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pk), ry,
                                                               in && g == 0 ? (o / COUT) * 16 : kBufOut, 0, 0);
                    } else if constexpr (OUT == kConvOutF32) {
                        const f32x4v pk = {v[0], v[1], v[2], v[3]};
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pk), ry,
                                                               in ? (o + co) * 4 : kBufOut, 0, 0);
                    } else {
                        const u32x2 pk = {(uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                                          (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16)};
                        __builtin_amdgcn_raw_buffer_store_b64(pk, ry, in ? (o + co) * 2 : kBufOut, 0, 0);
                    }
                }
            }
        }
        __syncthreads();  // every wave's reads of this tile are done
        stage();
        __syncthreads();
    }
}

// 3x3x3 convolution on an H x W x Dp node grid (channels last), tiled like
// k_conv_fwd: a tile is 4 node lines (j) x 16 NQ nodes (k) of one plane i,
// wave w computing line j0 + w as NQ 16-node groups; the tile's input and
// its one-node halo (3 planes x 6 lines x (16 NQ + 2) nodes) staged in LDS
// in 8-channel chunks outermost, the next tile's loaded into registers
// meanwhile; the layer's weights staged once per workgroup,
// [tap][chunk][Cout][8].  Per output the sum runs over taps 9 (di+1) +
// 3 (dj+1) + (dk+1), then input blocks of 16 channels, as in k_conv3_fwd, so
// the two kernels agree bit for bit.  OUT as for k_conv_fwd; the nodal output
// has three DOFs per node (Yn[3 n + c], c = 0..2).
constexpr int kConv3TJ = 4;
template <int CIN, int COUT, int OUT, int NQ>
__global__ void __launch_bounds__(256) k_conv3_fwd_tile(int H, int W, int Dp, const bf16* __restrict__ X,
                                                        const bf16* __restrict__ Wt, bf16* __restrict__ Y,
                                                        float* __restrict__ Yf, int relu,
                                                        const uint8_t* __restrict__ fix, double* __restrict__ Yn) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4v __attribute__((ext_vector_type(4)));
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    constexpr int CH = CIN / 8, CT = COUT / 16, KT = CIN / 16;
    constexpr int TK = 16 * NQ, SJ = kConv3TJ + 2, SK = TK + 2;
    constexpr int NW = 27 * COUT * CIN;
    constexpr int NPX = 3 * SJ * SK;
    constexpr int NPXP = NPX + ((16 / CH - NPX) % 16 + 16) % 16;
    constexpr int NE = NPX * CH;
    constexpr int PF = (NE + 255) / 256;
    constexpr int NOWN = kConv3TJ * TK, FPT = (NOWN + 255) / 256;  // own nodes, their fixity bytes per thread
    static_assert((CH * NPXP * 8 + NW) * 2 <= 160 * 1024 - 1024, "staged tile and weights within the LDS");
    __shared__ __align__(16) bf16 sx[CH * NPXP * 8];
    __shared__ __align__(16) bf16 sw[NW];
    __shared__ uint8_t sfix[OUT == kConvOutNodal ? 256 * FPT : 1];
    const uint32_t npix = (uint32_t)H * (uint32_t)W * (uint32_t)Dp;
    const __amdgpu_buffer_rsrc_t rx = conv_buf(X, npix * CIN * 2);
    const __amdgpu_buffer_rsrc_t ry = OUT == kConvOutNodal ? conv_buf(Yn, npix * 24)
                                      : OUT == kConvOutF32 ? conv_buf(Yf, npix * COUT * 4)
                                                           : conv_buf(Y, npix * COUT * 2);
    const __amdgpu_buffer_rsrc_t rf = conv_buf(fix, OUT == kConvOutNodal ? npix : 0);
    const int ntj = (W + kConv3TJ - 1) / kConv3TJ, ntk = (Dp + TK - 1) / TK;
    const int ntiles = H * ntj * ntk;
    u32x4 pre[PF];
    uint8_t fpre[FPT];
    auto origin = [&](int t, int& i, int& j0, int& k0) {
        i = t / (ntj * ntk);
        const int rem = t - i * (ntj * ntk);
        j0 = (rem / ntk) * kConv3TJ;
        k0 = (rem - (rem / ntk) * ntk) * TK;
    };
    // tile t's input (zeros outside the grid and for t >= ntiles)
    auto fetch = [&](int t) {
        int i, j0, k0;
        origin(t, i, j0, k0);
        if constexpr (OUT == kConvOutNodal) {
#pragma unroll
            for (int u = 0; u < FPT; u++) {
                const int o = threadIdx.x + 256 * u;
                const int j = j0 + o / TK, k = k0 + o % TK;
                const bool in = o < NOWN && i < H && j < W && k < Dp;
                fpre[u] =
                    __builtin_amdgcn_raw_buffer_load_b8(rf, in ? (uint32_t)((i * W + j) * Dp + k) : kBufOut, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + 256 * u;
            const int pix = e / CH, ch = e - pix * CH;
            const int a = pix / (SJ * SK), rem = pix - a * (SJ * SK);
            const int bj = rem / SK, bk = rem - bj * SK;
            const int ii = i - 1 + a, jj = j0 - 1 + bj, kk = k0 - 1 + bk;
            const bool in = e < NE && ii >= 0 && ii < H && jj >= 0 && jj < W && kk >= 0 && kk < Dp;
            const uint32_t off = in ? (((uint32_t)((ii * W + jj) * Dp + kk)) * CIN + ch * 8) * 2 : kBufOut;
            pre[u] = __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0);
        }
    };
    auto stage = [&] {
        if constexpr (OUT == kConvOutNodal) {
#pragma unroll
            for (int u = 0; u < FPT; u++) sfix[threadIdx.x + 256 * u] = fpre[u];
        }
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + 256 * u;
            if (NE % 256 == 0 || e < NE) {
                const int pix = e / CH, ch = e - pix * CH;
                *reinterpret_cast<u32x4*>(sx + (ch * NPXP + pix) * 8) = pre[u];
            }
        }
    };
    fetch(blockIdx.x);
    for (int e = threadIdx.x; e < NW / 8; e += 256) {
        const int ci = (8 * e) % CIN, co = ((8 * e) / CIN) % COUT, tap = (8 * e) / (CIN * COUT);
        *reinterpret_cast<uint4*>(sw + ((tap * CH + ci / 8) * COUT + co) * 8) =
            *reinterpret_cast<const uint4*>(Wt + 8 * e);
    }
    stage();
    __syncthreads();
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int g = l >> 4, pl = l & 15;
    const int hw = g >> 1, lo = (g & 1) * 4;
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        fetch(t + gridDim.x);  // in flight during this tile
        int i, j0, k0;
        origin(t, i, j0, k0);
        const int j = j0 + wave;
        // the lane's LDS offsets (elements), opaque to the compiler per tile,
        // so that a tap's offset stays an instruction immediate rather than
        // one of 27 x NQ hoisted addresses
        int xo = (hw * NPXP + wave * SK + pl) * 8 + lo, wo = (hw * COUT + pl) * 8 + lo;
        asm volatile("" : "+v"(xo), "+v"(wo));
        f32x4 acc[NQ][CT];
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int c = 0; c < CT; c++) acc[q][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tap = 0; tap < 27; tap++) {
            const int di = tap / 9, dj = (tap / 3) % 3, dk = tap % 3;
#pragma unroll
            for (int kc = 0; kc < KT; kc++) {
                bf16x4 b[NQ];
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    b[q] = *reinterpret_cast<const bf16x4*>(sx + xo +
                                                            (2 * kc * NPXP + (di * SJ + dj) * SK + q * 16 + dk) * 8);
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    const bf16x4 a = *reinterpret_cast<const bf16x4*>(sw + wo + ((tap * CH + 2 * kc) * COUT + c * 16) * 8);
#pragma unroll
                    for (int q = 0; q < NQ; q++)
                        acc[q][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[q], acc[q][c], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int k = k0 + q * 16 + pl;
            const bool in = j < W && k < Dp;
            const uint32_t n = (uint32_t)((i * W + j) * Dp + k);
#pragma unroll
            for (int c = 0; c < CT; c++) {
                float v[4];
#pragma unroll
                for (int tt = 0; tt < 4; tt++) {
                    v[tt] = acc[q][c][tt];
                    if (relu && v[tt] < 0.f) v[tt] = 0.f;
                }
                const uint32_t co = c * 16 + 4 * g;
                if constexpr (OUT == kConvOutNodal) {
                    // lanes g = 0 hold channels 0..3 of their node
                    const uint8_t fx = sfix[wave * TK + q * 16 + pl];
                    const f64x2 p01 = {(fx & 1) ? 0.0 : (double)v[0], (fx & 2) ? 0.0 : (double)v[1]};
                    const double v2 = (fx & 4) ? 0.0 : (double)v[2];
                    const bool w0 = in && g == 0;
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, p01), ry, w0 ? n * 24 : kBufOut,
                                                           0, 0);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v2), ry, w0 ? n * 24 + 16 : kBufOut,
                                                          0, 0);
                } else if constexpr (OUT == kConvOutF32) {
                    const f32x4v pk = {v[0], v[1], v[2], v[3]};
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pk), ry,
                                                           in ? (n * COUT + co) * 4 : kBufOut, 0, 0);
                } else {
                    const u32x2 pk = {(uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                                      (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16)};
                    __builtin_amdgcn_raw_buffer_store_b64(pk, ry, in ? (n * COUT + co) * 2 : kBufOut, 0, 0);
                }
            }
        }
        __syncthreads();  // every wave's reads of this tile are done
        stage();
        __syncthreads();
    }
}

// -------------------------------------------------------- weight gradient --
// dW[tap][co][ci] = sum_p dZ[p][co] X[p + off(tap)][ci] (2D: DIM = 2, taps
// 3 (di + 1) + (dj + 1); 3D: DIM = 3 on H x W x Dp, taps 9 (di + 1) +
// 3 (dj + 1) + (dk + 1)), FP32 partials per block of ppb pixels (reduced
// afterwards in a fixed order).  One workgroup per (block, line offset, tile of
// channels): it computes the three taps that differ along the contiguous axis from one
// staged copy of X.  dZ and X (the piece's pixels shifted by the line offset,
// and one more on each side) go to LDS as they are in memory, 256 pixels at a
// time, in planes of 16 channels, 32 bytes per pixel; the next piece is on its
// way in registers meanwhile, and the two LDS buffers alternate, one barrier
// per piece.  The matrix core wants four pixels of one channel per lane: the
// transposing LDS read gives them, lane i of a group of 16 pointing at channels
// 4 (i & 3) .. + 3 of pixel i >> 2 and getting channel i of the four pixels.
// A neighbour outside the grid is a lane pointing at a pixel of zeros, so a
// shift by one pixel is an address, and no copy per tap is needed.  Each
// accumulator sums its MFMAs over the block's 16-pixel chunks in pixel order.
//
// Bound by the latency of a block's 16 pieces, whose order is fixed.  At 1025 x 513
// nodes and below, per launch: 16 -> 16 channels 27.8 us, 32 -> 32 30.5, 16 <-> 32
// 26, 32 <-> 64 31; one workgroup per tap that transposed its own copies with
// 2-byte LDS stores took 53.8, 64.8, 56 and 102.  A wave per (16 x 16 pair, tap)
// and tiles of at most 32 x 32 channels: with the three taps in one wave 32 -> 32
// took 58.6 and 32 <-> 64 67; with the LDS reads next to their products instead
// of eight chunks ahead 68.7 and 75.
constexpr int wgrad_tile(int c) { return c < 32 ? c : 32; }
constexpr int wgrad_waves(int cin, int cout) { return 3 * (wgrad_tile(cin) / 16) * (wgrad_tile(cout) / 16); }
constexpr int wgrad_tiles(int cin, int cout) { return (cin / wgrad_tile(cin)) * (cout / wgrad_tile(cout)); }

template <int DIM, int CIN, int COUT>
__global__ void __launch_bounds__(64 * wgrad_waves(CIN, COUT))
    k_conv_wgrad(int H, int W, int Dp, const bf16* __restrict__ X, const bf16* __restrict__ dZ,
                 float* __restrict__ part, int ppb) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int NTAP = DIM == 3 ? 27 : 9;
    constexpr int TI = wgrad_tile(CIN), TO = wgrad_tile(COUT);  // the workgroup's channels
    constexpr int CT = TO / 16, KT = TI / 16;
    constexpr int NT = 64 * wgrad_waves(CIN, COUT);
    constexpr int SP = 256;                            // pixels per piece
    constexpr int XP = SP + 2, XS = XP + 1;            // staged pixels of X, and the pixel of zeros
    constexpr int NZ = SP * TO / 8, NX = XP * TI / 8;  // 16-byte chunks
    constexpr int RZ = (NZ + NT - 1) / NT, RX = (NX + NT - 1) / NT;
    constexpr int BZ = CT * SP * 16, BX = KT * XS * 16;
    __shared__ __align__(16) bf16 sm[2 * (BZ + BX)];
    const int outer = blockIdx.y;  // the tap's offset along all but the contiguous axis
    const int di = DIM == 3 ? outer / 3 - 1 : outer - 1;
    const int dj = DIM == 3 ? outer % 3 - 1 : 0;
    const int D = DIM == 3 ? Dp : W;         // pixels of a line
    const int L = DIM == 3 ? W : 1;          // lines per i
    const long npx = (long)H * L * D;
    const long off = ((long)di * L + dj) * D;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, c16 = l & 15;
    const int pair = wave / 3, tap = wave - 3 * pair, d = tap - 1;
    const int ct = pair / KT, kt = pair - ct * KT;
    const int ti = (int)blockIdx.z % (CIN / TI) * TI, to = (int)blockIdx.z / (CIN / TI) * TO;
    const long p_begin = (long)blockIdx.x * ppb;
    const long p_end = p_begin + ppb < npx ? p_begin + ppb : npx;
    for (int e = threadIdx.x; e < 2 * KT * 16; e += NT)
        sm[(e / (KT * 16)) * (BZ + BX) + BZ + ((e / 16) % KT) * XS * 16 + XP * 16 + e % 16] = 0;
    u32x4 rz[RZ], rx[RX];
    // pixels outside the tensor are read at its nearest pixel: dZ's are zeroed when
    // they are staged, X's belong to taps that point at the zeros
    auto fetch = [&](long s0) {
#pragma unroll
        for (int u = 0; u < RZ; u++) {
            const int e = threadIdx.x + NT * u, px = e / (TO / 8), ch = e - px * (TO / 8);
            const long p = s0 + px < npx ? s0 + px : npx - 1;
            rz[u] = *reinterpret_cast<const u32x4*>(dZ + p * COUT + to + ch * 8);
        }
#pragma unroll
        for (int u = 0; u < RX; u++) {
            const int e = threadIdx.x + NT * u, px = e / (TI / 8), ch = e - px * (TI / 8);
            long p = s0 + off - 1 + px;
            p = p < 0 ? 0 : p < npx ? p : npx - 1;
            rx[u] = *reinterpret_cast<const u32x4*>(X + p * CIN + ti + ch * 8);
        }
    };
    auto stage = [&](long s0, bf16* buf) {
#pragma unroll
        for (int u = 0; u < RZ; u++) {
            const int e = threadIdx.x + NT * u, px = e / (TO / 8), ch = e - px * (TO / 8);
            if (NZ % NT == 0 || e < NZ)
                *reinterpret_cast<u32x4*>(buf + ((ch >> 1) * SP + px) * 16 + (ch & 1) * 8) =
                    s0 + px < p_end ? rz[u] : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < RX; u++) {
            const int e = threadIdx.x + NT * u, px = e / (TI / 8), ch = e - px * (TI / 8);
            if (NX % NT == 0 || e < NX)
                *reinterpret_cast<u32x4*>(buf + BZ + ((ch >> 1) * XS + px) * 16 + (ch & 1) * 8) = rx[u];
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // the pixel this lane points at, 4 g + (c16 >> 2) of each chunk: its place on the
    // grid, advanced by 16 pixels per chunk
    const int lp = 4 * g + (c16 >> 2);
    int left = (int)(p_end - p_begin) - lp;  // pixels of the block from here on
    int pi, pj, pk;
    {
        const long p = p_begin + lp, line = p / D;
        pk = (int)(p - line * D);
        pi = (int)(line / L);
        pj = (int)(line - (long)pi * L);
    }
    const int sk = 16 % D, sj = (16 / D) % L, si = (16 / D) / L;
    fetch(p_begin);
    int b = 0;
    for (long s0 = p_begin; s0 < p_end; s0 += SP, b ^= 1) {
        bf16* buf = sm + b * (BZ + BX);
        stage(s0, buf);
        __syncthreads();  // staged; and every wave has read the piece before the last one
        if (s0 + SP < p_end) fetch(s0 + SP);
        const bf16* z = buf + ct * SP * 16 + lp * 16 + 4 * (c16 & 3);
        const bf16* x = buf + BZ + kt * XS * 16 + 4 * (c16 & 3);
        // whole pieces (chunks past the block add zeros), eight chunks at a time: their
        // LDS reads are all issued before their products
        for (int c0 = 0; c0 < SP / 16; c0 += 8) {
            bf16x4 a[8], v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int c = c0 + u;
                const bool in = (left > 0) & ((unsigned)(pi + di) < (unsigned)H) &
                                (DIM == 2 || (unsigned)(pj + dj) < (unsigned)W);
                a[u] = __builtin_bit_cast(bf16x4,
                                          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(z + c * 256)));
                const int px = (in & ((unsigned)(pk + d) < (unsigned)D)) ? 16 * c + lp + tap : XP;
                v[u] = __builtin_bit_cast(bf16x4,
                                          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(x + px * 16)));
                left -= 16;
                pk += sk;
                const int cy = pk >= D;
                pk -= cy ? D : 0;
                if (DIM == 2) {
                    pi += si + cy;
                } else {
                    pj += sj + cy;
                    const int cj = pj >= W;
                    pj -= cj ? W : 0;
                    pi += si + cj;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 8; u++) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[u], v[u], acc, 0, 0, 0);
        }
    }
    float* out = part + (long)blockIdx.x * NTAP * COUT * CIN;
#pragma unroll
    for (int t = 0; t < 4; t++)
        out[((long)(3 * outer + tap) * COUT + to + ct * 16 + 4 * g + t) * CIN + ti + kt * 16 + c16] = acc[t];
}

// The blocks' partials in block order, 16 loads in flight (4.8 us a layer; 14.6
// one by one).
__global__ void k_wgrad_reduce(const float* __restrict__ part, int nparts, int n, float* __restrict__ dW) {
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        float s = 0.f;
        int b = 0;
        for (; b + 16 <= nparts; b += 16) {
            float v[16];
#pragma unroll
            for (int t = 0; t < 16; t++) v[t] = part[(long)(b + t) * n + q];
#pragma unroll
            for (int t = 0; t < 16; t++) s += v[t];
        }
        for (; b < nparts; b++) s += part[(long)b * n + q];
        dW[q] = s;
    }
}

// ------------------------------------------------- elementwise / resample --
// average pooling 2x2 (ceil), coarse (Hc, Wc) from fine (H, W)
// Eight channels (16 bytes) per access: C is a multiple of 16.
__device__ inline void unpack8(uint4 v, float (&f)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int t = 0; t < 8; t++) f[t] = bf2f((bf16)((t & 1) ? (w[t >> 1] >> 16) : (w[t >> 1] & 0xFFFFu)));
}
__device__ inline uint4 pack8(const float (&f)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = (uint32_t)f2bf(f[2 * k]) | ((uint32_t)f2bf(f[2 * k + 1]) << 16);
    return uint4{w[0], w[1], w[2], w[3]};
}

__global__ void k_pool2(int H, int W, int C, const bf16* __restrict__ in, bf16* __restrict__ out) {
    const int Hc = (H + 1) / 2, Wc = (W + 1) / 2, C8 = C / 8;
    const long n8 = (long)Hc * Wc * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long pc = q / C8;
        const int I = (int)(pc / Wc), J = (int)(pc - (long)I * Wc);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        int cnt = 0;
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++) {
                int i = 2 * I + a, j = 2 * J + b;
                if (i < H && j < W) {
                    float f[8];
                    unpack8(*reinterpret_cast<const uint4*>(in + ((long)i * W + j) * C + 8 * c8), f);
#pragma unroll
                    for (int t = 0; t < 8; t++) s[t] += f[t];
                    cnt++;
                }
            }
#pragma unroll
        for (int t = 0; t < 8; t++) s[t] = s[t] / (float)cnt;
        *reinterpret_cast<uint4*>(out + 8 * q) = pack8(s);
    }
}

// ReLU's backward on eight channels: the gradient where the output is positive.
__device__ inline uint4 relu_mask8(uint4 y, uint4 d) {
    auto two = [](uint32_t v, uint32_t g) {
        return (bf2f((bf16)(v & 0xFFFFu)) > 0.f ? g & 0xFFFFu : 0u) | (bf2f((bf16)(v >> 16)) > 0.f ? g & 0xFFFF0000u : 0u);
    };
    return {two(y.x, d.x), two(y.y, d.y), two(y.z, d.z), two(y.w, d.w)};
}

__global__ void k_relu_bwd(long n8, const uint4* __restrict__ Y, uint4* __restrict__ dY) {
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x)
        dY[q] = relu_mask8(Y[q], dY[q]);
}

// The elementwise steps between two layers of the backward pass, in one sweep of
// 16-byte accesses each, for H x W x Dp nodes (Dp = 1 in 2D).  Bound by memory and,
// on the coarse levels, by the launch; as separate passes of 2-byte accesses they
// took 30 us (copy 7.5, pooling 15.9, ReLU 6.9) and 16 us (upsampling 9.4, ReLU
// 6.9) in the mean over the levels of 1025 x 513 nodes, the two kernels take 8.7
// and 5.7 us.
//
// An encoder output's gradient, at ReLU: the skip branch's plus the pooled
// branch's (average over the coarse node's children).  Y is the output.
__global__ void k_skip_pool_bwd(int H, int W, int Dp, int C, const bf16* __restrict__ dskip,
                                const bf16* __restrict__ dcoarse, const bf16* __restrict__ Y, bf16* __restrict__ dY) {
    const int Wc = (W + 1) / 2, Dc = (Dp + 1) / 2, C8 = C / 8;
    const long plane = (long)W * Dp, n8 = (long)H * plane * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long p = q / C8;
        const int i = (int)(p / plane);
        const long rem = p - (long)i * plane;
        const int j = (int)(rem / Dp), k = (int)(rem - (long)j * Dp);
        const int I = i / 2, J = j / 2, K = k / 2;
        const int cnt = ((2 * I + 1 < H) ? 2 : 1) * ((2 * J + 1 < W) ? 2 : 1) * ((2 * K + 1 < Dp) ? 2 : 1);
        float fs[8], fc[8];
        unpack8(*reinterpret_cast<const uint4*>(dskip + 8 * q), fs);
        unpack8(*reinterpret_cast<const uint4*>(dcoarse + (((long)I * Wc + J) * Dc + K) * C + 8 * c8), fc);
#pragma unroll
        for (int t = 0; t < 8; t++) fs[t] = fs[t] + fc[t] / (float)cnt;
        *reinterpret_cast<uint4*>(dY + 8 * q) = relu_mask8(*reinterpret_cast<const uint4*>(Y + 8 * q), pack8(fs));
    }
}

// A decoder output's gradient, at ReLU: the sum over the coarse node's children
// of the upsampled field's gradient.
__global__ void k_up_bwd(int H, int W, int Dp, int C, const bf16* __restrict__ dfine, const bf16* __restrict__ Y,
                         bf16* __restrict__ dY) {
    const int Hc = (H + 1) / 2, Wc = (W + 1) / 2, Dc = (Dp + 1) / 2, C8 = C / 8;
    const long n8 = (long)Hc * Wc * Dc * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long pc = q / C8;
        const int I = (int)(pc / ((long)Wc * Dc));
        const long rem = pc - (long)I * Wc * Dc;
        const int J = (int)(rem / Dc), K = (int)(rem - (long)J * Dc);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++)
                for (int cc = 0; cc < 2; cc++) {
                    const int i = 2 * I + a, j = 2 * J + b, k = 2 * K + cc;
                    if (i >= H || j >= W || k >= Dp) continue;
                    float f[8];
                    unpack8(*reinterpret_cast<const uint4*>(dfine + (((long)i * W + j) * Dp + k) * C + 8 * c8), f);
#pragma unroll
                    for (int t = 0; t < 8; t++) s[t] += f[t];
                }
        *reinterpret_cast<uint4*>(dY + 8 * q) = relu_mask8(*reinterpret_cast<const uint4*>(Y + 8 * q), pack8(s));
    }
}

// out (fine) = nearest-upsampled coarse + skip
__global__ void k_up2_add(int H, int W, int C, const bf16* __restrict__ coarse, const bf16* __restrict__ skip,
                          bf16* __restrict__ out) {
    const int Wc = (W + 1) / 2, C8 = C / 8;
    const long n8 = (long)H * W * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long p = q / C8;
        const int i = (int)(p / W), j = (int)(p - (long)i * W);
        float fc[8], fs[8];
        unpack8(*reinterpret_cast<const uint4*>(coarse + ((long)(i / 2) * Wc + j / 2) * C + 8 * c8), fc);
        unpack8(*reinterpret_cast<const uint4*>(skip + 8 * q), fs);
#pragma unroll
        for (int t = 0; t < 8; t++) fc[t] = fc[t] + fs[t];
        *reinterpret_cast<uint4*>(out + 8 * q) = pack8(fc);
    }
}

// ------------------------------------------------------- network input ----
// x0[p] = (2 rho_node - 1, r_x / s, r_y / s, 0 ...), 16 channels, where
// rho_node is the mean density of the node's elements and s the RMS of r.
// rs scales the residual channels; with rn_dev the scale is *rn_dev / sqrtN
// instead (1 when that is 0), read on the device.
__global__ void k_net_input(int nx, int ny, const double* __restrict__ rho, const double* __restrict__ r, double rs,
                            const double* __restrict__ rn_dev, double sqrtN, bf16* __restrict__ x0) {
    if (rn_dev) rs = *rn_dev > 0 ? *rn_dev / sqrtN : 1.0;
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        double s = 0.0;
        int cnt = 0;
        for (int a = -1; a <= 0; a++)
            for (int b = -1; b <= 0; b++) {
                int ei = i + a, ej = j + b;
                if (ei >= 0 && ei < nx && ej >= 0 && ej < ny) {
                    s += rho[(long)ny * ei + ej];
                    cnt++;
                }
            }
        // channels 0..2, then 13 zeros: two 16-byte stores
        const uint32_t c0 = f2bf((float)(2.0 * (s / cnt) - 1.0)), c1 = f2bf((float)(r[2 * n] / rs)),
                       c2 = f2bf((float)(r[2 * n + 1] / rs));
        uint4* dst = reinterpret_cast<uint4*>(x0 + n * 16);
        dst[0] = uint4{c0 | (c1 << 16), c2, 0u, 0u};
        dst[1] = uint4{0u, 0u, 0u, 0u};
    }
}

// ------------------------------------------------- hex8 (3D) network ----
// The same network on the H x W x Dp node grid of a hex8 mesh (node
// (i, j, k) at ((i W + j) Dp + k), channels last): 3x3x3 convolutions with
// tap = 9 (di + 1) + 3 (dj + 1) + (dk + 1), 2x2x2 pooling and upsampling.

// One workgroup = one (i, j) line, 4 wavefronts x 16 pixels along k; inputs
// and weights read from global memory per tap.
template <int CIN, int COUT>
__global__ void __launch_bounds__(256) k_conv3_fwd(int H, int W, int Dp, const bf16* __restrict__ X,
                                                   const bf16* __restrict__ Wt, bf16* __restrict__ Y,
                                                   float* __restrict__ Yf, int relu) {
    const int i = blockIdx.x / W, j = blockIdx.x - i * W;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int k0 = blockIdx.y * 64 + wave * 16;
    if (k0 >= Dp) return;
    const int pk = k0 + (l & 15);
    const int g = l >> 4;
    f32x4 acc[COUT / 16];
#pragma unroll
    for (int c = 0; c < COUT / 16; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x4 zero = {0, 0, 0, 0};
    for (int tap = 0; tap < 27; tap++) {
        const int ii = i + tap / 9 - 1, jj = j + (tap / 3) % 3 - 1, kk = pk + tap % 3 - 1;
        const bool in = ii >= 0 && ii < H && jj >= 0 && jj < W && kk >= 0 && kk < Dp;
        const bf16* xp = X + (((long)ii * W + jj) * Dp + kk) * CIN;
#pragma unroll
        for (int kc = 0; kc < CIN / 16; kc++) {
            const int ci = kc * 16 + 4 * g;
            const bf16x4 b = in ? ld4(xp + ci) : zero;
#pragma unroll
            for (int c = 0; c < COUT / 16; c++) {
                const int co = c * 16 + (l & 15);
                const bf16x4 a = ld4(Wt + ((long)(tap * COUT + co) * CIN + ci));
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[c], 0, 0, 0);
            }
        }
    }
    if (pk >= Dp) return;
    const long o = (((long)i * W + j) * Dp + pk) * COUT;
#pragma unroll
    for (int c = 0; c < COUT / 16; c++) {
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            v[t] = acc[c][t];
            if (relu && v[t] < 0.f) v[t] = 0.f;
        }
        const int co = c * 16 + 4 * g;
        if (Yf) {
#pragma unroll
            for (int t = 0; t < 4; t++) Yf[o + co + t] = v[t];
        } else {
            bf16x4 pk4 = {(short)f2bf(v[0]), (short)f2bf(v[1]), (short)f2bf(v[2]), (short)f2bf(v[3])};
            *reinterpret_cast<bf16x4*>(Y + o + co) = pk4;
        }
    }
}

// 2x2x2 average pooling with ceil (partial blocks divide by their own
// count), eight channels per thread
__global__ void k_pool3(int H, int W, int Dp, int C, const bf16* __restrict__ in, bf16* __restrict__ out) {
    const int Hc = (H + 1) / 2, Wc = (W + 1) / 2, Dc = (Dp + 1) / 2, C8 = C / 8;
    const long n8 = (long)Hc * Wc * Dc * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long pc = q / C8;
        const int I = (int)(pc / ((long)Wc * Dc));
        const long rem = pc - (long)I * Wc * Dc;
        const int J = (int)(rem / Dc), K = (int)(rem - (long)J * Dc);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        int cnt = 0;
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++)
                for (int c = 0; c < 2; c++) {
                    const int i = 2 * I + a, j = 2 * J + b, k = 2 * K + c;
                    if (i < H && j < W && k < Dp) {
                        float f[8];
                        unpack8(*reinterpret_cast<const uint4*>(in + (((long)i * W + j) * Dp + k) * C + 8 * c8), f);
#pragma unroll
                        for (int t = 0; t < 8; t++) s[t] += f[t];
                        cnt++;
                    }
                }
#pragma unroll
        for (int t = 0; t < 8; t++) s[t] = s[t] / (float)cnt;
        *reinterpret_cast<uint4*>(out + 8 * q) = pack8(s);
    }
}

// out (fine) = nearest-upsampled coarse + skip, eight channels per thread
__global__ void k_up3_add(int H, int W, int Dp, int C, const bf16* __restrict__ coarse, const bf16* __restrict__ skip,
                          bf16* __restrict__ out) {
    const int Wc = (W + 1) / 2, Dc = (Dp + 1) / 2, C8 = C / 8;
    const long plane = (long)W * Dp, n8 = (long)H * plane * C8;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n8; q += (long)gridDim.x * blockDim.x) {
        const int c8 = (int)(q % C8);
        const long p = q / C8;
        const int i = (int)(p / plane);
        const long rem = p - (long)i * plane;
        const int j = (int)(rem / Dp), k = (int)(rem - (long)j * Dp);
        float fc[8], fs[8];
        unpack8(*reinterpret_cast<const uint4*>(coarse + (((long)(i / 2) * Wc + j / 2) * Dc + k / 2) * C + 8 * c8), fc);
        unpack8(*reinterpret_cast<const uint4*>(skip + 8 * q), fs);
#pragma unroll
        for (int t = 0; t < 8; t++) fc[t] = fc[t] + fs[t];
        *reinterpret_cast<uint4*>(out + 8 * q) = pack8(fc);
    }
}

// (2 rho_node - 1, r_x / s, r_y / s, r_z / s) on the hex8 nodes, rho_node the
// mean over the node's (up to eight) elements; element (ei, ej, ek) at
// (ny nz) ei + nz ej + ek
__global__ void k_net_input3(int nx, int ny, int nz, const double* __restrict__ rho, const double* __restrict__ r,
                             double rs, const double* __restrict__ rn_dev, double sqrtN, bf16* __restrict__ x0) {
    if (rn_dev) rs = *rn_dev > 0 ? *rn_dev / sqrtN : 1.0;
    const long plane = (long)(ny + 1) * (nz + 1), nn = (long)(nx + 1) * plane;
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        const int i = (int)(n / plane);
        const long rem = n - (long)i * plane;
        const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
        double s = 0.0;
        int cnt = 0;
        for (int a = -1; a <= 0; a++)
            for (int b = -1; b <= 0; b++)
                for (int c = -1; c <= 0; c++) {
                    const int ei = i + a, ej = j + b, ek = k + c;
                    if (ei >= 0 && ei < nx && ej >= 0 && ej < ny && ek >= 0 && ek < nz) {
                        s += rho[((long)ny * nz) * ei + (long)nz * ej + ek];
                        cnt++;
                    }
                }
        float f[16] = {0};
        f[0] = (float)(2.0 * (s / cnt) - 1.0);
        f[1] = (float)(r[3 * n] / rs);
        f[2] = (float)(r[3 * n + 1] / rs);
        f[3] = (float)(r[3 * n + 2] / rs);
        for (int c = 0; c < 16; c++) x0[n * 16 + c] = f2bf(f[c]);
    }
}

// Up to 32 dot products against one vector in a single pass:
// part[block * nb + j] = sum_i a_i * b_j[i], fixed-order block sums.
struct PtrPack {
    const double* p[32];
};
struct CoefPack {
    double c[32];
};

// NB: the accumulator count (>= nb), so that they stay in registers.  Pairs
// of entries per load; an odd last entry is added by thread 0 of block 0.
template <int NB>
__global__ void __launch_bounds__(256) k_multidot(long n, int nb, const double* __restrict__ a, PtrPack B,
                                                  double* __restrict__ part) {
    __shared__ double lds[16 * NB];
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = 0.0;
    const long n2 = n >> 1;
    const double2* a2 = reinterpret_cast<const double2*>(a);
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n2; i += (long)gridDim.x * blockDim.x) {
        const double2 ai = a2[i];
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (j < nb) {
                const double2 bi = reinterpret_cast<const double2*>(B.p[j])[i];
                acc[j] += ai.x * bi.x;
                acc[j] += ai.y * bi.y;
            }
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (j < nb) acc[j] += a[n - 1] * B.p[j][n - 1];
    }
    block_sum<NB>(acc, lds);
    if (threadIdx.x == 0)
        for (int j = 0; j < nb; j++) part[blockIdx.x * nb + j] = acc[j];
}

// Which partials make up dot d of a batch: part[off[d] + b * nb[d] + q[d]]
// for b < g.
struct DotIdx {
    int off[128];
    short nb[128], q[128];
};

// out[d] = the sum of dot d's g partials, in a fixed order (one workgroup
// per dot)
__global__ void __launch_bounds__(256) k_multidot_final(const double* __restrict__ part, int g, DotIdx idx,
                                                        double* __restrict__ out) {
    __shared__ double lds[16];
    const int d = blockIdx.x;
    const double* p = part + idx.off[d] + idx.q[d];
    const int stride = idx.nb[d];
    double v[1] = {0.0};
    for (int b = threadIdx.x; b < g; b += blockDim.x) v[0] += p[(long)b * stride];
    block_sum<1>(v, lds);
    if (threadIdx.x == 0) out[d] = v[0];
}

// ------------------------------------------- device-resident flexible CG ---
// The learned flexible CG keeps its scalars on the device, so the host
// enqueues iteration k while iteration k-1 still runs and reads a copy of
// this state one iteration behind.  flag: 0 running; 1 the recursive
// residual fell below eps |b| (the host confirms on the true residual);
// 2 fall back to Jacobi-PCG (breakdown, a non-finite residual, divergence
// or stall).  k counts the iterations completed, as the host loop counted
// them; once done is set every later FCG launch leaves x, r and the stored
// directions alone.
struct FcgDev {
    double rn, bn, best, eps, a, c;
    double pq[32], cf[32];
    int k, done, flag, since_best;
};

__global__ void k_fcg_init(FcgDev* __restrict__ S, double bn, double eps) {
    S->rn = bn;
    S->bn = bn;
    S->best = bn;
    S->eps = eps;
    S->a = 1.0;
    S->c = 0.0;
    S->k = 0;
    S->done = 0;
    S->flag = 0;
    S->since_best = 0;
}

// after a recursive residual below eps |b| that the true residual tn did not
// confirm: r has been replaced by the true residual; continue from it
__global__ void k_fcg_resume(FcgDev* __restrict__ S, double tn, double best, int since_best, int fallback) {
    S->rn = tn;
    S->best = best;
    S->since_best = since_best;
    S->flag = fallback ? 2 : 0;
    S->done = fallback ? 1 : 0;
    if (fallback) S->k -= 1;  // that iteration is not counted, as in a stall exit
}

// (a, c) minimising ||a t + c y - e||_K from the five sums t.Kt, t.Ky, t.r,
// y.Ky, y.r; the best-scaled t alone when the 2x2 Gram matrix is singular.
__host__ __device__ inline void pair_from_sums(double tkt, double tky, double tr, double yky, double yr, double* a,
                                               double* c) {
    const double det = tkt * yky - tky * tky;
    if (__builtin_isfinite(det) && det > 1e-12 * tkt * yky && yky > 0.0) {
        *a = (yky * tr - tky * yr) / det;
        *c = (tkt * yr - tky * tr) / det;
    } else {
        *a = tkt > 0.0 ? tr / tkt : 1.0;
        *c = 0.0;
    }
}

// Iteration k's pair (a, c) and orthogonalisation weights
// c_j = z.q_j / p_j.q_j (z = a t + c y) from the first batch of sums:
// T = (t.Kt, t.Ky, t.r, t.q_1..t.q_nst), then Y = (y.Ky, y.r, y.q_1..y.q_nst);
// q_j is the direction stored j + 1 iterations back (slot (k-1-j) mod m).
__global__ void k_fcg_coef(FcgDev* __restrict__ S, const double* __restrict__ sums, int k, int m, int nst) {
    if (S->done || threadIdx.x != 0) return;
    const double* T = sums;
    const double* Y = sums + 3 + nst;
    double a, c;
    pair_from_sums(T[0], T[1], T[2], Y[0], Y[1], &a, &c);
    S->a = a;
    S->c = c;
    for (int j = 0; j < nst; j++) S->cf[j] = (a * T[3 + j] + c * Y[2 + j]) / S->pq[(k - 1 - j + m) % m];
}

// The direction and its image without an operator application: with
// z = a t + c y and K z = a Kt + c Ky,
//   p = z - sum_j c_j P_j,  q = K p = K z - sum_j c_j Q_j.
__global__ void __launch_bounds__(256) k_fcg_direction(long n, int nst, const FcgDev* __restrict__ S,
                                                       const double* __restrict__ t, const double* __restrict__ y,
                                                       const double* __restrict__ Kt, const double* __restrict__ Ky,
                                                       PtrPack P, PtrPack Q, double* __restrict__ p,
                                                       double* __restrict__ q) {
    if (S->done) return;
    const double a = S->a, c = S->c;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        double v = a * t[i] + c * y[i];
        double w = a * Kt[i] + c * Ky[i];
        for (int j = 0; j < nst; j++) {
            v -= S->cf[j] * P.p[j][i];
            w -= S->cf[j] * Q.p[j][i];
        }
        p[i] = v;
        q[i] = w;
    }
}

// x += alpha p, r -= alpha q with alpha = p.r / p.q (sums = (p.q, p.r)), and
// per-workgroup partial sums of the new r.r; nothing on a breakdown (p.q <= 0
// or a non-finite p.r), which k_fcg_check reports
__global__ void __launch_bounds__(256) k_fcg_step(long n, const FcgDev* __restrict__ S,
                                                  const double* __restrict__ sums, const double* __restrict__ p,
                                                  const double* __restrict__ q, double* __restrict__ x,
                                                  double* __restrict__ r, double* __restrict__ part) {
    __shared__ double lds[16];
    if (S->done) return;
    const double pqv = sums[0], pr = sums[1];
    if (!(pqv > 0.0) || !isfinite(pr)) return;
    const double alpha = pr / pqv;
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        x[i] += alpha * p[i];
        const double ri = r[i] - alpha * q[i];
        r[i] = ri;
        acc[0] += ri * ri;
    }
    block_sum<1>(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = acc[0];
}

// |r| from k_fcg_step's partials (fixed order) and the decisions the host
// loop made: breakdown, non-finite, converged (to be confirmed), stall or
// divergence (no halving of the best |r| in `stall` iterations, or 10x above it)
__global__ void __launch_bounds__(256) k_fcg_check(FcgDev* __restrict__ S, const double* __restrict__ sums,
                                                   const double* __restrict__ part, int nb, int slot, int stall) {
    __shared__ double lds[16];
    if (S->done) return;
    const double pqv = sums[0], pr = sums[1];
    const bool breakdown = !(pqv > 0.0) || !isfinite(pr);
    double v[1] = {0.0};
    if (!breakdown)
        for (int b = threadIdx.x; b < nb; b += blockDim.x) v[0] += part[b];
    block_sum<1>(v, lds);
    if (threadIdx.x != 0) return;
    if (breakdown) {
        S->flag = 2;
        S->done = 1;
        return;
    }
    S->pq[slot] = pqv;
    const double rn = sqrt(v[0]);
    if (!isfinite(rn)) {
        S->flag = 2;
        S->done = 1;
        return;
    }
    S->rn = rn;
    if (rn <= S->eps * S->bn) {
        S->k += 1;
        S->flag = 1;
        S->done = 1;
        return;
    }
    if (rn < 0.5 * S->best) {
        S->best = rn;
        S->since_best = 0;
    } else if (++S->since_best >= stall || rn > 10.0 * S->best) {
        S->flag = 2;
        S->done = 1;
        return;
    }
    S->k += 1;
}

// nodal FP64 gradient -> 16-channel BF16 output gradient (channels 0 .. nd-1)
__global__ void k_net_dy_from_nodal(long nn, int nd, const double* __restrict__ g, const uint8_t* __restrict__ fix,
                                    bf16* __restrict__ dy) {
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        uint8_t f = fix[n];
        float v[16] = {0};
        for (int c = 0; c < nd; c++) v[c] = (f & (1u << c)) ? 0.f : (float)g[nd * n + c];
        for (int c = 0; c < 16; c++) dy[n * 16 + c] = f2bf(v[c]);
    }
}

// Smooth random displacement field for synthetic training pairs (K v, v):
// a sum over scales s = 2^l of bilinearly interpolated lattice noise of
// amplitude s (hash-based, seeded), zero on fixed DOFs.
__device__ inline double lattice_noise(uint64_t seed, int l, int I, int J, int c) {
    uint64_t z = seed ^ (0x9E3779B97F4A7C15ull * (uint64_t)(l + 1)) ^ ((uint64_t)(uint32_t)I << 21) ^
                 ((uint64_t)(uint32_t)J << 42) ^ (uint64_t)c;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

__global__ void k_random_field(int nx, int ny, uint64_t seed, int levels, const uint8_t* __restrict__ fix,
                               double* __restrict__ v) {
    const long nn = (long)(nx + 1) * (ny + 1);
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        const int i = (int)(n / (ny + 1)), j = (int)(n - (long)i * (ny + 1));
        const uint8_t f = fix[n];
        for (int c = 0; c < 2; c++) {
            double acc = 0.0;
            for (int l = 0; l < levels; l++) {
                const int sp = 1 << l;
                const int I = i / sp, J = j / sp;
                const double fi = (double)(i - I * sp) / sp, fj = (double)(j - J * sp) / sp;
                double a = lattice_noise(seed, l, I, J, c), b = lattice_noise(seed, l, I + 1, J, c);
                double cc = lattice_noise(seed, l, I, J + 1, c), d = lattice_noise(seed, l, I + 1, J + 1, c);
                acc += (double)sp * ((1 - fi) * ((1 - fj) * a + fj * cc) + fi * ((1 - fj) * b + fj * d));
            }
            v[2 * n + c] = (f & (1u << c)) ? 0.0 : acc;
        }
    }
}

// the random field of k_random_field on hex8 nodes: trilinear lattice noise
__global__ void k_random_field3(int nx, int ny, int nz, uint64_t seed, int levels, const uint8_t* __restrict__ fix,
                                double* __restrict__ v) {
    const long plane = (long)(ny + 1) * (nz + 1), nn = (long)(nx + 1) * plane;
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        const int i = (int)(n / plane);
        const long rem = n - (long)i * plane;
        const int j = (int)(rem / (nz + 1)), k = (int)(rem - (long)j * (nz + 1));
        const uint8_t f = fix[n];
        for (int c = 0; c < 3; c++) {
            double acc = 0.0;
            for (int l = 0; l < levels; l++) {
                const int sp = 1 << l;
                const int I = i / sp, J = j / sp, K = k / sp;
                const double fi = (double)(i - I * sp) / sp, fj = (double)(j - J * sp) / sp,
                             fk = (double)(k - K * sp) / sp;
                double val = 0.0;
                for (int a = 0; a < 2; a++)
                    for (int b = 0; b < 2; b++)
                        for (int cc = 0; cc < 2; cc++) {
                            const double w = (a ? fi : 1 - fi) * (b ? fj : 1 - fj) * (cc ? fk : 1 - fk);
                            // the lattice index packs (J, K) into the second coordinate
                            val += w * lattice_noise(seed, l, I + a, (J + b) * 65536 + (K + cc), c);
                        }
                acc += (double)sp * val;
            }
            v[3 * n + c] = (f & (1u << c)) ? 0.0 : acc;
        }
    }
}

// d = (r + s y) ./ D on free DOFs (0 on fixed), y = network output channels 0, 1
__global__ void k_net_output(long nn, const float* __restrict__ y, const double* __restrict__ r,
                             const double* __restrict__ D, const uint8_t* __restrict__ fix, double rs,
                             double* __restrict__ d) {
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        uint8_t f = fix[n];
        for (int c = 0; c < 2; c++) {
            double v = (r[2 * n + c] + rs * (double)y[n * 16 + c]) / D[2 * n + c];
            d[2 * n + c] = (f & (1u << c)) ? 0.0 : v;
        }
    }
}

// loss gradient wrt y: dy = s g ./ D on free DOFs, g = dL/dd
__global__ void k_net_output_bwd(long nn, const double* __restrict__ g, const double* __restrict__ D,
                                 const uint8_t* __restrict__ fix, double rs, bf16* __restrict__ dy) {
    for (long n = blockIdx.x * (long)blockDim.x + threadIdx.x; n < nn; n += (long)gridDim.x * blockDim.x) {
        uint8_t f = fix[n];
        float v[16] = {0};
        for (int c = 0; c < 2; c++) v[c] = (f & (1u << c)) ? 0.f : (float)(rs * g[2 * n + c] / D[2 * n + c]);
        for (int c = 0; c < 16; c++) dy[n * 16 + c] = f2bf(v[c]);
    }
}

__device__ inline void store_weight_bf16(int q, float w, int ntap, int cout, int cin, bf16* Wb, bf16* Wtb) {
    const int tap = q / (cout * cin), rem = q - tap * cout * cin, co = rem / cin, ci = rem - co * cin;
    const bf16 h = f2bf(w);
    Wb[q] = h;
    Wtb[((long)(ntap - 1 - tap) * cin + ci) * cout + co] = h;
}

// Wb[tap][co][ci] = bf16(W); Wtb[tap'][ci][co] = bf16(W[ntap - 1 - tap'][co][ci])
// (ntap = 9 or 27: reversing the tap index negates every offset)
__global__ void k_weights_bf16(int ntap, int cout, int cin, const float* __restrict__ W, bf16* __restrict__ Wb,
                               bf16* __restrict__ Wtb) {
    const int n = ntap * cout * cin;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        store_weight_bf16(q, W[q], ntap, cout, cin, Wb, Wtb);
    }
}

// Adam's step and the BF16 copies of the new weights, for every layer in one
// launch (blockIdx.y is the layer).  Bound by the launch: two launches per
// layer took 24 x 3.6 = 86 us per training step, this one about 6 us.
constexpr int kNetLayers = 12;
struct AdamLayers {
    struct {
        float *w, *m, *v;
        const float* grad;
        bf16 *Wb, *Wtb;
        int ntap, cout, cin;
    } l[kNetLayers];
};
__global__ void k_adam(AdamLayers P, float lr, float b1, float b2, float eps, float c1, float c2) {
    const auto& L = P.l[blockIdx.y];
    const int n = L.ntap * L.cout * L.cin;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        const float gq = L.grad[q];
        const float mq = b1 * L.m[q] + (1.f - b1) * gq;
        const float vq = b2 * L.v[q] + (1.f - b2) * gq * gq;
        const float w = L.w[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
        L.m[q] = mq;
        L.v[q] = vq;
        L.w[q] = w;
        store_weight_bf16(q, w, L.ntap, L.cout, L.cin, L.Wb, L.Wtb);
    }
}


// training pair (r, e) -> FP32 dataset slots
__global__ void k_pair_store(long n, const double* __restrict__ r, const double* __restrict__ e,
                             float* __restrict__ rout, float* __restrict__ eout) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        rout[i] = (float)r[i];
        eout[i] = (float)e[i];
    }
}

__global__ void k_d2f(long n, const double* __restrict__ a, float* __restrict__ b) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = (float)a[i];
}

__global__ void k_f2d(long n, const float* __restrict__ a, double* __restrict__ b) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = (double)a[i];
}

__global__ void k_sub_scale(long n, const double* __restrict__ a, const double* __restrict__ b, double s,
                            double* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = s * (a[i] - b[i]);
}

}  // namespace pf
