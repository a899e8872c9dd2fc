// denoise.hip — a small U-Net denoiser for the tracer's low-sample images,
// trained and run on gfx950 matrix cores (pt_dn_*). No counterpart in the
// reference.
//
// Network (NHWC BF16 activations, FP32 accumulation, FP32 master weights):
//   in  16 ch: log1p(XYZ) (3), albedo (3), normal (3), 1 / (1 + depth) (1), log1p(standard error) (1),
//              1 / sqrt(samples) (1), zeros (4)
//   e0: conv 16->32, conv 32->32                      (H x W)      skip0
//   e1: avgpool 2, conv 32->64, conv 64->64           (H/2)        skip1
//   b : avgpool 2, conv 64->128, conv 128->128        (H/4)
//   d1: upsample 2, conv [128 | skip1 64]->64, conv 64->64
//   d0: upsample 2, conv [64 | skip0 32]->32, conv 32->32
//   out: conv 32->16 (channels 0..2 used), no activation
// Every conv is 3x3, zero padding 1, bias, ReLU except the output. The output
// is a correction in log space: log1p(denoised XYZ) = log1p(input XYZ) + out.
// Loss: mean |log1p(denoised) - log1p(target)| over pixels and the 3 channels.
//
// Convolutions are implicit GEMMs on v_mfma_f32_32x32x16_bf16 (lane l holds
// A[row l % 32][k (l / 32) * 8 + i], B[k (l / 32) * 8 + i][col l % 32]; the
// 16 results of lane l are rows (v / 4) * 8 + (l / 32) * 4 + v % 4, column
// l % 32):
//   forward / backward-data: rows = pixels, columns = output channels,
//     K = 9 taps x input channels in steps of 16 (each lane reads 8
//     consecutive channels: 16 bytes of NHWC), both operands staged in LDS per
//     tile; backward-data runs the forward kernel on the output gradient with
//     the weights flipped and transposed;
//   backward-weights: rows = output channels, columns = input channels,
//     K = pixels; a block stages tiles of 4 x 32 pixels of both operands in LDS,
//     transposed, for all 9 taps, and writes its FP32 partial sums, which
//     k_grad_sum adds in order (into the gradient with atomics where there is
//     no memory for partials).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/pathtracer.h"
#include "tracer.hpp"

namespace ptdn {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned short u16;

constexpr int kIn = 16;      // input channels (12 used)
constexpr int kFeat = 12;    // floats per pixel of a feature image
constexpr int kOutC = 16;    // output channels (3 used)
constexpr int kThreads = 256;

__device__ __forceinline__ u16 f2bf(float x) {  // round to nearest even
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u16)0x7fc0;  // NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((uint32_t)h << 16); }

union Frag {
    uint4 u;
    bf8 v;
};
// A compile-time range of 32-channel output tiles [J0, J0 + N) (k_conv_t's epilogue).
template <int J0, int N>
struct SliceRange {
    static constexpr int j0 = J0, count = N;
};

// ---------------------------------------------------------------------------------
// Conv forward (also backward-data). X1 (C1 channels) and X2 (C2 channels, may
// be null) form the input [N, H, W, C1 + C2]; Wt is [9][Cout][C1 + C2] BF16;
// output channels [0, Co1) go to Y1 (Co1 channels) and [Co1, Cout) to Y2;
// bias and ReLU are applied at the store. `flip` reads tap 8 - t
// (backward-data).
// Pixel index of (n, y, x) of an H x W tensor (q), or with `up`, of the
// (H / 2) x (W / 2) tensor that a nearest-neighbour 2x upsample turns into it:
// the skip layers read their upsampled input this way instead of a stored copy.
__device__ __forceinline__ size_t up_index(int up, size_t q, int n, int y, int x, int H, int W) {
    return up ? ((size_t)n * (H >> 1) + (y >> 1)) * (W >> 1) + (x >> 1) : q;
}

struct ConvArgs {
    const u16* X1;
    const u16* X2;
    int C1, C2;
    const u16* Wt;
    const float* bias;  // null: none
    u16* Y1;
    u16* Y2;
    int Co1, Cout;
    int N, H, W;
    int relu;
    int flip;
    int tiles_per_block;  // consecutive pixel tiles a block computes in turn
    int up1;              // X1 is at half resolution, upsampled 2x (nearest) as it is read
    const u16* mask;      // null, or the activation (as Y1) whose ReLU the output goes back through
};

// The 8 BF16 values v where those of y are positive, else 0: the gradient through
// the ReLU that produced y.
__device__ __forceinline__ uint32_t relu_mask(uint32_t v, uint32_t y) {
    const uint32_t lo = (y & 0xffffu) - 1u < 0x7f80u ? 0xffffu : 0u, hi = (y >> 16) - 1u < 0x7f80u ? 0xffff0000u : 0u;
    return v & (lo | hi);
}
__device__ __forceinline__ uint4 relu_mask(uint4 v, uint4 y) {
    return make_uint4(relu_mask(v.x, y.x), relu_mask(v.y, y.y), relu_mask(v.z, y.z), relu_mask(v.w, y.w));
}

// ---------------------------------------------------------------------------------
// Conv forward (also backward-data), tiled: a block computes tiles of TH rows x
// 32 columns of one image's pixels x 32 * NC output channels. Per chunk of 32
// input channels it stages in LDS the (TH + 2) x 34 input tile around its
// pixels (zero outside the image) and the chunk's weights for all 9 taps; each
// wave then runs its TH / 4 pixel rows x NC channel tiles of 32 x 32 MFMAs over
// 9 taps x 2 steps of 16 channels with both operands read from LDS. Every input
// pixel is read from memory by about (TH + 2)(34) / (32 TH) tiles instead of
// once per tap. Pixels per 16-byte vector in LDS are padded to 40 channels so
// that 32 lanes reading 32 neighbouring pixels spread over the banks.
//
// Staging goes through registers: each thread issues all of its 16-byte loads
// of a chunk back to back (one wait for the lot), and the next chunk's loads
// are issued before the current chunk's MFMAs, so they are in flight while the
// matrix cores work. The 9 taps are unrolled, which lets the compiler issue the
// LDS reads of the next MFMAs ahead of the current ones.
//  - Several input chunks: a block computes one tile; its output goes through
//    the weight tile's LDS to 16-byte stores.
//  - One input chunk (ONE_CHUNK, Cin <= 32: the full-resolution layers whose
//    load, MFMAs and store would otherwise follow one another): a block
//    computes `tiles_per_block` consecutive tiles (along x first) with the
//    weights staged once; the next tile's input loads are in flight under the
//    current tile's MFMAs and output stores, and the output goes through the
//    input tile's LDS, 32 channels at a time.
// Register budget: the LDS tiles allow 2 blocks per CU at NC = 2 (73 KB each)
// and 3 at NC = 1 (50 KB), so the launch bounds ask for that many waves per SIMD.
template <int NC, int TH, bool ONE_CHUNK>
__global__ void __launch_bounds__(kThreads, NC == 2 ? 2 : 3) k_conv_t(ConvArgs a) {
    constexpr int CK = 32, CKP = CK + 8;  // channels per chunk; LDS pitch per pixel / weight row
    constexpr int TW = 32, IW = TW + 2, IH = TH + 2;
    constexpr int R = TH / 4;             // pixel rows per wave
    constexpr int NXV = IH * IW * (CK / 8), NWV = 9 * 32 * NC * (CK / 8);  // 16-byte vectors per chunk
    constexpr int NXT = (NXV + kThreads - 1) / kThreads, NWT = (NWV + kThreads - 1) / kThreads;
    __shared__ __align__(16) u16 s_x[IH * IW * CKP];
    __shared__ __align__(16) u16 s_w[9 * 32 * NC * CKP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tiles_x = (a.W + TW - 1) / TW, tiles_y = (a.H + TH - 1) / TH;
    const int co0 = blockIdx.y * 32 * NC;
    const int Cin = a.C1 + a.C2;
    const int kq = (lane >> 5) * 8;  // this lane's 8 channels within a 16-channel step
    const int col = lane & 31;
    f16v acc[R][NC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < NC; ++j) acc[r][j] = f16v{};
    float bias[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const int co = co0 + j * 32 + col;
        bias[j] = a.bias && co < a.Cout ? a.bias[co] : 0.0f;
    }
    // tile -> image n and the tile's first pixel (x0, y0)
    auto origin = [&](int tile, int& n, int& x0, int& y0) {
        x0 = (tile % tiles_x) * TW;
        const int rest = tile / tiles_x;
        y0 = (rest % tiles_y) * TH;
        n = rest / tiles_y;
    };
    uint4 xr[NXT], wr[NWT];
    // this thread's share of a chunk: input vectors i = threadIdx.x + u * kThreads
    // (pixel i / 4 of the halo tile, channels 8 (i % 4) ..), weight vectors likewise
    // (tap, output row, 8 channels)
    auto fetch_x = [&](int n, int x0, int y0, int c0) {
#pragma unroll
        for (int u = 0; u < NXT; ++u) {
            const int i = threadIdx.x + u * kThreads;
            const int v = i % (CK / 8), pix = i / (CK / 8);
            const int y = y0 + pix / IW - 1, x = x0 + pix % IW - 1;
            const int c = c0 + v * 8;
            uint4 val = make_uint4(0, 0, 0, 0);
            if (i < NXV && y >= 0 && y < a.H && x >= 0 && x < a.W && c < Cin) {
                const size_t q = ((size_t)n * a.H + y) * a.W + x;
                const u16* src = c < a.C1 ? a.X1 + up_index(a.up1, q, n, y, x, a.H, a.W) * a.C1 + c
                                          : a.X2 + q * a.C2 + (c - a.C1);
                val = *reinterpret_cast<const uint4*>(src);
            }
            xr[u] = val;
        }
    };
    auto fetch_w = [&](int c0) {
#pragma unroll
        for (int u = 0; u < NWT; ++u) {
            const int i = threadIdx.x + u * kThreads;
            const int v = i % (CK / 8), row = (i / (CK / 8)) % (32 * NC), t = i / ((CK / 8) * 32 * NC);
            const int tt = a.flip ? 8 - t : t;
            const int co = co0 + row, c = c0 + v * 8;
            uint4 val = make_uint4(0, 0, 0, 0);
            if (i < NWV && co < a.Cout && c < Cin)
                val = *reinterpret_cast<const uint4*>(a.Wt + ((size_t)tt * a.Cout + co) * Cin + c);
            wr[u] = val;
        }
    };
    auto put_x = [&]() {
#pragma unroll
        for (int u = 0; u < NXT; ++u) {
            const int i = threadIdx.x + u * kThreads;
            if (i < NXV) *reinterpret_cast<uint4*>(&s_x[(i / (CK / 8)) * CKP + (i % (CK / 8)) * 8]) = xr[u];
        }
    };
    auto put_w = [&]() {
#pragma unroll
        for (int u = 0; u < NWT; ++u) {
            const int i = threadIdx.x + u * kThreads;
            if (i < NWV) *reinterpret_cast<uint4*>(&s_w[(i / (CK / 8)) * CKP + (i % (CK / 8)) * 8]) = wr[u];
        }
    };
    // the MFMAs of the chunk at c0 staged in LDS
    auto mma = [&](int c0) {
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int dy = t / 3, dx = t % 3;  // offsets into the halo-padded tile
#pragma unroll
            for (int k = 0; k < CK; k += 16) {
                if (c0 + k >= Cin) break;  // a 16-channel input's second step is all zeros
                Frag A[R];
#pragma unroll
                for (int r = 0; r < R; ++r)
                    A[r].u = *reinterpret_cast<const uint4*>(&s_x[((wave * R + r + dy) * IW + col + dx) * CKP + k + kq]);
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    Frag B;
                    B.u = *reinterpret_cast<const uint4*>(&s_w[(t * 32 * NC + j * 32 + col) * CKP + k + kq]);
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[r].v, B.v, acc[r][j], 0, 0, 0);
                }
            }
        }
    };
    // Output channels [j0, j0 + 32 J) of the tile at (n, x0, y0) staged in s_o
    // (pitch OP per pixel): bias, ReLU and BF16 rounding per accumulator into LDS
    // in pixel-major order, then 16-byte vectors of 8 channels to memory (the
    // tensors' channel counts and the Y1 / Y2 split are multiples of 8), one
    // bounds check per vector. The caller synchronises before (LDS free) and
    // after (LDS read) it.
    auto store_slices = [&](u16* s_o, auto jc, int n, int x0, int y0) {
        constexpr int J0 = decltype(jc)::j0, J = decltype(jc)::count, OP = 32 * J + 8;
#pragma unroll
        for (int jj = 0; jj < J; ++jj) {
            const int j = J0 + jj;
            const int co = co0 + j * 32 + col;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int row = wave * R + r;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int px = (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
                    float o = acc[r][j][v] + bias[j];
                    if (a.relu) o = fmaxf(o, 0.0f);
                    s_o[(row * TW + px) * OP + jj * 32 + col] = co < a.Cout ? f2bf(o) : (u16)0;
                }
            }
        }
        __syncthreads();
        constexpr int VPP = 32 * J / 8;  // 16-byte vectors per pixel
#pragma unroll
        for (int u = 0; u < (TH * TW * VPP) / kThreads; ++u) {
            const int i = threadIdx.x + u * kThreads;
            const int g = i % VPP, pix = i / VPP;
            const int y = y0 + pix / TW, x = x0 + pix % TW, c = co0 + J0 * 32 + g * 8;
            if (y >= a.H || x >= a.W || c >= a.Cout) continue;
            uint4 val = *reinterpret_cast<const uint4*>(&s_o[pix * OP + g * 8]);
            const size_t p = ((size_t)n * a.H + y) * a.W + x;
            if (a.mask) val = relu_mask(val, *reinterpret_cast<const uint4*>(a.mask + p * a.Co1 + c));
            u16* dst = c < a.Co1 ? a.Y1 + p * a.Co1 + c : a.Y2 + p * (a.Cout - a.Co1) + (c - a.Co1);
            *reinterpret_cast<uint4*>(dst) = val;
        }
    };
    if constexpr (!ONE_CHUNK) {
        int n, x0, y0;
        origin(blockIdx.x, n, x0, y0);
        fetch_x(n, x0, y0, 0);
        fetch_w(0);
#pragma unroll 1
        for (int c0 = 0; c0 < Cin; c0 += CK) {
            __syncthreads();  // every wave is done with the previous chunk's tiles
            put_x();
            put_w();
            __syncthreads();
            if (c0 + CK < Cin) {
                fetch_x(n, x0, y0, c0 + CK);
                fetch_w(c0 + CK);
            }
            mma(c0);
        }
        static_assert(TH * TW * (32 * NC + 8) <= 9 * 32 * NC * CKP, "the output tile must fit the weight tile's LDS");
        __syncthreads();  // every wave is done with the last chunk's tiles
        store_slices(s_w, SliceRange<0, NC>{}, n, x0, y0);
    } else {
        static_assert(TH * TW * (32 + 8) <= IH * IW * CKP, "an output slice must fit the input tile's LDS");
        const int ntiles = a.N * tiles_x * tiles_y;
        const int t_begin = blockIdx.x * a.tiles_per_block;
        const int t_count = min(a.tiles_per_block, ntiles - t_begin);
        int n, x0, y0;
        origin(t_begin, n, x0, y0);
        fetch_x(n, x0, y0, 0);
        fetch_w(0);
#pragma unroll 1
        for (int k = 0; k < t_count; ++k) {
            __syncthreads();  // every wave is done with the previous tile's output
            put_x();
            if (k == 0) put_w();
            __syncthreads();
            int n1 = n, x1 = x0, y1 = y0;
            if (k + 1 < t_count) {
                origin(t_begin + k + 1, n1, x1, y1);
                fetch_x(n1, x1, y1, 0);
            }
            mma(0);
            __syncthreads();  // every wave is done with the input tile
            store_slices(s_x, SliceRange<0, 1>{}, n, x0, y0);
            if constexpr (NC == 2) {
                __syncthreads();
                store_slices(s_x, SliceRange<1, 1>{}, n, x0, y0);
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int j = 0; j < NC; ++j) acc[r][j] = f16v{};
            n = n1;
            x0 = x1;
            y0 = y1;
        }
    }
}

// ---------------------------------------------------------------------------------
// Conv backward-weights: dW[t][co][ci] = sum over pixels of dZ[p][co] * X[p + tap t][ci],
// dbias[co] = sum of dZ[p][co]. Grid: x = pixel tiles of kWR rows x 32 columns, taken
// in turn by a block, y = co tiles of 32, z = ci tiles of 32. The blocks of one x write
// their sums to partial x (k_grad_sum adds the partials in order, so a gradient does
// not depend on the order in which blocks end), or add them to the cleared gradient
// with FP32 atomics when there is no memory for partials.
struct WgradArgs {
    const u16* dZ;
    int Cout;
    const u16* X1;
    const u16* X2;
    int C1, C2;
    float* g;     // the layer's gradient: [9][Cout][C1 + C2], then [Cout]
    float* part;  // gridDim.x copies of it, or null
    int N, H, W;
    int up1;      // X1 at half resolution, as in ConvArgs
};
constexpr int kWR = 4;          // pixel rows of a tile
constexpr int kWThreads = 192;  // three waves, one per row of taps

// Pixels are the K dimension, so both MFMA operands are read transposed: a tile's dZ
// and X (with its halo) go into LDS channel-major, pairs of neighbouring pixels per
// 4-byte write, and all 9 taps run from the staged tile, each wave one row of taps: per
// 16 pixels one 16-byte read of dZ and one of X with the pixel pairs beside it, from
// which the left and right taps' 8 pixels are funnel-shifted, for 3 MFMAs. (The kernel
// before staged both operands again for each tap and gathered them element by element;
// X staged once per column offset instead of shifted took 398 us for the 11 layers.)
// The next tile's loads are in flight under the MFMAs. LDS rows are 4 modulo 16 dwords
// apart, so that 16 rows read in turn hit different banks. All 11 layers of a step, us
// before and after with the partials' sum: 8 crops of 96 x 96 315 -> 215, 16 of 128 x 128
// 651 -> 390, one of 32 x 32 77 -> 115 (its launches' latency; the step is shorter all the
// same). Bound by the chain of a tile: loads, transposing writes, 24 MFMAs per wave.
__global__ void __launch_bounds__(kWThreads) k_conv_wgrad(WgradArgs a) {
    constexpr int ZP = kWR * 32 + 8;                    // row: kWR x 32 pixels
    constexpr int XR = 48, XP = (kWR + 2) * XR + 8;     // row: kWR + 2 lines of pixels -8 .. 39 (-2 .. 33 used)
    constexpr int NZ = kWR * 16 * 4, NX = (kWR + 2) * 18 * 4;  // staging tasks: line, pixel pair, 8 channels
    constexpr int NZT = (NZ + kWThreads - 1) / kWThreads, NXT = (NX + kWThreads - 1) / kWThreads;
    __shared__ __align__(16) u16 s_z[32 * ZP];
    __shared__ __align__(16) u16 s_x[32 * XP];
    const int lane = threadIdx.x & 63, dy = threadIdx.x >> 6;
    const int Cin = a.C1 + a.C2;
    const int co0 = blockIdx.y * 32, ci0 = blockIdx.z * 32;
    const int tiles_x = (a.W + 31) / 32, tiles_y = (a.H + kWR - 1) / kWR, ntiles = a.N * tiles_y * tiles_x;
    const bool bias = ci0 == 0 && dy == 1;
    f16v acc[3] = {f16v{}, f16v{}, f16v{}}, accb = f16v{};
    Frag one;
    one.u = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);  // BF16 ones
    uint4 zr[NZT][2], xr[NXT][2];
    auto fetch = [&](int tile) {
        const int x0 = (tile % tiles_x) * 32, rest = tile / tiles_x;
        const int y0 = (rest % tiles_y) * kWR, n = rest / tiles_y;
#pragma unroll
        for (int u = 0; u < NZT; ++u) {
            const int i = threadIdx.x + u * kWThreads;
            const int g = i & 3, px = (i >> 2) & 15, y = y0 + (i >> 6), x = x0 + 2 * px, c = co0 + g * 8;
#pragma unroll
            for (int k = 0; k < 2; ++k)
                zr[u][k] = i < NZ && y < a.H && x + k < a.W && c < a.Cout
                               ? *reinterpret_cast<const uint4*>(a.dZ + (((size_t)n * a.H + y) * a.W + x + k) * a.Cout + c)
                               : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < NXT; ++u) {
            const int i = threadIdx.x + u * kWThreads;
            const int g = i & 3, px = (i >> 2) % 18, y = y0 + (i >> 2) / 18 - 1, c = ci0 + g * 8;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int x = x0 + 2 * px - 2 + k;
                uint4 val = make_uint4(0, 0, 0, 0);
                if (i < NX && y >= 0 && y < a.H && x >= 0 && x < a.W && c < Cin) {
                    const size_t q = ((size_t)n * a.H + y) * a.W + x;
                    const u16* src = c < a.C1 ? a.X1 + up_index(a.up1, q, n, y, x, a.H, a.W) * a.C1 + c
                                              : a.X2 + q * a.C2 + (c - a.C1);
                    val = *reinterpret_cast<const uint4*>(src);
                }
                xr[u][k] = val;
            }
        }
    };
    // channels 8 g .. 8 g + 7 of a pixel pair into rows 8 g .. of dst at `at`
    auto put = [](u16* dst, int pitch, int g, int at, uint4 p0, uint4 p1) {
        const uint32_t u[4] = {p0.x, p0.y, p0.z, p0.w}, v[4] = {p1.x, p1.y, p1.z, p1.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            *reinterpret_cast<uint32_t*>(&dst[(g * 8 + 2 * k) * pitch + at]) = (u[k] & 0xffffu) | (v[k] << 16);
            *reinterpret_cast<uint32_t*>(&dst[(g * 8 + 2 * k + 1) * pitch + at]) = (u[k] >> 16) | (v[k] & 0xffff0000u);
        }
    };
    const int row = lane & 31, kq = (lane >> 5) * 8;
    if ((int)blockIdx.x < ntiles) fetch(blockIdx.x);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        __syncthreads();  // every wave is done with the previous tile
#pragma unroll
        for (int u = 0; u < NZT; ++u) {
            const int i = threadIdx.x + u * kWThreads;
            if (i < NZ) put(s_z, ZP, i & 3, (i >> 6) * 32 + 2 * ((i >> 2) & 15), zr[u][0], zr[u][1]);
        }
#pragma unroll
        for (int u = 0; u < NXT; ++u) {
            const int i = threadIdx.x + u * kWThreads;
            if (i < NX) put(s_x, XP, i & 3, (i >> 2) / 18 * XR + 2 * ((i >> 2) % 18) + 6, xr[u][0], xr[u][1]);
        }
        __syncthreads();
        if (tile + (int)gridDim.x < ntiles) fetch(tile + gridDim.x);
#pragma unroll
        for (int r = 0; r < kWR; ++r) {
#pragma unroll
            for (int k = 0; k < 32; k += 16) {
                Frag A, L, C, R;
                A.u = *reinterpret_cast<const uint4*>(&s_z[row * ZP + r * 32 + k + kq]);
                const u16* xp = &s_x[row * XP + (r + dy) * XR + 8 + k + kq];
                C.u = *reinterpret_cast<const uint4*>(xp);
                const uint32_t before = *reinterpret_cast<const uint32_t*>(xp - 2);
                const uint32_t after = *reinterpret_cast<const uint32_t*>(xp + 8);
                // 8 pixels from one to the left and one to the right
                auto shift = [](uint32_t lo, uint32_t hi) { return __builtin_amdgcn_alignbit(hi, lo, 16); };
                L.u = make_uint4(shift(before, C.u.x), shift(C.u.x, C.u.y), shift(C.u.y, C.u.z), shift(C.u.z, C.u.w));
                R.u = make_uint4(shift(C.u.x, C.u.y), shift(C.u.y, C.u.z), shift(C.u.z, C.u.w), shift(C.u.w, after));
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v, L.v, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v, C.v, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v, R.v, acc[2], 0, 0, 0);
                if (bias) accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v, one.v, accb, 0, 0, 0);
            }
        }
    }
    const int nw = 9 * a.Cout * Cin;
    float* part = a.part ? a.part + (size_t)blockIdx.x * (nw + a.Cout) : nullptr;
    auto sink = [&](int j, float v) {
        if (part) part[j] = v;
        else if (v != 0.0f) atomicAdd(&a.g[j], v);
    };
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int co = co0 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3), ci = ci0 + (lane & 31);
        if (co >= a.Cout) continue;
        if (ci < Cin) {
#pragma unroll
            for (int s = 0; s < 3; ++s) sink(((dy * 3 + s) * a.Cout + co) * Cin + ci, acc[s][v]);
        }
        if (bias && (lane & 31) == 0) sink(nw + co, accb[v]);
    }
}

// ---------------------------------------------------------------------------------
// Elementwise kernels (NHWC BF16). Pooling and upsampling move 8 channels (one
// 16-byte vector) per thread: C is a multiple of 8, and the tensors hold fewer
// than 2^31 such groups (the denoiser's size limits), so index arithmetic is
// 32-bit. Each channel's arithmetic is the one-channel formula, in the same order.
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t bf_pack(float lo, float hi) {
    return (uint32_t)f2bf(lo) | ((uint32_t)f2bf(hi) << 16);
}
// per channel: scale * (((a + b) + c) + d)
__device__ __forceinline__ uint32_t sum4(uint32_t a, uint32_t b, uint32_t c, uint32_t d, float scale) {
    return bf_pack(scale * (((bf_lo(a) + bf_lo(b)) + bf_lo(c)) + bf_lo(d)),
                   scale * (((bf_hi(a) + bf_hi(b)) + bf_hi(c)) + bf_hi(d)));
}
__device__ __forceinline__ uint4 sum4(uint4 a, uint4 b, uint4 c, uint4 d, float scale) {
    return make_uint4(sum4(a.x, b.x, c.x, d.x, scale), sum4(a.y, b.y, c.y, d.y, scale),
                      sum4(a.z, b.z, c.z, d.z, scale), sum4(a.w, b.w, c.w, d.w, scale));
}
__device__ __forceinline__ uint32_t scale2(uint32_t a, float scale) {
    return bf_pack(scale * bf_lo(a), scale * bf_hi(a));
}

__global__ void k_pool2(const u16* x, u16* y, int N, int H, int W, int C) {  // 2x2 average
    const uint32_t Ho = H / 2, Wo = W / 2, C8 = C >> 3;
    const uint32_t n = (uint32_t)N * Ho * Wo * C8;
    const uint4* xv = reinterpret_cast<const uint4*>(x);
    uint4* yv = reinterpret_cast<uint4*>(y);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t g = i % C8, r = i / C8;
        const uint32_t xo = r % Wo, r2 = r / Wo;
        const uint32_t yo = r2 % Ho, b = r2 / Ho;
        const uint32_t q = (b * (uint32_t)H + 2 * yo) * (uint32_t)W + 2 * xo;
        yv[i] = sum4(xv[q * C8 + g], xv[(q + 1) * C8 + g], xv[(q + W) * C8 + g], xv[(q + W + 1) * C8 + g], 0.25f);
    }
}
__device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b) {
    return bf_pack(bf_lo(a) + bf_lo(b), bf_hi(a) + bf_hi(b));
}
// dZ of an encoder level's output y: the gradient of its 2x2 average (0.25 dY) plus
// the skip connection's `add`, through the ReLU that produced y (in one pass; they
// were two kernels with the sum's first term stored in between, rounded as here).
__global__ void k_pool2_bwd(const u16* dy, const u16* add, const u16* y, u16* dz, int N, int H, int W, int C) {
    const uint32_t C8 = C >> 3;
    const uint32_t n = (uint32_t)N * H * W * C8;
    const uint4* dyv = reinterpret_cast<const uint4*>(dy);
    const uint4* addv = reinterpret_cast<const uint4*>(add);
    const uint4* yv = reinterpret_cast<const uint4*>(y);
    uint4* dzv = reinterpret_cast<uint4*>(dz);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t g = i % C8, r = i / C8;
        const uint32_t x = r % W, r2 = r / W;
        const uint32_t yy = r2 % H, b = r2 / H;
        const uint4 v = dyv[((b * (uint32_t)(H / 2) + yy / 2) * (uint32_t)(W / 2) + x / 2) * C8 + g], s = addv[i];
        const uint4 sum = make_uint4(add2(scale2(v.x, 0.25f), s.x), add2(scale2(v.y, 0.25f), s.y),
                                     add2(scale2(v.z, 0.25f), s.z), add2(scale2(v.w, 0.25f), s.w));
        dzv[i] = relu_mask(sum, yv[i]);
    }
}
// dZ of a decoder level's output y: the gradient of the nearest 2x upsample the skip
// layers apply to it as they read it (up_index; the sum of the 4 dY it fed), through
// the ReLU that produced y.
__global__ void k_up2_bwd(const u16* dy, const u16* y, u16* dz, int N, int H, int W, int C) {
    const uint32_t C8 = C >> 3;
    const uint32_t n = (uint32_t)N * H * W * C8;
    const uint4* dyv = reinterpret_cast<const uint4*>(dy);
    const uint4* yv = reinterpret_cast<const uint4*>(y);
    uint4* dzv = reinterpret_cast<uint4*>(dz);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t g = i % C8, r = i / C8;
        const uint32_t x = r % W, r2 = r / W;
        const uint32_t yy = r2 % H, b = r2 / H;
        const uint32_t q = (b * 2 * (uint32_t)H + 2 * yy) * 2 * (uint32_t)W + 2 * x;
        dzv[i] = relu_mask(sum4(dyv[q * C8 + g], dyv[(q + 1) * C8 + g], dyv[(q + 2 * W) * C8 + g],
                                dyv[(q + 2 * W + 1) * C8 + g], 1.0f), yv[i]);
    }
}
// features (N, H, W, 12) FP32 -> input tensor (16 channels BF16), a pixel per thread in
// 16-byte vectors; before a backward pass also clears the nz floats at `zero` (the
// gradients and, after them, the loss).
__global__ void k_prep(const float* f, u16* x, size_t P, float* zero, size_t nz) {
    for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
        const float4* s = reinterpret_cast<const float4*>(f + p * kFeat);
        const float4 a = s[0], b = s[1], c = s[2];
        auto log_in = [](float v) { return f2bf(log1pf(fmaxf(v, 0.0f))); };
        auto pair = [](u16 lo, u16 hi) { return (uint32_t)lo | ((uint32_t)hi << 16); };
        uint4* d = reinterpret_cast<uint4*>(x + p * kIn);
        d[0] = make_uint4(pair(log_in(a.x), log_in(a.y)), pair(log_in(a.z), f2bf(a.w)), bf_pack(b.x, b.y),
                          bf_pack(b.z, b.w));
        d[1] = make_uint4(pair(f2bf(c.x), f2bf(1.0f / (1.0f + fmaxf(c.y, 0.0f)))),
                          pair(log_in(c.z), f2bf(rsqrtf(fmaxf(c.w, 1.0f)))), 0u, 0u);
    }
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < nz; i += (size_t)gridDim.x * blockDim.x)
        zero[i] = 0.0f;
}
// prediction z = log1p(denoised) = log1p(in) + out[0..2]; loss and its
// gradient with respect to z, mean over 3P values: |z - log1p(target)|
// (l2 == 0) or (expm1(z) - target)^2 (l2 == 1); also the denoised image
// max(expm1(z), 0). The loss takes one atomic per block: one per wave (1152 on one
// address for 8 crops of 96 x 96, 12 ns each) was most of the kernel's 24 us.
__global__ void __launch_bounds__(kThreads) k_head(const float* f, const u16* out, const float* target, float* denoised,
                                                   u16* dout, float* loss, size_t P, int l2) {
    __shared__ float s_l[kThreads / 64];
    float l = 0.0f;
    const float inv = 1.0f / (3.0f * (float)P);
    for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
        const float4 in = *reinterpret_cast<const float4*>(f + p * kFeat);
        const uint2 o = *reinterpret_cast<const uint2*>(out + p * kOutC);
        const float xin[3] = {in.x, in.y, in.z}, res[3] = {bf_lo(o.x), bf_hi(o.x), bf_lo(o.y)};
        u16 dz[3] = {0, 0, 0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float z = log1pf(fmaxf(xin[c], 0.0f)) + res[c];
            if (denoised) denoised[p * 3 + c] = fmaxf(expm1f(z), 0.0f);
            if (target && l2) {
                const float y = expm1f(z), d = y - fmaxf(target[p * 3 + c], 0.0f);
                l += d * d;
                dz[c] = f2bf(2.0f * d * (y + 1.0f) * inv);
            } else if (target) {
                const float d = z - log1pf(fmaxf(target[p * 3 + c], 0.0f));
                l += fabsf(d);
                dz[c] = f2bf(d > 0.0f ? inv : (d < 0.0f ? -inv : 0.0f));
            }
        }
        if (dout) {
            uint4* dv = reinterpret_cast<uint4*>(dout + p * kOutC);
            dv[0] = make_uint4((uint32_t)dz[0] | ((uint32_t)dz[1] << 16), (uint32_t)dz[2], 0u, 0u);
            dv[1] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    if (loss) {
        for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off);
        if ((threadIdx.x & 63) == 0) s_l[threadIdx.x >> 6] = l;
        __syncthreads();
        if (threadIdx.x == 0) {
            float t = 0.0f;
            for (int w = 0; w < kThreads / 64; ++w) t += s_l[w];
            if (t != 0.0f) atomicAdd(loss, t * inv);
        }
    }
}
// A layer's parameters: FP32 masters at w (weights [9][Cout][Cin], then Cout biases),
// and their BF16 copies: forward Wf[t][co][ci] and backward-data Wb[t][ci][co]
// (k_conv_t with `flip` reads tap 8 - t: the gradient of tap t's offset o is gathered
// from offset -o, which is tap 8 - t).
struct LayerParams {
    uint32_t off, cout, cin;
    u16 *wf, *wb;
};
constexpr int kLayers = 11;
struct AllParams {
    LayerParams l[kLayers];
};
// The gradients from k_conv_wgrad's partials, one launch for the network: blockIdx.y is
// the layer, a block adds 32 parameters' partials in 8 slices and the slices in order.
struct PartialSums {
    struct {
        const float* part;
        uint32_t off, n, count;  // first parameter, parameters, partials
    } l[kLayers];
};
__global__ void __launch_bounds__(kThreads) k_grad_sum(PartialSums A, float* g) {
    __shared__ float s_p[8][32];
    const auto l = A.l[blockIdx.y];
    const uint32_t j = blockIdx.x * 32 + (threadIdx.x & 31), slice = threadIdx.x >> 5;
    if (blockIdx.x * 32 >= l.n) return;  // the whole block
    float t = 0.0f;
    if (j < l.n) {
        const uint32_t per = (l.count + 7) / 8, b0 = slice * per, b1 = min(b0 + per, l.count);
#pragma unroll 8
        for (uint32_t b = b0; b < b1; ++b) t += l.part[(size_t)b * l.n + j];
    }
    s_p[slice][threadIdx.x & 31] = t;
    __syncthreads();
    if (slice == 0 && j < l.n) {
        for (int k = 1; k < 8; ++k) t += s_p[k][threadIdx.x];
        g[l.off + j] = t;
    }
}

struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
};
// Adam on the FP32 masters (ADAM), then their BF16 copies; blockIdx.y is the layer. One
// launch for the network, where Adam and a copy kernel per layer were twelve of 6 us.
template <bool ADAM>
__global__ void k_params(AllParams A, float* w, const float* g, float* m, float* v, AdamArgs h) {
    const LayerParams l = A.l[blockIdx.y];
    const uint32_t nw = 9 * l.cout * l.cin, n = nw + l.cout;
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t i = l.off + j;
        float x = w[i];
        if (ADAM) {
            const float gi = g[i];
            const float mi = h.b1 * m[i] + (1.0f - h.b1) * gi;
            const float vi = h.b2 * v[i] + (1.0f - h.b2) * gi * gi;
            m[i] = mi;
            v[i] = vi;
            x -= h.lr * (mi / h.c1) / (sqrtf(vi / h.c2) + h.eps);
            w[i] = x;
        }
        if (j < nw) {
            const uint32_t ci = j % l.cin, r = j / l.cin, co = r % l.cout, t = r / l.cout;
            const u16 b = f2bf(x);
            l.wf[j] = b;
            l.wb[(t * l.cin + ci) * l.cout + co] = b;
        }
    }
}

// ---------------------------------------------------------------------------------
// Served requests: feature images assembled from a request's per-pixel moments
// and its first-hit features, and the error sums of the dual-buffer estimate.

// which: 0 all samples, 1 the even-index half, 2 the odd-index half. XYZ and
// the standard error of Y in texel units times inv_scale; the standard error
// of a half uses the sample variance of all samples.
__global__ void k_dn_assemble(ptk::DnRequest q, int which, float inv_scale, float* feat) {
    const int P = q.W * q.H;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += gridDim.x * blockDim.x) {
        const int n = q.nsamp[p], no = q.n_odd[p];
        const int cnt = which == 0 ? n : (which == 1 ? n - no : no);
        float* f = feat + (size_t)p * kFeat;
        const float k = cnt > 0 ? q.exposure * inv_scale / (float)cnt : 0.0f;
        for (int c = 0; c < 3; ++c) {
            const float s = q.sum[c * P + p], so = q.sum_odd[c * P + p];
            f[c] = (which == 0 ? s : (which == 1 ? s - so : so)) * k;
        }
        float var = 0.0f;
        if (n > 1) {
            const float s1 = q.sum[P + p], s2 = q.sumsq[P + p];
            var = fmaxf(s2 - s1 * (s1 / (float)n), 0.0f) / (float)(n - 1);
        }
        f[10] = cnt > 0 ? sqrtf(var / (float)cnt) * q.exposure * inv_scale : 0.0f;
        f[11] = (float)cnt;
        const int na = q.aov_n[p];
        const float ka = na > 0 ? 1.0f / (float)na : 0.0f;
        for (int c = 3; c < 10; ++c) f[c] = q.aov[(size_t)p * kFeat + c] * ka;
    }
}

// Against the other half (other: 1 even, 2 odd) of the same request, per block
// then one double atomic per block into line blockIdx.x % 64 (stride 32):
// slot 0 sum (den - other)^2, slot 1 sum of the other half's variance of the
// mean, slot 2 sum of the full mean^2, slot 3 sum (den - prev)^2 when prev
// (the other half's denoised image) is given; all over pixels and XYZ in
// texel units times inv_scale.
__global__ void k_dn_cross(ptk::DnRequest q, const float* den, const float* prev, int other, float inv_scale,
                           double* lines) {
    __shared__ double red[4][4];
    const int P = q.W * q.H;
    double e = 0.0, v = 0.0, m = 0.0, dd = 0.0;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += gridDim.x * blockDim.x) {
        const int n = q.nsamp[p], no = q.n_odd[p];
        const int cnt = other == 1 ? n - no : no;
        if (cnt < 1 || n < 2) continue;
        const double k = (double)q.exposure * inv_scale;
        for (int c = 0; c < 3; ++c) {
            const double s = q.sum[c * P + p], so = q.sum_odd[c * P + p], s2 = q.sumsq[c * P + p];
            const double o = (other == 1 ? s - so : so) / cnt * k;
            const double d = (double)den[(size_t)p * 3 + c] - o;
            e += d * d;
            const double var = fmax(s2 - s * (s / n), 0.0) / (double)(n - 1);
            v += var / cnt * k * k;
            const double mean = s / n * k;
            m += mean * mean;
            if (prev) {
                const double g = (double)den[(size_t)p * 3 + c] - (double)prev[(size_t)p * 3 + c];
                dd += g * g;
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        e += __shfl_down(e, off);
        v += __shfl_down(v, off);
        m += __shfl_down(m, off);
        dd += __shfl_down(dd, off);
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[0][wv] = e; red[1][wv] = v; red[2][wv] = m; red[3][wv] = dd; }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += red[threadIdx.x][i];
        atomicAdd(lines + (size_t)(blockIdx.x % 64) * 32 + threadIdx.x, t);
    }
}

__global__ void k_dn_scale(const float* den, float scale, float* out, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) out[i] = den[i] * scale;
}

// ---------------------------------------------------------------------------------
// Host side.
struct Layer {
    int cin1, cin2, cout;  // input split (concat), output channels
    bool relu;
    bool up1;              // the first input is the half-resolution decoder tensor, upsampled as it is read
    size_t w_off, b_off;   // into the FP32 parameter vector
    u16 *wf = nullptr, *wb = nullptr;
};

}  // namespace ptdn

using namespace ptdn;

struct pt_denoiser {
    pt_ctx* ctx = nullptr;
    int cus = 256;  // compute units of the context's device
    int maxN = 0, maxH = 0, maxW = 0;
    std::vector<Layer> L;
    size_t nparam = 0;
    int64_t step = 0;
    int loss_kind = PT_DN_LOSS_L1_LOG;
    DevAlloc mem;
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    u16* wbf = nullptr;  // BF16 copies, 2 per weight
    // activations (BF16) and gradients
    u16 *x0 = nullptr, *e0a = nullptr, *e0 = nullptr, *p1 = nullptr, *e1a = nullptr, *e1 = nullptr, *p2 = nullptr,
        *ba = nullptr, *bb = nullptr, *d1a = nullptr, *d1 = nullptr, *d0a = nullptr, *d0 = nullptr, *out = nullptr;
    u16 *ga = nullptr, *gb = nullptr, *gc = nullptr, *gs1 = nullptr, *gs0 = nullptr;  // gradient scratch
    float *feat = nullptr, *tgt = nullptr, *den = nullptr, *loss = nullptr;
    std::string err;
};

namespace {

int dn_fail(pt_denoiser* d, int st, const std::string& msg) {
    d->err = msg;
    return st;
}

void conv(pt_denoiser* d, const Layer& l, const u16* x1, const u16* x2, u16* y, int N, int H, int W, bool bwd_data,
          u16* y2 = nullptr, int co1 = 0, const u16* mask = nullptr) {
    ConvArgs a{};
    a.N = N;
    a.H = H;
    a.W = W;
    if (!bwd_data) {
        a.X1 = x1; a.X2 = x2; a.C1 = l.cin1; a.C2 = l.cin2;
        a.up1 = l.up1 ? 1 : 0;
        a.Wt = l.wf; a.bias = d->w + l.b_off;
        a.Y1 = y; a.Y2 = nullptr; a.Co1 = l.cout; a.Cout = l.cout;
        a.relu = l.relu; a.flip = 0;
    } else {  // input = dZ (cout channels), output = dX split (cin1 | cin2)
        a.X1 = x1; a.X2 = nullptr; a.C1 = l.cout; a.C2 = 0;
        a.Wt = l.wb; a.bias = nullptr;
        a.Y1 = y; a.Y2 = y2; a.Co1 = co1 ? co1 : l.cin1 + l.cin2; a.Cout = l.cin1 + l.cin2;
        a.relu = 0; a.flip = 1; a.mask = mask;
    }
    // Tiles of 8 x 32 pixels x 64 output channels (32 below 64 channels). A grid of those
    // that leaves compute units idle (training crops: 48 blocks on the quarter-resolution
    // layers of 8 crops of 96 x 96) takes 32 channels a block, then 4 rows: the same sums
    // in the same order, more blocks and shorter chains in each. All layers of a forward
    // pass (of a training step for the crops), us before and after: 64x64 149 -> 96,
    // 256x256 155 -> 105, 512x512 206 -> 186, 1024x768 403 -> 396, 1920x1080 the same;
    // 8 crops of 96x96 312 -> 233, 16 of 128x128 407 -> 383. Splitting from fewer blocks on
    // (1 and 1 per compute unit) left 249 for the 8 crops.
    const bool one = a.C1 + a.C2 <= 32;  // one input chunk: the weights stay in LDS for all the block's tiles
    auto ntiles = [&](int th) { return N * ((H + th - 1) / th) * ((W + 31) / 32); };
    auto cotiles = [&](int nc) { return (a.Cout + 32 * nc - 1) / (32 * nc); };
    int nc = a.Cout >= 64 ? 2 : 1, th = 8;
    if (nc == 2 && ntiles(8) * cotiles(2) < 2 * d->cus) nc = 1;
    if (nc == 1 && ntiles(8) * cotiles(1) < 2 * d->cus) th = 4;
    // each block takes consecutive tiles so that the grid is about two rounds of the
    // blocks the CUs hold at once (2 per CU at 64 channels, 3 at 32), at most 16
    const int tiles = ntiles(th);
    const int64_t resident = (int64_t)d->cus * (nc == 2 ? 2 : 3);
    const int64_t want = ((int64_t)tiles * cotiles(nc) + 2 * resident - 1) / (2 * resident);
    a.tiles_per_block = one ? (int)std::max<int64_t>(1, std::min<int64_t>(16, want)) : 1;
    dim3 grid((unsigned)((tiles + a.tiles_per_block - 1) / a.tiles_per_block), cotiles(nc));
    auto run = [&](auto kernel) { ptk::launch(d->ctx, "k_dn_conv", kernel, grid, dim3(kThreads), a); };
    if (nc == 2) run(one ? k_conv_t<2, 8, true> : k_conv_t<2, 8, false>);
    else if (th == 8) run(one ? k_conv_t<1, 8, true> : k_conv_t<1, 8, false>);
    else run(one ? k_conv_t<1, 4, true> : k_conv_t<1, 4, false>);
}

// Blocks of a layer's k_conv_wgrad over all its channel tiles, and so the memory of its
// partials (36 KB a block): 256, and 512 where those take more than 8 tiles each. A tile
// costs a block about 3 us, a partial the sum's reading of it: 8 crops of 96 x 96 with
// 128 / 256 / 512 blocks a layer 270 / 193 / 168 us and 18 / 24 / 35 us for the sum.
dim3 wgrad_grid(const Layer& l, int N, int H, int W) {
    const int cot = (l.cout + 31) / 32, cit = (l.cin1 + l.cin2 + 31) / 32;
    const int tiles = N * ((H + kWR - 1) / kWR) * ((W + 31) / 32);
    const int blocks = (int64_t)tiles * cot * cit >= 2048 ? 512 : 256;
    return dim3((unsigned)std::min(tiles, std::max(1, blocks / (cot * cit))), cot, cit);
}
// The level of a layer: its resolution is the image's over 1, 2 or 4.
constexpr int kLevel[kLayers] = {0, 0, 1, 1, 2, 2, 1, 1, 0, 0, 0};
size_t layer_params(const Layer& l) { return (size_t)9 * l.cout * (l.cin1 + l.cin2) + l.cout; }

// `part`: the partials of all layers, one after the other (null: atomics).
void wgrad(pt_denoiser* d, int layer, const u16* dz, const u16* x1, const u16* x2, int N, int H, int W, float*& part) {
    const Layer& l = d->L[(size_t)layer];
    WgradArgs a{};
    a.dZ = dz; a.Cout = l.cout; a.X1 = x1; a.X2 = x2; a.C1 = l.cin1; a.C2 = l.cin2;
    a.up1 = l.up1 ? 1 : 0;
    a.g = d->g + l.w_off;
    a.part = part;
    a.N = N; a.H = H; a.W = W;
    const dim3 grid = wgrad_grid(l, N, H, W);
    if (part) part += grid.x * layer_params(l);
    ptk::launch(d->ctx, "k_dn_wgrad", k_conv_wgrad, grid, dim3(kWThreads), a);
}

dim3 ew_grid(size_t n) { return dim3((unsigned)std::min<size_t>((n + 255) / 256, 8192)); }

// Forward pass of features already in d->feat (N images H x W).
// With `grads` the gradients and the loss are cleared for a backward pass.
void forward(pt_denoiser* d, int N, int H, int W, bool grads = false) {
    pt_ctx* ctx = d->ctx;
    const int P = N * H * W, P1 = P / 4, P2 = P / 16;
    const int H1 = H / 2, W1 = W / 2, H2 = H / 4, W2 = W / 4;
    ptk::launch(ctx, "k_dn_prep", k_prep, ew_grid(P), dim3(256), (const float*)d->feat, d->x0, (size_t)P, d->g,
                grads ? d->nparam + 1 : (size_t)0);
    conv(d, d->L[0], d->x0, nullptr, d->e0a, N, H, W, false);
    conv(d, d->L[1], d->e0a, nullptr, d->e0, N, H, W, false);
    ptk::launch(ctx, "k_dn_pool", k_pool2, ew_grid((size_t)P1 * 32 / 8), dim3(256), (const u16*)d->e0, d->p1, N, H, W, 32);
    conv(d, d->L[2], d->p1, nullptr, d->e1a, N, H1, W1, false);
    conv(d, d->L[3], d->e1a, nullptr, d->e1, N, H1, W1, false);
    ptk::launch(ctx, "k_dn_pool", k_pool2, ew_grid((size_t)P2 * 64 / 8), dim3(256), (const u16*)d->e1, d->p2, N, H1, W1, 64);
    conv(d, d->L[4], d->p2, nullptr, d->ba, N, H2, W2, false);
    conv(d, d->L[5], d->ba, nullptr, d->bb, N, H2, W2, false);
    conv(d, d->L[6], d->bb, d->e1, d->d1a, N, H1, W1, false);  // bb upsampled as it is read
    conv(d, d->L[7], d->d1a, nullptr, d->d1, N, H1, W1, false);
    conv(d, d->L[8], d->d1, d->e0, d->d0a, N, H, W, false);    // d1 upsampled as it is read
    conv(d, d->L[9], d->d0a, nullptr, d->d0, N, H, W, false);
    conv(d, d->L[10], d->d0, nullptr, d->out, N, H, W, false);
}

// Backward pass: d->gc holds dL/d(out) (kOutC channels); gradients summed into d->g.
void backward(pt_denoiser* d, int N, int H, int W) {
    pt_ctx* ctx = d->ctx;
    // the weight gradients' partials, in the context's scratch memory until they are summed;
    // without it (a budget) the layers add to the gradients with atomics
    PartialSums sums{};
    size_t floats = 0;
    for (int i = 0; i < kLayers; ++i)
        floats += wgrad_grid(d->L[(size_t)i], N, H >> kLevel[i], W >> kLevel[i]).x * layer_params(d->L[(size_t)i]);
    ptk::ScratchUse scratch(ctx);
    const std::string err = ctx->err;
    const bool partials = scratch.take(floats * sizeof(float)) == PT_OK;
    if (!partials) {
        (void)hipGetLastError();
        ctx->err = err;
    }
    float* part = partials ? static_cast<float*>(scratch.p) : nullptr;
    uint32_t most = 0;
    const float* at = part;
    for (const int i : {10, 9, 8, 7, 6, 5, 4, 3, 2, 1, 0}) {  // the order of the layers below
        const Layer& l = d->L[(size_t)i];
        const uint32_t n = (uint32_t)layer_params(l), count = wgrad_grid(l, N, H >> kLevel[i], W >> kLevel[i]).x;
        sums.l[i].part = at;
        sums.l[i].off = (uint32_t)l.w_off;
        sums.l[i].n = n;
        sums.l[i].count = count;
        if (at) at += (size_t)n * count;
        most = std::max(most, n);
    }
    const int P = N * H * W, P1 = P / 4, P2 = P / 16;
    const int H1 = H / 2, W1 = W / 2, H2 = H / 4, W2 = W / 4;
    // Each conv's gradient with respect to its input goes through the ReLU that
    // produced that input as it is stored (the mask), into the other of ga / gb.
    // out = conv10(d0): no activation
    wgrad(d, 10, d->gc, d->d0, nullptr, N, H, W, part);
    conv(d, d->L[10], d->gc, nullptr, d->gb, N, H, W, true, nullptr, 0, d->d0);    // dZ9
    wgrad(d, 9, d->gb, d->d0a, nullptr, N, H, W, part);
    conv(d, d->L[9], d->gb, nullptr, d->ga, N, H, W, true, nullptr, 0, d->d0a);    // dZ8
    wgrad(d, 8, d->ga, d->d1, d->e0, N, H, W, part);
    conv(d, d->L[8], d->ga, nullptr, d->gc, N, H, W, true, d->gs0, 64);  // dL/d up(d1) (64) | dL/d e0 via skip (32)
    ptk::launch(ctx, "k_dn_up_bwd", k_up2_bwd, ew_grid((size_t)P1 * 64 / 8), dim3(256), (const u16*)d->gc,
                (const u16*)d->d1, d->gb, N, H1, W1, 64);                // dZ7
    wgrad(d, 7, d->gb, d->d1a, nullptr, N, H1, W1, part);
    conv(d, d->L[7], d->gb, nullptr, d->ga, N, H1, W1, true, nullptr, 0, d->d1a);  // dZ6
    wgrad(d, 6, d->ga, d->bb, d->e1, N, H1, W1, part);
    conv(d, d->L[6], d->ga, nullptr, d->gc, N, H1, W1, true, d->gs1, 128);  // dL/d up(bb) (128) | dL/d e1 via skip (64)
    ptk::launch(ctx, "k_dn_up_bwd", k_up2_bwd, ew_grid((size_t)P2 * 128 / 8), dim3(256), (const u16*)d->gc,
                (const u16*)d->bb, d->gb, N, H2, W2, 128);               // dZ5
    wgrad(d, 5, d->gb, d->ba, nullptr, N, H2, W2, part);
    conv(d, d->L[5], d->gb, nullptr, d->ga, N, H2, W2, true, nullptr, 0, d->ba);   // dZ4
    wgrad(d, 4, d->ga, d->p2, nullptr, N, H2, W2, part);
    conv(d, d->L[4], d->ga, nullptr, d->gc, N, H2, W2, true);            // dL/d p2 (64)
    ptk::launch(ctx, "k_dn_pool_bwd", k_pool2_bwd, ew_grid((size_t)P1 * 64 / 8), dim3(256), (const u16*)d->gc,
                (const u16*)d->gs1, (const u16*)d->e1, d->gb, N, H1, W1, 64);  // dZ3 (pool + skip)
    wgrad(d, 3, d->gb, d->e1a, nullptr, N, H1, W1, part);
    conv(d, d->L[3], d->gb, nullptr, d->ga, N, H1, W1, true, nullptr, 0, d->e1a);  // dZ2
    wgrad(d, 2, d->ga, d->p1, nullptr, N, H1, W1, part);
    conv(d, d->L[2], d->ga, nullptr, d->gc, N, H1, W1, true);            // dL/d p1 (32)
    ptk::launch(ctx, "k_dn_pool_bwd", k_pool2_bwd, ew_grid((size_t)P * 32 / 8), dim3(256), (const u16*)d->gc,
                (const u16*)d->gs0, (const u16*)d->e0, d->gb, N, H, W, 32);    // dZ1 (pool + skip)
    wgrad(d, 1, d->gb, d->e0a, nullptr, N, H, W, part);
    conv(d, d->L[1], d->gb, nullptr, d->ga, N, H, W, true, nullptr, 0, d->e0a);    // dZ0
    wgrad(d, 0, d->ga, d->x0, nullptr, N, H, W, part);
    if (partials)
        ptk::launch(ctx, "k_dn_grad_sum", k_grad_sum, dim3((most + 31) / 32, kLayers), dim3(kThreads), sums, d->g);
}

// The BF16 copies of the masters, after one Adam step on them when `adam` is given.
void update_params(pt_denoiser* d, const AdamArgs* adam) {
    AllParams A{};
    size_t most = 0;
    for (int i = 0; i < kLayers; ++i) {
        const Layer& l = d->L[(size_t)i];
        const int cin = l.cin1 + l.cin2;
        A.l[i] = LayerParams{(uint32_t)l.w_off, (uint32_t)l.cout, (uint32_t)cin, l.wf, l.wb};
        most = std::max(most, (size_t)9 * l.cout * cin + (size_t)l.cout);
    }
    const dim3 grid((unsigned)((most + 255) / 256), kLayers);
    if (adam)
        ptk::launch(d->ctx, "k_dn_adam", k_params<true>, grid, dim3(256), A, d->w, (const float*)d->g, d->m, d->v, *adam);
    else
        ptk::launch(d->ctx, "k_dn_wcopy", k_params<false>, grid, dim3(256), A, d->w, (const float*)d->g, d->m, d->v,
                    AdamArgs{});
}

int upload(pt_denoiser* d, float* dst, const float* src, size_t n) {
    hipError_t e = d->ctx->copies.to_device(dst, src, n * 4, d->ctx->stream);
    if (e != hipSuccess) return dn_fail(d, ptk::hip_fail(d->ctx, e, "denoiser upload"), d->ctx->err);
    return PT_OK;
}

int check_shape(pt_denoiser* d, int N, int H, int W) {
    if (N <= 0 || H <= 0 || W <= 0 || N > d->maxN || H > d->maxH || W > d->maxW || H % 4 || W % 4)
        return dn_fail(d, PT_ERR_INVALID_ARG, "denoiser: batch shape outside the network's limits (H, W multiples of 4)");
    return PT_OK;
}

}  // namespace

namespace ptk {

int dn_fits(const pt_denoiser* d, int W, int H) {
    return d && W > 0 && H > 0 && W <= d->maxW && H <= d->maxH && W % 4 == 0 && H % 4 == 0;
}

pt_ctx* dn_ctx(const pt_denoiser* d) { return d ? d->ctx : nullptr; }

namespace {
// Denoises half `which` of the request into d->den (texel units / scale).
void dn_half(pt_denoiser* d, const DnRequest& q, int which, float inv_scale) {
    const size_t P = (size_t)q.W * q.H;
    ptk::launch(d->ctx, "k_dn_assemble", k_dn_assemble, ew_grid(P), dim3(256), q, which, inv_scale, d->feat);
    forward(d, 1, q.H, q.W);
    ptk::launch(d->ctx, "k_dn_head", k_head, ew_grid(P), dim3(256), (const float*)d->feat, (const u16*)d->out,
                (const float*)nullptr, d->den, (u16*)nullptr, (float*)nullptr, P, 0);
}
// Both halves in one batch of 2: D(even half) into d->den, D(odd half) into
// d->den + 3 P. Each image's pixels are computed as in a batch of one, so the
// results equal two dn_half calls; a small image's two passes share the launches.
void dn_halves(pt_denoiser* d, const DnRequest& q, float inv_scale) {
    const size_t P = (size_t)q.W * q.H;
    ptk::launch(d->ctx, "k_dn_assemble", k_dn_assemble, ew_grid(P), dim3(256), q, 1, inv_scale, d->feat);
    ptk::launch(d->ctx, "k_dn_assemble", k_dn_assemble, ew_grid(P), dim3(256), q, 2, inv_scale, d->feat + P * kFeat);
    forward(d, 2, q.H, q.W);
    ptk::launch(d->ctx, "k_dn_head", k_head, ew_grid(2 * P), dim3(256), (const float*)d->feat, (const u16*)d->out,
                (const float*)nullptr, d->den, (u16*)nullptr, (float*)nullptr, 2 * P, 0);
}
}  // namespace

int dn_request_estimate(pt_denoiser* d, const DnRequest& q, float scale, int spp, double* d_lines, double* rel) {
    if (!dn_fits(d, q.W, q.H)) return dn_fail(d, PT_ERR_INVALID_ARG, "denoiser: request outside the network's limits");
    pt_ctx* ctx = d->ctx;
    const size_t P = (size_t)q.W * q.H;
    const float inv = 1.0f / scale;
    hipError_t e = hipMemsetAsync(d_lines, 0, 2 * 64 * 32 * sizeof(double), ctx->stream);
    if (e != hipSuccess) return dn_fail(d, ptk::hip_fail(ctx, e, "denoiser estimate"), ctx->err);
    const dim3 grid((unsigned)std::min<size_t>((P + 255) / 256, 2048));
    if (d->maxN >= 2) {
        dn_halves(d, q, inv);
        // D(even half) against the odd half; D(odd half) against the even half and D(even half)
        ptk::launch(ctx, "k_dn_cross", k_dn_cross, grid, dim3(256), q, (const float*)d->den, (const float*)nullptr, 2,
                    inv, d_lines);
        ptk::launch(ctx, "k_dn_cross", k_dn_cross, grid, dim3(256), q, (const float*)(d->den + P * 3),
                    (const float*)d->den, 1, inv, d_lines + 64 * 32);
    } else {
        dn_half(d, q, 1, inv);  // D(even half) against the odd half
        ptk::launch(ctx, "k_dn_cross", k_dn_cross, grid, dim3(256), q, (const float*)d->den, (const float*)nullptr, 2,
                    inv, d_lines);
        // keep D(A) (the training-target buffer is free during inference)
        e = hipMemcpyAsync(d->tgt, d->den, P * 3 * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) return dn_fail(d, ptk::hip_fail(ctx, e, "denoiser estimate"), ctx->err);
        dn_half(d, q, 2, inv);  // D(odd half) against the even half, and against D(even half)
        ptk::launch(ctx, "k_dn_cross", k_dn_cross, grid, dim3(256), q, (const float*)d->den, (const float*)d->tgt, 1,
                    inv, d_lines + 64 * 32);
    }
    std::vector<double> h((size_t)2 * 64 * 32);
    e = hipMemcpyAsync(h.data(), d_lines, h.size() * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return dn_fail(d, ptk::hip_fail(ctx, e, "denoiser estimate"), ctx->err);
    double s[2][4] = {};
    for (int k = 0; k < 2; ++k)
        for (int l = 0; l < 64; ++l)
            for (int j = 0; j < 4; ++j) s[k][j] += h[(size_t)k * 64 * 32 + (size_t)l * 32 + j];
    // E|D(A) - B|^2 = |D(A) - mu|^2 + E|B - mu|^2 for independent halves A, B:
    // the squared error of a denoised half image, bias included
    const double err2_half = 0.5 * ((s[0][0] - s[0][1]) + (s[1][0] - s[1][1]));
    // E|D(A) - D(B)|^2 = 2 var(D(half)). With the bias independent of the
    // sample count and the variance falling as 1/n, the full image's squared
    // error is err2_half - var(D(half)) / 2. At few samples the network's
    // output variance falls more slowly than 1/n (it smooths low-sample
    // inputs harder), so that credit is phased in linearly up to 64 samples.
    const double credit = std::min(1.0, spp / 64.0);
    const double err2 = err2_half - credit * 0.25 * s[1][3];
    const double m = s[0][2];
    // Both terms are differences of sums. On heavy-tailed scenes at few samples
    // (fireflies in a half's variance) they can come out zero or negative: the
    // estimate is then inconclusive, never a zero error that would finish the
    // request denoised.
    *rel = (m > 0.0 && err2_half > 0.0 && err2 > 0.0) ? std::sqrt(err2 / m) : INFINITY;
    return PT_OK;
}

int dn_request_denoise(pt_denoiser* d, const DnRequest& q, float scale, float* d_out) {
    if (!dn_fits(d, q.W, q.H)) return dn_fail(d, PT_ERR_INVALID_ARG, "denoiser: request outside the network's limits");
    const size_t P = (size_t)q.W * q.H;
    dn_half(d, q, 0, 1.0f / scale);
    ptk::launch(d->ctx, "k_dn_scale", k_dn_scale, ew_grid(P * 3), dim3(256), (const float*)d->den, scale, d_out,
                (int)(P * 3));
    return PT_OK;
}

}  // namespace ptk

extern "C" {

pt_status pt_dn_create(pt_ctx* ctx, int max_batch, int max_height, int max_width, uint64_t seed, pt_denoiser** out) {
    if (!ctx || !out || max_batch <= 0 || max_height <= 0 || max_width <= 0 || max_height % 4 || max_width % 4)
        return PT_ERR_INVALID_ARG;
    *out = nullptr;
    pt_denoiser* d = new (std::nothrow) pt_denoiser();
    if (!d) return PT_ERR_INVALID_ARG;
    d->ctx = ctx;
    {
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, ctx->device) == hipSuccess && cu > 0)
            d->cus = cu;
    }
    d->maxN = max_batch;
    d->maxH = max_height;
    d->maxW = max_width;
    const int spec[11][4] = {{kIn, 0, 32, 1}, {32, 0, 32, 1}, {32, 0, 64, 1}, {64, 0, 64, 1}, {64, 0, 128, 1},
                             {128, 0, 128, 1}, {128, 64, 64, 1}, {64, 0, 64, 1}, {64, 32, 32, 1}, {32, 0, 32, 1},
                             {32, 0, kOutC, 0}};
    size_t off = 0;
    for (auto& sp : spec) {
        Layer l;
        l.cin1 = sp[0]; l.cin2 = sp[1]; l.cout = sp[2]; l.relu = sp[3] != 0;
        l.up1 = l.cin2 > 0;  // the decoder layers that concatenate a skip connection
        l.w_off = off;
        off += (size_t)9 * l.cout * (l.cin1 + l.cin2);
        l.b_off = off;
        off += (size_t)l.cout;
        d->L.push_back(l);
        // k_conv_t reads and writes 8 channels per 16-byte vector, splits the
        // input at C1 and the output at Co1, and skips the second 16-channel
        // step of a 16-channel input: channel counts of both passes (forward,
        // backward-data) are multiples of 16
        const int cin = l.cin1 + l.cin2;
        if (cin % 16 || l.cout % 16 || l.cin1 % 16) {
            delete d;
            return PT_ERR_INVALID_ARG;
        }
    }
    d->nparam = off;
    const size_t P = (size_t)max_batch * max_height * max_width;
    // activations: BF16 element counts
    const size_t act[] = {P * kIn, P * 32, P * 32, P / 4 * 32, P / 4 * 64, P / 4 * 64, P / 16 * 64, P / 16 * 128,
                          P / 16 * 128, P / 4 * 64, P / 4 * 64, P * 32, P * 32, P * kOutC,
                          P * 64, P * 64, P * 64, P / 4 * 64, P * 32};
    size_t bytes = 4 * off * 4 + 2 * off * 2 + (P * kFeat + P * 3 + P * 3 + 64) * 4 + 64 * 256;
    for (size_t a : act) bytes += (a * 2 + 255) / 256 * 256;
    int st = ptk::dev_alloc(ctx, d->mem, bytes);
    if (st != PT_OK) {
        delete d;
        return st;
    }
    char* p = static_cast<char*>(d->mem.p);
    auto carve = [&](size_t b) {
        char* q = p;
        p += (b + 255) / 256 * 256;
        return q;
    };
    d->w = reinterpret_cast<float*>(carve(off * 4));
    d->g = reinterpret_cast<float*>(carve(off * 4 + 4));
    d->loss = d->g + off;  // cleared with the gradients
    d->m = reinterpret_cast<float*>(carve(off * 4));
    d->v = reinterpret_cast<float*>(carve(off * 4));
    d->wbf = reinterpret_cast<u16*>(carve(off * 4));
    u16** acts[] = {&d->x0, &d->e0a, &d->e0, &d->p1, &d->e1a, &d->e1, &d->p2, &d->ba, &d->bb, &d->d1a, &d->d1,
                    &d->d0a, &d->d0, &d->out, &d->ga, &d->gb, &d->gc, &d->gs1, &d->gs0};
    static_assert(sizeof(act) / sizeof(act[0]) == sizeof(acts) / sizeof(acts[0]), "one size per activation");
    for (size_t i = 0; i < sizeof(act) / sizeof(act[0]); ++i) *acts[i] = reinterpret_cast<u16*>(carve(act[i] * 2));
    d->feat = reinterpret_cast<float*>(carve(P * kFeat * 4));
    d->tgt = reinterpret_cast<float*>(carve(P * 3 * 4));
    d->den = reinterpret_cast<float*>(carve(P * 3 * 4));
    u16* wb = d->wbf;
    for (Layer& l : d->L) {
        const size_t n = (size_t)9 * l.cout * (l.cin1 + l.cin2);
        l.wf = wb;
        l.wb = wb + n;
        wb += 2 * n;
    }
    // He-normal weights, zero biases
    std::vector<float> h(off, 0.0f);
    std::mt19937_64 rng(seed);
    for (const Layer& l : d->L) {
        const int cin = l.cin1 + l.cin2;
        std::normal_distribution<float> nd(0.0f, std::sqrt(2.0f / (9.0f * (float)cin)));
        for (size_t i = 0; i < (size_t)9 * l.cout * cin; ++i) h[l.w_off + i] = nd(rng);
    }
    for (int t = 0; t < 9; ++t)  // the output layer starts small: the network starts near the identity
        for (int co = 0; co < kOutC; ++co)
            for (int ci = 0; ci < 32; ++ci) h[d->L[10].w_off + ((size_t)t * kOutC + co) * 32 + ci] *= 0.1f;
    (void)hipSetDevice(ctx->device);
    hipError_t e = hipMemcpyAsync(d->w, h.data(), off * 4, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(d->m, 0, off * 4, ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(d->v, 0, off * 4, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        ptk::dev_free(ctx, d->mem);
        delete d;
        return ptk::hip_fail(ctx, e, "pt_dn_create");
    }
    update_params(d, nullptr);
    *out = d;
    return PT_OK;
}

void pt_dn_destroy(pt_denoiser* d) {
    if (!d) return;
    (void)hipSetDevice(d->ctx->device);
    (void)hipStreamSynchronize(d->ctx->stream);
    ptk::dev_free(d->ctx, d->mem);
    delete d;
}

const char* pt_dn_last_error(const pt_denoiser* d) { return d ? d->err.c_str() : ""; }

int64_t pt_dn_param_count(const pt_denoiser* d) { return d ? (int64_t)d->nparam : 0; }

pt_status pt_dn_set_loss(pt_denoiser* d, int kind) {
    if (!d || (kind != PT_DN_LOSS_L1_LOG && kind != PT_DN_LOSS_L2)) return PT_ERR_INVALID_ARG;
    d->loss_kind = kind;
    return PT_OK;
}

pt_status pt_dn_get_params(pt_denoiser* d, float* host, size_t n) {
    if (!d || !host || n != d->nparam) return PT_ERR_INVALID_ARG;
    hipError_t e = d->ctx->copies.to_host(host, d->w, n * 4, d->ctx->stream);
    return e == hipSuccess ? PT_OK : dn_fail(d, ptk::hip_fail(d->ctx, e, "pt_dn_get_params"), d->ctx->err);
}

pt_status pt_dn_set_params(pt_denoiser* d, const float* host, size_t n) {
    if (!d || !host || n != d->nparam) return PT_ERR_INVALID_ARG;
    int st = upload(d, d->w, host, n);
    if (st != PT_OK) return st;
    update_params(d, nullptr);
    hipError_t e = hipStreamSynchronize(d->ctx->stream);
    return e == hipSuccess ? PT_OK : dn_fail(d, ptk::hip_fail(d->ctx, e, "pt_dn_set_params"), d->ctx->err);
}

pt_status pt_dn_denoise(pt_denoiser* d, const float* features, int N, int H, int W, float* denoised) {
    if (!d || !features || !denoised) return PT_ERR_INVALID_ARG;
    int st = check_shape(d, N, H, W);
    if (st != PT_OK) return st;
    const size_t P = (size_t)N * H * W;
    (void)hipSetDevice(d->ctx->device);
    st = upload(d, d->feat, features, P * kFeat);
    if (st != PT_OK) return st;
    forward(d, N, H, W);
    ptk::launch(d->ctx, "k_dn_head", k_head, ew_grid(P), dim3(256), (const float*)d->feat, (const u16*)d->out,
                (const float*)nullptr, d->den, (u16*)nullptr, (float*)nullptr, P, 0);
    hipError_t e = d->ctx->copies.to_host(denoised, d->den, P * 3 * 4, d->ctx->stream);
    return e == hipSuccess ? PT_OK : dn_fail(d, ptk::hip_fail(d->ctx, e, "pt_dn_denoise"), d->ctx->err);
}

pt_status pt_dn_gradients(pt_denoiser* d, const float* features, const float* target, int N, int H, int W,
                          float* loss, float* host_grads, size_t n_grads) {
    if (!d || !features || !target) return PT_ERR_INVALID_ARG;
    if (host_grads && n_grads != d->nparam) return PT_ERR_INVALID_ARG;
    int st = check_shape(d, N, H, W);
    if (st != PT_OK) return st;
    const size_t P = (size_t)N * H * W;
    pt_ctx* ctx = d->ctx;
    (void)hipSetDevice(ctx->device);
    st = upload(d, d->feat, features, P * kFeat);
    if (st == PT_OK) st = upload(d, d->tgt, target, P * 3);
    if (st != PT_OK) return st;
    hipError_t e = hipSuccess;
    forward(d, N, H, W, true);
    ptk::launch(ctx, "k_dn_head", k_head, ew_grid(P), dim3(256), (const float*)d->feat, (const u16*)d->out,
                (const float*)d->tgt, (float*)nullptr, d->gc, d->loss, P, d->loss_kind);
    backward(d, N, H, W);
    if (loss) e = hipMemcpyAsync(loss, d->loss, 4, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess && host_grads) e = ctx->copies.to_host(host_grads, d->g, n_grads * 4, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return e == hipSuccess ? PT_OK : dn_fail(d, ptk::hip_fail(ctx, e, "pt_dn_gradients"), ctx->err);
}

pt_status pt_dn_train_step(pt_denoiser* d, const float* features, const float* target, int N, int H, int W, float lr,
                           float* loss) {
    int st = pt_dn_gradients(d, features, target, N, H, W, loss, nullptr, 0);
    if (st != PT_OK) return st;
    d->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)d->step), c2 = 1.0f - std::pow(b2, (float)d->step);
    const AdamArgs adam{lr, b1, b2, 1e-8f, c1, c2};
    update_params(d, &adam);
    hipError_t e = hipStreamSynchronize(d->ctx->stream);
    return e == hipSuccess ? PT_OK : dn_fail(d, ptk::hip_fail(d->ctx, e, "pt_dn_train_step"), d->ctx->err);
}

}  // extern "C"
