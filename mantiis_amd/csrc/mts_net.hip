// Learned warm start: a four-level convolutional encoder-decoder (U-Net)
// that maps (fluid mask, log10 Kn, forcing) to the steady velocity field of a
// periodic porous lattice, with its own forward and backward kernels.
//
// Every convolution (3x3 and 1x1, periodic padding) runs on BF16 matrix cores
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation):
//   forward        Y[p, co]      = sum_{kk, ci} X[p + o(kk), ci] W[kk, co, ci]
//   backward data  dX[p, ci]     = sum_{kk, co} dY[p - o(kk), co] W[kk, co, ci]
//   backward wgt   dW[kk, co, ci] = sum_p dY[p, co] X[p + o(kk), ci]
// k_conv (the first two) holds a tile of pixels with its halo in LDS and takes
// all nine offsets from there; k_convw (the third) takes its operands, whose
// contraction runs over pixels, from LDS with transposing reads.  The concatenated
// and upsampled inputs of the decoder are read from their two sources, never
// written.  Activations are NHWC BF16.  Gradients enter a product in BF16 with
// the ReLU mask applied (the producing pass rounds and masks where nothing is
// added in between) and are FP32 where parts are summed; parameters FP32
// masters with BF16 copies in the order the products read them; Adam in FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "mantiis_hip.h"

namespace mts {
int set_error(int code, const std::string& msg);  // mts_api.hip
}
using mts::set_error;

#define NET_TRY(expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess)                                                              \
            return set_error(e_ == hipErrorOutOfMemory ? MTS_ERR_OOM : MTS_ERR_HIP,        \
                             std::string(#expr) + ": " + hipGetErrorString(e_));           \
    } while (0)

namespace net {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef uint4 v16;

// ---------------------------------------------------------------- convolution
__device__ __forceinline__ int wrapn(int v, int n) {  // v >= -n
    v = v < 0 ? v + n : v;
    return v >= n ? v % n : v;
}
// offset of kernel index kk: 3 (dy + 1) + (dx + 1) for 3x3, 0 for 1x1
__device__ __forceinline__ void koff(int kk, int ksz, int& dy, int& dx) {
    dy = ksz == 3 ? kk / 3 - 1 : 0;
    dx = ksz == 3 ? kk % 3 - 1 : 0;
}

// Input of a convolution: C1 channels of X -- at half the resolution when
// up -- and then C2 channels of X2 (the decoder's upsampled and skip parts).
struct ConvIn {
    const bf16 *X, *X2;
    int C1, C2, up;
    int H, W;
    __device__ __forceinline__ const bf16* at(int b, int y, int x, int c) const {
        if (c < C1) {
            const int64_t p = up ? ((int64_t)b * (H / 2) + y / 2) * (W / 2) + x / 2 : ((int64_t)b * H + y) * W + x;
            return X + p * C1 + c;
        }
        return X2 + (((int64_t)b * H + y) * W + x) * C2 + (c - C1);
    }
};

// Forward and backward-data convolution.
struct ConvArgs {
    ConvIn in;
    int Cin, Cout, ksz, sgn;  // sgn: +1 forward, -1 backward data (offsets reversed)
    int steps;                // products of 32 deep: ceil(ksz^2 Cin / 32)
    int tilesX, tilesY;
    const bf16* Wf;           // packed weights (k_pack)
    const float* bias;        // forward
    const bf16* mask;         // backward, BF16 output: the ReLU output whose gradient this is
    bf16* Y;                  // BF16 output, or
    float* Yf;                // FP32 output
    int relu;
};

// Pixel stride of a staged tile: an odd number of 16-byte units, so that eight
// neighbouring pixels' vectors fall into different banks.
__host__ __device__ inline int conv_stride(int Cin) { return Cin % 8 ? 8 : ((Cin / 8) | 1) * 16; }
__host__ __device__ inline int conv_off_bytes(int steps, bool small) { return small ? 32 * 4 : (steps * 4 * 4 + 15) / 16 * 16; }
inline size_t conv_lds(int Cin, int ksz, int steps, int rows) {
    const int pad = ksz / 2;
    return (size_t)conv_off_bytes(steps, Cin % 8 != 0) + (size_t)(rows + 2 * pad) * (16 + 2 * pad) * conv_stride(Cin);
}

// One block: 16 x (WM MTW) pixels of one image times CH = WN NTW tiles of 16
// output channels (blockIdx.y: which).  A product step takes four groups of
// eight channels, group g being channels 8 (g mod Cin/8) of offset g / (Cin/8),
// so narrow layers fill the 32-deep products across offsets; every output's
// terms are added in the order (offset, channel).  A layer with fewer than
// eight channels (the three of the input, the two of the head's gradient) is
// one step whose eight elements per lane are picked one by one.
//
// Bound: latency, with no unit busy (counters: matrix cores 12 to 22% of the
// time, LDS 8 to 21%; the head 2 to 8%): a block stages its tile and then
// multiplies, and the accumulators and read-ahead leave two or three waves per
// SIMD.  With offsets, weights and pixels read when they were used every step
// also waited for the LDS twice: predicting four 512 x 512 images (191 GFLOP)
// took 767 us against 605 with them read ahead (one pixel read feeds NTW
// products, one weight read MTW).  The 64x64 implicit GEMM before it, which
// fetched every input element nine times through per-element index divisions,
// took 1703 us; a training step on eight 256 x 256 images went from 5.02 to
// 2.00 ms with k_convw.
// MEM: operands from memory, for tiles that do not fit in LDS.
template <int MTW, int NTW, int WM, int WN, bool MEM>
__global__ void __launch_bounds__(256) k_conv(ConvArgs a) {
    extern __shared__ char lds[];
    constexpr int TH = WM * MTW, CH = WN * NTW;
    const int t = threadIdx.x, l = t & 63, w = t >> 6, i = l & 15, q = l >> 4;
    const int wm = w % WM, wn = w / WM;
    const bool small = a.Cin % 8 != 0;
    const int C8 = a.Cin / 8, pad = a.ksz / 2, LW = 16 + 2 * pad, PS = conv_stride(a.Cin);
    const int H = a.in.H, W = a.in.W;
    int bid = blockIdx.x;
    const int x0 = bid % a.tilesX * 16;
    bid /= a.tilesX;
    const int y0 = bid % a.tilesY * TH, b = bid / a.tilesY;
    int* s_off = (int*)lds;
    char* tile = lds + conv_off_bytes(a.steps, small);
    const int ng = a.ksz * a.ksz * (small ? a.Cin : C8);
    if (!MEM) {
        for (int g = t; g < (small ? 32 : a.steps * 4); g += 256) {
            const int d = small ? a.Cin : C8, kk = g / d, c = g - kk * d;
            int dy, dx;
            koff(kk, a.ksz, dy, dx);
            s_off[g] = g < ng ? ((pad + a.sgn * dy) * LW + pad + a.sgn * dx) * PS + c * (small ? 2 : 16) : 0;
        }
        const int rows = TH + 2 * pad;
        if (small) {
            for (int v = t; v < rows * LW; v += 256) {
                const int ly = v / LW, lx = v - ly * LW;
                const bf16* src = a.in.at(b, wrapn(y0 - pad + ly, H), wrapn(x0 - pad + lx, W), 0);
                for (int c = 0; c < a.Cin; c++) *(bf16*)(tile + v * PS + 2 * c) = src[c];
            }
        } else {
            // a wave per row: LW C8 vectors, the pixel by a fixed-point
            // division (exact: 18 C8^2 < 2^20 for every tile that fits)
            const uint32_t inv = (1u << 20) / (uint32_t)C8 + 1u;
            const int n1 = a.in.C1 / 8, C1 = a.in.C1, C2 = a.in.C2, up = a.in.up;
            for (int ly = w; ly < rows; ly += 4) {
                const int gy = wrapn(y0 - pad + ly, H);
                const bf16* r1 = a.in.X + (up ? ((int64_t)b * (H / 2) + gy / 2) * (W / 2) : ((int64_t)b * H + gy) * W) * C1;
                const bf16* r2 = a.in.X2 + ((int64_t)b * H + gy) * W * C2;
                char* to = tile + ly * LW * PS;
                for (int v = l; v < LW * C8; v += 64) {
                    const int px = (int)(((uint32_t)v * inv) >> 20), c8 = v - px * C8;
                    const int gx = wrapn(x0 - pad + px, W);
                    const bf16* src = c8 < n1 ? r1 + (up ? gx >> 1 : gx) * C1 + c8 * 8 : r2 + gx * C2 + (c8 - n1) * 8;
                    *(v16*)(to + px * PS + c8 * 16) = *(const v16*)src;
                }
            }
        }
    }
    f32x4 acc[MTW][NTW];
#pragma unroll
    for (int m = 0; m < MTW; m++)
#pragma unroll
        for (int n = 0; n < NTW; n++) acc[m][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // weights of step k: CH tiles of 64 lanes x 8 elements
    const bf16x8* wp = (const bf16x8*)a.Wf + ((int64_t)blockIdx.y * a.steps * CH + wn * NTW) * 64 + l;
    const char* px0 = tile + ((wm * MTW) * LW + i) * PS;
    if (!MEM && !small) {
        // Weights and offsets are read two steps ahead and pixels one, so that
        // a step's products wait for nothing they have just asked for; the
        // rings' places are fixed by unrolling six steps.
        bf16x8 wr[3][NTW], xf[2][MTW];
        int of[3];
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (u < a.steps)
#pragma unroll
                for (int n = 0; n < NTW; n++) wr[u][n] = wp[(u * CH + n) * 64];
        __syncthreads();
        of[0] = s_off[q];
        of[1] = s_off[a.steps > 1 ? 4 + q : q];
#pragma unroll
        for (int m = 0; m < MTW; m++) xf[0][m] = *(const bf16x8*)(px0 + m * LW * PS + of[0]);
        for (int k0 = 0; k0 < a.steps; k0 += 6) {
#pragma unroll
            for (int u = 0; u < 6; u++) {
                const int k = k0 + u;
                if (k >= a.steps) break;
                if (k + 2 < a.steps) {
#pragma unroll
                    for (int n = 0; n < NTW; n++) wr[(u + 2) % 3][n] = wp[((k + 2) * CH + n) * 64];
                    of[(u + 2) % 3] = s_off[4 * (k + 2) + q];
                }
                if (k + 1 < a.steps) {
                    const int o = of[(u + 1) % 3];
#pragma unroll
                    for (int m = 0; m < MTW; m++) xf[(u + 1) % 2][m] = *(const bf16x8*)(px0 + m * LW * PS + o);
                }
                // lanes past the last group hold zeros (their weights are zero,
                // but an infinite activation would make a NaN of the product)
                if (4 * k + 3 >= ng && 4 * k + q >= ng)
#pragma unroll
                    for (int m = 0; m < MTW; m++) xf[u % 2][m] = bf16x8{};
#pragma unroll
                for (int n = 0; n < NTW; n++)
#pragma unroll
                    for (int m = 0; m < MTW; m++)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u % 3][n], xf[u % 2][m], acc[m][n], 0, 0, 0);
            }
        }
    } else if (!MEM) {
        __syncthreads();
        for (int k = 0; k < a.steps; k++) {
            bf16x8 xf[MTW];
#pragma unroll
            for (int m = 0; m < MTW; m++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const bf16 v = *(const bf16*)(px0 + m * LW * PS + s_off[8 * q + e]);
                    xf[m][e] = 8 * q + e < ng ? v : (bf16)0.0f;
                }
#pragma unroll
            for (int n = 0; n < NTW; n++) {
                const bf16x8 wv = wp[(k * CH + n) * 64];
#pragma unroll
                for (int m = 0; m < MTW; m++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xf[m], acc[m][n], 0, 0, 0);
            }
        }
    } else {
        // A step's operands are read AHEAD steps before its products: reading
        // them when they are used made every step a round trip to memory (one
        // 128 x 128 image, 96 base channels: 912 us, 614 so, 831 in the former
        // implicit GEMM).
        constexpr int AHEAD = 4;
        bf16x8 wr[AHEAD][NTW], xf[AHEAD][MTW];
        auto fetch = [&](int k, bf16x8* wv, bf16x8* xv) {
            const int g = 4 * k + q, kk = min(g / C8, a.ksz * a.ksz - 1), c8 = g - g / C8 * C8;
            int dy, dx;
            koff(kk, a.ksz, dy, dx);
#pragma unroll
            for (int n = 0; n < NTW; n++) wv[n] = wp[(k * CH + n) * 64];
#pragma unroll
            for (int m = 0; m < MTW; m++)
                xv[m] = *(const bf16x8*)a.in.at(b, wrapn(y0 + wm * MTW + m + a.sgn * dy, H), wrapn(x0 + i + a.sgn * dx, W),
                                                c8 * 8);
        };
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
            if (u < a.steps) fetch(u, wr[u], xf[u]);
        for (int k0 = 0; k0 < a.steps; k0 += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                const int k = k0 + u;
                if (k >= a.steps) break;
                if (4 * k + 3 >= ng && 4 * k + q >= ng)  // past the last group (see above)
#pragma unroll
                    for (int m = 0; m < MTW; m++) xf[u][m] = bf16x8{};
#pragma unroll
                for (int n = 0; n < NTW; n++)
#pragma unroll
                    for (int m = 0; m < MTW; m++)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u][n], xf[u][m], acc[m][n], 0, 0, 0);
                if (k + AHEAD < a.steps) fetch(k + AHEAD, wr[u], xf[u]);
            }
        }
    }
    // lane (i, q) holds channels 4 q .. + 3 of pixel i of each row
    const int x = x0 + i, y1 = y0 + wm * MTW;
    if (x >= W) return;
    const int64_t o0 = (((int64_t)b * H + y1) * W + x) * a.Cout;
    const int rowStep = W * a.Cout;
#pragma unroll
    for (int n = 0; n < NTW; n++) {
        const int c = ((blockIdx.y * WN + wn) * NTW + n) * 16 + 4 * q;
        if (c >= a.Cout) continue;
        if (a.Cout & 3) {  // the head's two channels, odd widths of the check
            for (int m = 0; m < MTW && y1 + m < H; m++)
                for (int e = 0; e < min(4, a.Cout - c); e++) {
                    const int64_t o = o0 + (int64_t)m * rowStep + c + e;
                    float v = acc[0][n][e];
#pragma unroll
                    for (int mm = 1; mm < MTW; mm++) v = m == mm ? acc[mm][n][e] : v;
                    if (a.bias) v += a.bias[c + e];
                    if (a.relu) v = fmaxf(v, 0.0f);
                    if (a.Yf) a.Yf[o] = v;
                    else a.Y[o] = (bf16)((a.mask && (float)a.mask[o] <= 0.0f) ? 0.0f : v);
                }
            continue;
        }
        f32x4 bs = {0.0f, 0.0f, 0.0f, 0.0f};
        if (a.bias) {
#pragma unroll
            for (int e = 0; e < 4; e++) bs[e] = a.bias[c + e];
        }
        if (a.Yf) {
#pragma unroll
            for (int m = 0; m < MTW; m++)
                if (y1 + m < H) {
                    f32x4 v = acc[m][n];
                    if (a.bias) v += bs;
                    if (a.relu) {
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = fmaxf(v[e], 0.0f);
                    }
                    *(f32x4*)(a.Yf + o0 + m * rowStep + c) = v;
                }
        } else if (a.mask) {
            bf16x4 mk[MTW];
#pragma unroll
            for (int m = 0; m < MTW; m++)
                mk[m] = y1 + m < H ? *(const bf16x4*)(a.mask + o0 + m * rowStep + c) : bf16x4{};
#pragma unroll
            for (int m = 0; m < MTW; m++)
                if (y1 + m < H) {
                    bf16x4 r;
#pragma unroll
                    for (int e = 0; e < 4; e++) r[e] = (bf16)((float)mk[m][e] <= 0.0f ? 0.0f : acc[m][n][e]);
                    *(bf16x4*)(a.Y + o0 + m * rowStep + c) = r;
                }
        } else {
#pragma unroll
            for (int m = 0; m < MTW; m++)
                if (y1 + m < H) {
                    bf16x4 r;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float v = acc[m][n][e] + bs[e];
                        if (a.relu) v = fmaxf(v, 0.0f);
                        r[e] = (bf16)v;
                    }
                    *(bf16x4*)(a.Y + o0 + m * rowStep + c) = r;
                }
        }
    }
}

// Output-channel tiles per block: of 6, 4, 3, 2, 1 the one that pads least,
// the largest of those.
inline int conv_chunk(int C) {
    const int nt = (C + 15) / 16;
    int best = 1, cost = 1 << 30;
    for (int ch : {6, 4, 3, 2, 1}) {
        const int c = (nt + ch - 1) / ch * ch;
        if (c < cost) {
            cost = c;
            best = ch;
        }
    }
    return best;
}
inline int conv_chunks(int C) {
    const int ch = conv_chunk(C);
    return ((C + 15) / 16 + ch - 1) / ch;
}
inline int conv_steps(int Cin, int ksz) { return (ksz * ksz * Cin + 31) / 32; }
inline int64_t conv_pack_elems(int Cin, int Cout, int ksz) {
    return (int64_t)conv_chunks(Cout) * conv_steps(Cin, ksz) * conv_chunk(Cout) * 512;
}

template <int MTW, int NTW, int WM, int WN, bool MEM = false>
int launch_conv_t(ConvArgs& a, int B, size_t lds, hipStream_t st) {
    a.tilesX = (a.in.W + 15) / 16;
    a.tilesY = (a.in.H + WM * MTW - 1) / (WM * MTW);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)k_conv<MTW, NTW, WM, WN, MEM>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL((k_conv<MTW, NTW, WM, WN, MEM>), dim3(a.tilesX * a.tilesY * B, conv_chunks(a.Cout)), dim3(256), lds, st, a);
    return 0;
}

// Rows per block: 16 while two blocks fit in a CU's LDS and the launch has at
// least two blocks per CU; otherwise 8, then 4.  The rule looks at LDS only: the
// 16-row form of six output tiles (more than 80 output channels) takes 308
// registers, one wave per SIMD, and two of its blocks never share a CU.
inline int launch_conv(ConvArgs a, int B, hipStream_t st) {
    a.steps = conv_steps(a.Cin, a.ksz);
    constexpr size_t CU_LDS = 160 * 1024;
    int rows = 16;
    auto blocks = [&](int r) {
        return (int64_t)((a.in.W + 15) / 16) * ((a.in.H + r - 1) / r) * B * conv_chunks(a.Cout);
    };
    while (rows > 4 && (conv_lds(a.Cin, a.ksz, a.steps, rows) > CU_LDS / 2 || blocks(rows) < 512)) rows /= 2;
    const size_t lds = conv_lds(a.Cin, a.ksz, a.steps, rows);
    if (lds > CU_LDS) switch (conv_chunk(a.Cout)) {
        case 1: return launch_conv_t<1, 1, 4, 1, true>(a, B, 0, st);
        case 2: return launch_conv_t<1, 2, 4, 1, true>(a, B, 0, st);
        case 3: return launch_conv_t<1, 3, 4, 1, true>(a, B, 0, st);
        case 4: return launch_conv_t<2, 2, 2, 2, true>(a, B, 0, st);
        default: return launch_conv_t<2, 3, 2, 2, true>(a, B, 0, st);
    }
    switch (conv_chunk(a.Cout) * 100 + rows) {
        case 116: return launch_conv_t<4, 1, 4, 1>(a, B, lds, st);
        case 108: return launch_conv_t<2, 1, 4, 1>(a, B, lds, st);
        case 104: return launch_conv_t<1, 1, 4, 1>(a, B, lds, st);
        case 216: return launch_conv_t<4, 2, 4, 1>(a, B, lds, st);
        case 208: return launch_conv_t<2, 2, 4, 1>(a, B, lds, st);
        case 204: return launch_conv_t<1, 2, 4, 1>(a, B, lds, st);
        case 316: return launch_conv_t<4, 3, 4, 1>(a, B, lds, st);
        case 308: return launch_conv_t<2, 3, 4, 1>(a, B, lds, st);
        case 304: return launch_conv_t<1, 3, 4, 1>(a, B, lds, st);
        case 416: return launch_conv_t<8, 2, 2, 2>(a, B, lds, st);
        case 408: return launch_conv_t<4, 2, 2, 2>(a, B, lds, st);
        case 404: return launch_conv_t<2, 2, 2, 2>(a, B, lds, st);
        case 616: return launch_conv_t<8, 3, 2, 2>(a, B, lds, st);
        case 608: return launch_conv_t<4, 3, 2, 2>(a, B, lds, st);
        default: return launch_conv_t<2, 3, 2, 2>(a, B, lds, st);
    }
}

// BF16 weights in the order k_conv reads them, for every layer and direction
// (blockIdx.y: job): element e of lane l of tile j of chunk z at step k is
// W[kk][n][c] with n = 16 (z CH + j) + l % 16 and (kk, c) element 32 k + 8 (l / 16) + e
// of the (offset, channel) order; zero beyond them.
struct PackJob {
    int64_t src, dst;  // offsets in the parameters and in the packed weights
    int cin, cout, ksz, back;
};
constexpr int MAX_JOBS = 30;
struct PackJobs {
    PackJob j[MAX_JOBS];
};
__global__ void __launch_bounds__(256) k_pack(const float* __restrict__ P, bf16* __restrict__ out, PackJobs J) {
    const PackJob& j = J.j[blockIdx.y];
    const int K = j.back ? j.cout : j.cin, N = j.back ? j.cin : j.cout;  // contracted, output channels
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int nt = (N + 15) / 16;
    int ch = 1, cost = 1 << 30;  // conv_chunk(N)
    for (int k = 0; k < 5; k++) {
        const int h = k == 0 ? 6 : 5 - k, c = (nt + h - 1) / h * h;
        if (c < cost) {
            cost = c;
            ch = h;
        }
    }
    const int steps = (j.ksz * j.ksz * K + 31) / 32;
    if (v >= (int64_t)cost * steps * 512) return;
    const int e = (int)(v & 7), l = (int)(v >> 3) & 63;
    int64_t r = v >> 9;
    const int tj = (int)(r % ch);
    r /= ch;
    const int k = (int)(r % steps), z = (int)(r / steps);
    const int n = 16 * (z * ch + tj) + (l & 15), kc = 32 * k + 8 * (l >> 4) + e, kk = kc / K, c = kc - kk * K;
    float x = 0.0f;
    if (n < N && kk < j.ksz * j.ksz)
        x = P[j.src + (j.back ? ((int64_t)kk * j.cout + c) * j.cin + n : ((int64_t)kk * j.cout + n) * j.cin + c)];
    out[j.dst + v] = (bf16)x;
}

// Weight and bias gradients of a convolution.
struct WgArgs {
    ConvIn in;
    const bf16* dY;  // [p][Cout]
    float* part;     // [split][Cout][nkk * Cin + 1], the last column the bias
    int Cin, Cout, ksz, B, tilesX, tilesY, nsplit;
};
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
// Eight pixels of one channel from a pixel-major tile: the 16 lanes of a group
// address four pixels' 16 channels (8 bytes each), and the read hands lane i
// the four pixels of channel i; two reads make the operand's eight.
__device__ __forceinline__ bf16x8 tr8(const char* p, int stride4) {
    union {
        s16x4 h[2];
        bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + stride4));
    return u.v;
}

// One block: MT tiles of 16 output channels (blockIdx.z) times 32 input
// channels (blockIdx.y) of all nine offsets, summed over the pixel tiles
// (16 x 8) of its split.  Wave w takes three of the 18 (offset, 16 channels)
// tiles; a product step contracts 32 pixels, two rows of the tile.  The
// offsets' shifts are shifts of whole pixels in the staged tile, which the
// transposing reads take as they are.  Pixels past the image have zero
// gradient; channels past the layer's give rows and columns that are not
// stored.  The bias is the product with a vector of ones.
//
// Bound: the LDS comes nearest at few output channels (33% busy for 24 of them,
// half of it conflicts; 12 to 15% above; matrix cores 8 to 14%): 2 MT / (MT + 3)
// of a product's operands are reused, and staging lies between the tiles.  The
// GEMM it replaces gathered the shifted pixels from memory per offset and
// transposed through 4-byte LDS stores: 118 us per layer on average of a training
// step on eight 256 x 256 images (42 now), and a separate 31 us pass for the bias.
constexpr int WG_H = 8, WG_XS = 80;
template <int MT>
__global__ void __launch_bounds__(384) k_convw(WgArgs a) {
    constexpr int YS = MT * 32 + 16;
    __shared__ __align__(16) char sX[(WG_H + 2) * 18 * WG_XS];
    __shared__ __align__(16) char sY[WG_H * 16 * YS + 16];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, i = l & 15, q = l >> 4;
    const int H = a.in.H, W = a.in.W, nkk = a.ksz * a.ksz;
    const int ci0 = blockIdx.y * 32, co0 = blockIdx.z * MT * 16;
    const int nci = min(32, a.Cin - ci0), nco = min(MT * 16, a.Cout - co0);
    const int ntiles = a.tilesX * a.tilesY * a.B;
    const int t0 = (int)((int64_t)ntiles * blockIdx.x / a.nsplit), t1 = (int)((int64_t)ntiles * (blockIdx.x + 1) / a.nsplit);
    f32x4 acc[3][MT], accb[MT];
    bool use[3];
    int xo[3];
#pragma unroll
    for (int n = 0; n < 3; n++) {
        const int id = 3 * w + n, kk = id >> 1, ct = id & 1;
        int dy, dx;
        koff(kk, a.ksz, dy, dx);
        use[n] = kk < nkk && ct * 16 < nci;
        xo[n] = ((1 + dy) * 18 + 1 + dx) * WG_XS + ct * 32;
#pragma unroll
        for (int m = 0; m < MT; m++) acc[n][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int m = 0; m < MT; m++) accb[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const bool bias = w == 0 && blockIdx.y == 0;
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (bf16)1.0f;
    // the thread's vectors of a tile: the next tile's are loaded while the
    // current one is multiplied
    constexpr int NX = ((WG_H + 2) * 18 * 4 + 383) / 384, NY = (WG_H * 16 * MT * 2 + 383) / 384;
    v16 xr[NX], yr[NY];
    const bool vx = a.Cin % 8 == 0, vy = a.Cout % 8 == 0;
    auto fetch = [&](int tl) {
        const int x0 = tl % a.tilesX * 16, y0 = tl / a.tilesX % a.tilesY * WG_H, b = tl / a.tilesX / a.tilesY;
        if (vx) {
#pragma unroll
            for (int k = 0; k < NX; k++) {
                const int v = t + 384 * k, px = v >> 2, c = (v & 3) * 8, ly = px / 18, lx = px - ly * 18;
                xr[k] = v16{0u, 0u, 0u, 0u};
                if (v < (WG_H + 2) * 18 * 4 && c < nci)
                    xr[k] = *(const v16*)a.in.at(b, wrapn(y0 - 1 + ly, H), wrapn(x0 - 1 + lx, W), ci0 + c);
            }
        }
        if (vy) {
            const bf16* base = a.dY + ((int64_t)b * H * W) * a.Cout + co0;
#pragma unroll
            for (int k = 0; k < NY; k++) {
                const int v = t + 384 * k, px = v / (MT * 2), c = (v - px * (MT * 2)) * 8, y = y0 + (px >> 4), x = x0 + (px & 15);
                yr[k] = v16{0u, 0u, 0u, 0u};
                if (v < WG_H * 16 * MT * 2 && c < nco && y < H && x < W) yr[k] = *(const v16*)(base + ((int64_t)y * W + x) * a.Cout + c);
            }
        }
    };
    if (t0 < t1) fetch(t0);
    for (int tl = t0; tl < t1; tl++) {
        __syncthreads();
        if (vx) {
#pragma unroll
            for (int k = 0; k < NX; k++) {
                const int v = t + 384 * k;
                if (v < (WG_H + 2) * 18 * 4) *(v16*)(sX + (v >> 2) * WG_XS + (v & 3) * 16) = xr[k];
            }
        } else {
            const int x0 = tl % a.tilesX * 16, y0 = tl / a.tilesX % a.tilesY * WG_H, b = tl / a.tilesX / a.tilesY;
            for (int v = t; v < (WG_H + 2) * 18; v += 384) {
                const int ly = v / 18, lx = v - ly * 18;
                const bf16* src = a.in.at(b, wrapn(y0 - 1 + ly, H), wrapn(x0 - 1 + lx, W), ci0);
                for (int c = 0; c < nci; c++) *(bf16*)(sX + v * WG_XS + 2 * c) = src[c];
            }
        }
        if (vy) {
#pragma unroll
            for (int k = 0; k < NY; k++) {
                const int v = t + 384 * k, px = v / (MT * 2), c = (v - px * (MT * 2)) * 8;
                if (v < WG_H * 16 * MT * 2) *(v16*)(sY + px * YS + 2 * c) = yr[k];
            }
        } else {
            const int x0 = tl % a.tilesX * 16, y0 = tl / a.tilesX % a.tilesY * WG_H, b = tl / a.tilesX / a.tilesY;
            for (int v = t; v < WG_H * 16; v += 384) {
                const int y = y0 + (v >> 4), x = x0 + (v & 15);
                const bool in = y < H && x < W;
                for (int c = 0; c < nco; c++)
                    *(bf16*)(sY + v * YS + 2 * c) = in ? a.dY[(((int64_t)b * H + y) * W + x) * a.Cout + co0 + c] : (bf16)0.0f;
            }
        }
        __syncthreads();
        if (tl + 1 < t1) fetch(tl + 1);
#pragma unroll
        for (int s = 0; s < WG_H / 2; s++) {
            const int row = 2 * s + (q >> 1), px = (q & 1) * 8 + (i >> 2);
            const char* py = sY + (row * 16 + px) * YS + (i & 3) * 8;
            const char* pxx = sX + (row * 18 + px) * WG_XS + (i & 3) * 8;
            bf16x8 yf[MT];
#pragma unroll
            for (int m = 0; m < MT; m++) yf[m] = tr8(py + m * 32, 4 * YS);
#pragma unroll
            for (int n = 0; n < 3; n++) {
                if (!use[n]) continue;
                const bf16x8 xf = tr8(pxx + xo[n], 4 * WG_XS);
#pragma unroll
                for (int m = 0; m < MT; m++)
                    acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yf[m], xf, acc[n][m], 0, 0, 0);
            }
            if (bias)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    accb[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yf[m], ones, accb[m], 0, 0, 0);
        }
    }
    const int64_t ncol = (int64_t)nkk * a.Cin + 1;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int co = co0 + 16 * m + 4 * q + e;
            if (co >= a.Cout) continue;
            float* o = a.part + ((int64_t)blockIdx.x * a.Cout + co) * ncol;
#pragma unroll
            for (int n = 0; n < 3; n++) {
                const int id = 3 * w + n, c = (id & 1) * 16 + i;
                if (use[n] && c < nci) o[(id >> 1) * a.Cin + ci0 + c] = acc[n][m][e];
            }
            if (bias && i == 0) o[ncol - 1] = accb[m][e];
        }
}

// Pixel splits of a layer's weight gradient: two blocks per CU, at most 4 M
// partial sums (three and 8 M: 2.08 ms per training step on eight 256 x 256
// images instead of 2.04, twice the sums to write and add), at most one split
// per pixel tile.
inline int wg_cap(int Cin, int Cout, int ksz) {
    const int64_t blocks = (int64_t)((Cin + 31) / 32) * conv_chunks(Cout);
    const int64_t n = ((int64_t)ksz * ksz * Cin + 1) * Cout;
    return (int)std::max<int64_t>(1, std::min<int64_t>(512 / blocks + 1, ((int64_t)4 << 20) / n));
}
inline void launch_convw(WgArgs a, hipStream_t st) {
    a.tilesX = (a.in.W + 15) / 16;
    a.tilesY = (a.in.H + WG_H - 1) / WG_H;
    const dim3 grid(a.nsplit, (a.Cin + 31) / 32, conv_chunks(a.Cout));
    switch (conv_chunk(a.Cout)) {
        case 1: hipLaunchKernelGGL(k_convw<1>, grid, dim3(384), 0, st, a); break;
        case 2: hipLaunchKernelGGL(k_convw<2>, grid, dim3(384), 0, st, a); break;
        case 3: hipLaunchKernelGGL(k_convw<3>, grid, dim3(384), 0, st, a); break;
        case 4: hipLaunchKernelGGL(k_convw<4>, grid, dim3(384), 0, st, a); break;
        default: hipLaunchKernelGGL(k_convw<6>, grid, dim3(384), 0, st, a); break;
    }
}

// The gradients of all layers (blockIdx.y) from their splits' partial sums: a
// block takes 32 neighbouring sums, thread (e, k) the splits k, k + 8, ... of
// sum e, and the eight parts are added by a fixed tree.
struct SumJob {
    int64_t part, woff, boff;
    int cin, cout, nkk, nsplit;
};
struct SumJobs {
    SumJob j[MAX_JOBS / 2];
};
__global__ void __launch_bounds__(256) k_wsum(const float* __restrict__ part, float* __restrict__ G, SumJobs J) {
    __shared__ float sm[8][32];
    const SumJob& j = J.j[blockIdx.y];
    const int64_t ncol = (int64_t)j.nkk * j.cin + 1, n = ncol * j.cout;
    const int e = threadIdx.x & 31, k0 = threadIdx.x >> 5;
    const int64_t v = (int64_t)blockIdx.x * 32 + e;
    if ((int64_t)blockIdx.x * 32 >= n) return;  // whole blocks
    float s = 0.0f;
    if (v < n) {
        const float* p = part + j.part + v;
#pragma unroll 8
        for (int k = k0; k < j.nsplit; k += 8) s += p[k * n];
    }
    sm[k0][e] = s;
    __syncthreads();
    if (k0 || v >= n) return;
    s = ((sm[0][e] + sm[1][e]) + (sm[2][e] + sm[3][e])) + ((sm[4][e] + sm[5][e]) + (sm[6][e] + sm[7][e]));
    const int64_t co = v / ncol, col = v - co * ncol;
    if (col == ncol - 1) {
        G[j.boff + co] = s;
    } else {
        const int64_t kk = col / j.cin, ci = col - kk * j.cin;
        G[j.woff + (kk * j.cout + co) * j.cin + ci] = s;
    }
}

// ---------------------------------------------------------------- small kernels
__global__ void k_f2bf(const float* in, bf16* out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (bf16)in[i];
}

// 2x2 average pool (NHWC), eight channels per thread: out [B][H/2][W/2][C]
__global__ void __launch_bounds__(256) k_pool(const bf16* in, bf16* out, int B, int H, int W, int C) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int h = H / 2, w = W / 2, C8 = C / 8;
    if (v >= (int64_t)B * h * w * C8) return;
    const int c = (int)(v % C8) * 8;
    const int64_t p = v / C8;
    const int x = (int)(p % w), y = (int)(p / w % h), b = (int)(p / w / h);
    const bf16* s = in + (((int64_t)b * H + 2 * y) * W + 2 * x) * C + c;
    const bf16x8 a0 = *(const bf16x8*)s, a1 = *(const bf16x8*)(s + C), a2 = *(const bf16x8*)(s + (int64_t)W * C),
                 a3 = *(const bf16x8*)(s + (int64_t)W * C + C);
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = (bf16)(0.25f * ((float)a0[e] + (float)a1[e] + (float)a2[e] + (float)a3[e]));
    *(bf16x8*)(out + p * C + c) = r;
}

// Gradient operands where parts are summed, eight channels per thread, FP32
// until the rounding, the ReLU mask of y applied.
// k_grad_lo: the upsampled part [0, C1) of a concatenated input's gradient g
// [B][H][W][C1 + C2], summed over the four children -> out [B][H/2][W/2][C1].
__global__ void __launch_bounds__(256) k_grad_lo(const float* g, const bf16* y, bf16* out, int B, int H, int W, int C1, int C2) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int h = H / 2, w = W / 2, C8 = C1 / 8, C = C1 + C2;
    if (v >= (int64_t)B * h * w * C8) return;
    const int c = (int)(v % C8) * 8;
    const int64_t p = v / C8;
    const int x = (int)(p % w), yy = (int)(p / w % h), b = (int)(p / w / h);
    const bf16x8 m = *(const bf16x8*)(y + p * C1 + c);
    float s[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int d = 0; d < 4; d++) {
        const float* q = g + (((int64_t)b * H + 2 * yy + (d >> 1)) * W + 2 * x + (d & 1)) * C + c;
        const f32x4 u0 = *(const f32x4*)q, u1 = *(const f32x4*)(q + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s[e] += u0[e];
            s[4 + e] += u1[e];
        }
    }
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = (bf16)((float)m[e] <= 0.0f ? 0.0f : s[e]);
    *(bf16x8*)(out + p * C1 + c) = r;
}
// k_grad_skip: the skip part [C1, C1 + C2) of g plus the gradient of the pooled
// tensor gp [B][H/2][W/2][C2] -> out [B][H][W][C2].
__global__ void __launch_bounds__(256) k_grad_skip(const float* g, const float* gp, const bf16* y, bf16* out, int B, int H,
                                                   int W, int C1, int C2) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int C8 = C2 / 8;
    if (v >= (int64_t)B * H * W * C8) return;
    const int c = (int)(v % C8) * 8;
    const int64_t p = v / C8;
    const int x = (int)(p % W), yy = (int)(p / W % H), b = (int)(p / W / H);
    const float* q = g + p * (C1 + C2) + C1 + c;
    const float* r = gp + (((int64_t)b * (H / 2) + yy / 2) * (W / 2) + x / 2) * C2 + c;
    const bf16x8 m = *(const bf16x8*)(y + p * C2 + c);
    bf16x8 o;
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        const f32x4 u = *(const f32x4*)(q + 4 * hh), w4 = *(const f32x4*)(r + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float s = u[e] + 0.25f * w4[e];
            o[4 * hh + e] = (bf16)((float)m[4 * hh + e] <= 0.0f ? 0.0f : s);
        }
    }
    *(bf16x8*)(out + p * C2 + c) = o;
}

// masked mean-square loss over B*H*W pixels of 2 channels:
// loss = sum m (o - t)^2 / (2 sum m); grad = m (o - t) / sum m.
// Pass 1: per chunk of LOSS_CHUNK pixels, (sum m (o - t)^2, sum m) by a
// fixed tree; pass 2 (one wave): the chunks; pass 3: the gradient.
constexpr int LOSS_CHUNK = 4096;
__global__ void __launch_bounds__(256) k_loss_part(const float* o, const float* t, const float* mask, int64_t P,
                                                   float* part) {
    __shared__ float s[2][256];
    const int tid = threadIdx.x;
    const int64_t p0 = (int64_t)blockIdx.x * LOSS_CHUNK, p1 = min(P, p0 + LOSS_CHUNK);
    float se = 0.0f, sm = 0.0f;
    for (int64_t p = p0 + tid; p < p1; p += 256) {
        const float m = mask[p];
        const float d0 = o[2 * p] - t[2 * p], d1 = o[2 * p + 1] - t[2 * p + 1];
        se += m * (d0 * d0 + d1 * d1);
        sm += m;
    }
    s[0][tid] = se;
    s[1][tid] = sm;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) {
            s[0][tid] += s[0][tid + h];
            s[1][tid] += s[1][tid + h];
        }
        __syncthreads();
    }
    if (tid == 0) {
        part[2 * blockIdx.x] = s[0][0];
        part[2 * blockIdx.x + 1] = s[1][0];
    }
}
// one wave: lane l adds the chunks l, l + 64, ..., then a fixed tree
__global__ void __launch_bounds__(64) k_loss_sum(const float* part, int nchunk, float* out2) {
    float se = 0.0f, sm = 0.0f;
    for (int b = threadIdx.x; b < nchunk; b += 64) {
        se += part[2 * b];
        sm += part[2 * b + 1];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        se += __shfl_xor(se, o, 64);
        sm += __shfl_xor(sm, o, 64);
    }
    if (threadIdx.x) return;
    out2[0] = se / (2.0f * fmaxf(sm, 1.0f));
    out2[1] = sm;
}
// gradient of the loss as the BF16 operand of the head's backward products
__global__ void k_loss_grad(const float* o, const float* t, const float* mask, int64_t P, const float* out2, bf16* grad) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const float m = mask[p] / fmaxf(out2[1], 1.0f);
    grad[2 * p] = (bf16)(m * (o[2 * p] - t[2 * p]));
    grad[2 * p + 1] = (bf16)(m * (o[2 * p + 1] - t[2 * p + 1]));
}

__global__ void k_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi, vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline unsigned nblk(int64_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

}  // namespace net

using namespace net;

// ---------------------------------------------------------------- the network
struct ConvL {
    int cin, cout, ksz, relu;
    int64_t woff, boff;  // offsets in the parameter array
};
struct Tens {
    int C = 0, level = 0;  // level: resolution H >> level
    bf16* a = nullptr;     // activation (the decoder's concatenated inputs have none)
    float* g = nullptr;    // FP32 gradient (concatenated and pooled tensors)
};

struct mts_net_s {
    hipStream_t stream = nullptr;
    int c[4];
    int maxB = 0, maxH = 0, maxW = 0;
    std::vector<ConvL> L;
    int64_t nparam = 0;
    float *P = nullptr, *G = nullptr, *Mo = nullptr, *Vo = nullptr;
    bf16* Wp = nullptr;   // packed BF16 weights of both directions (k_pack)
    int64_t wp_n = 0;
    std::vector<int64_t> wf, wb;  // offsets of each layer's forward and backward weights in Wp
    std::vector<int64_t> wpart;   // and of its weight-gradient partials in part
    // tensors
    enum {
        X0, E0A, E0, P0, E1A, E1, P1, E2A, E2, P2, E3A, E3, C2, D2A, D2, C1, D1A, D1, C0, D0A, D0, NT
    };
    Tens T[NT];
    float* out = nullptr;         // [B][H][W][2]
    bf16* gb[2] = {nullptr, nullptr};  // BF16 gradient operands (a layer's own and the next one's)
    float* part = nullptr;        // weight-gradient partials, one region per layer
    float* loss = nullptr;  // 2 floats
    float* red = nullptr;   // partial sums of the loss
    int B = 0, H = 0, W = 0;
    std::vector<void*> allocs;
    template <class Tp>
    int alloc(Tp** p, size_t n) {
        void* q = nullptr;
        hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(Tp));
        if (e != hipSuccess) {
            (void)hipGetLastError();  // a failed allocation must not surface at a later launch check
            return set_error(MTS_ERR_OOM, std::string("hipMalloc: ") + hipGetErrorString(e));
        }
        allocs.push_back(q);
        *p = (Tp*)q;
        return MTS_OK;
    }
    ~mts_net_s() {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void* q : allocs) (void)hipFree(q);
        if (stream) (void)hipStreamDestroy(stream);
    }
    int64_t npix(int level) const { return (int64_t)B * (H >> level) * (W >> level); }
    // BF16 copies of the FP32 weights in the products' order
    void refresh_bf16() {
        PackJobs J{};
        int64_t most = 0;
        for (size_t i = 0; i < L.size(); i++) {
            const ConvL& l = L[i];
            J.j[2 * i] = PackJob{l.woff, wf[i], l.cin, l.cout, l.ksz, 0};
            J.j[2 * i + 1] = PackJob{l.woff, wb[i], l.cin, l.cout, l.ksz, 1};
            most = std::max({most, conv_pack_elems(l.cin, l.cout, l.ksz), conv_pack_elems(l.cout, l.cin, l.ksz)});
        }
        hipLaunchKernelGGL(k_pack, dim3(nblk(most), (unsigned)(2 * L.size())), dim3(256), 0, stream, P, Wp, J);
    }
    // input of a layer: a tensor, or `lo` upsampled next to `skip`
    ConvIn input(const Tens& x) const { return ConvIn{x.a, nullptr, x.C, 0, 0, H >> x.level, W >> x.level}; }
    ConvIn input(const Tens& lo, const Tens& skip) const {
        return ConvIn{lo.a, skip.a, lo.C, skip.C, 1, H >> skip.level, W >> skip.level};
    }
    int conv_fwd(int li, const ConvIn& in, bf16* y, float* yf) {
        const ConvL& l = L[li];
        ConvArgs a{};
        a.in = in;
        a.Cin = l.cin;
        a.Cout = l.cout;
        a.ksz = l.ksz;
        a.sgn = 1;
        a.Wf = Wp + wf[li];
        a.bias = P + l.boff;
        a.relu = l.relu;
        a.Y = y;
        a.Yf = yf;
        return launch_conv(a, B, stream);
    }
    // weight and bias gradient partials of layer li from its input and the
    // gradient gb[k] of its output; the gradient of its input goes to gin
    // (FP32), or to gb[k ^ 1] with the ReLU mask of `mask`, or nowhere
    int conv_bwd(int li, const ConvIn& in, int k, const bf16* mask, float* gin) {
        const ConvL& l = L[li];
        WgArgs w{in, gb[k], part + wpart[li], l.cin, l.cout, l.ksz, B, 0, 0, nsplit(li)};
        launch_convw(w, stream);
        if (!mask && !gin) return 0;
        ConvArgs a{};
        a.in = ConvIn{gb[k], nullptr, l.cout, 0, 0, in.H, in.W};
        a.Cin = l.cout;
        a.Cout = l.cin;
        a.ksz = l.ksz;
        a.sgn = -1;
        a.Wf = Wp + wb[li];
        a.mask = mask;
        a.Y = gb[k ^ 1];
        a.Yf = gin;
        return launch_conv(a, B, stream);
    }
    int nsplit(int li) const;
    void sum_grads() {
        SumJobs J{};
        int64_t most = 0;
        for (size_t i = 0; i < L.size(); i++) {
            const ConvL& l = L[i];
            J.j[i] = SumJob{wpart[i], l.woff, l.boff, l.cin, l.cout, l.ksz * l.ksz, nsplit((int)i)};
            most = std::max(most, ((int64_t)l.ksz * l.ksz * l.cin + 1) * l.cout);
        }
        hipLaunchKernelGGL(k_wsum, dim3(nblk(most, 32), (unsigned)L.size()), dim3(256), 0, stream, part, G, J);
    }
};

namespace {

int check_net(mts_net n) { return n ? MTS_OK : set_error(MTS_ERR_ARG, "null network handle"); }

// resolution level of each layer's input: two convolutions per encoder level
// 0..3, two per decoder level 2..0, then the 1x1 head at level 0
int layer_level(size_t i) {
    static const int level[15] = {0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0};
    return i < 15 ? level[i] : 0;
}

}  // namespace

int mts_net_s::nsplit(int li) const {
    const int h = H >> layer_level(li), w = W >> layer_level(li);
    const int64_t tiles = (int64_t)((w + 15) / 16) * ((h + WG_H - 1) / WG_H) * B;
    return (int)std::min<int64_t>(tiles, wg_cap(L[li].cin, L[li].cout, L[li].ksz));
}

namespace {

// layer table of the U-Net (widths c0..c3, input 3 channels, output 2)
void layers(mts_net_s* n) {
    const int* c = n->c;
    const int spec[15][4] = {{3, c[0], 3, 1},          {c[0], c[0], 3, 1},        {c[0], c[1], 3, 1},
                             {c[1], c[1], 3, 1},       {c[1], c[2], 3, 1},        {c[2], c[2], 3, 1},
                             {c[2], c[3], 3, 1},       {c[3], c[3], 3, 1},        {c[3] + c[2], c[2], 3, 1},
                             {c[2], c[2], 3, 1},       {c[2] + c[1], c[1], 3, 1}, {c[1], c[1], 3, 1},
                             {c[1] + c[0], c[0], 3, 1}, {c[0], c[0], 3, 1},       {c[0], 2, 1, 0}};
    int64_t off = 0;
    for (auto& s : spec) {
        ConvL l{s[0], s[1], s[2], s[3], 0, 0};
        l.woff = off;
        off += (int64_t)l.ksz * l.ksz * l.cout * l.cin;
        l.boff = off;
        off += l.cout;
        n->L.push_back(l);
    }
    n->nparam = off;
}

}  // namespace

extern "C" {

int mts_net_create(int c0, int max_batch, int max_h, int max_w, uint64_t seed, mts_net* out) {
    // c0 % 8 == 0 keeps every layer's weights 16-byte aligned for the vector loads
    if (!out || c0 <= 0 || c0 % 8 || max_batch <= 0 || max_h <= 0 || max_w <= 0 || max_h % 8 || max_w % 8)
        return set_error(MTS_ERR_ARG, "bad network shape (c0 and the sizes must be multiples of 8)");
    *out = nullptr;
    mts_net_s* n = new (std::nothrow) mts_net_s();
    if (!n) return set_error(MTS_ERR_OOM, "host allocation");
    auto bail = [&](int rc) {
        delete n;
        return rc;
    };
    n->c[0] = c0;
    n->c[1] = 2 * c0;
    n->c[2] = 4 * c0;
    n->c[3] = 8 * c0;
    n->maxB = max_batch;
    n->maxH = max_h;
    n->maxW = max_w;
    layers(n);
    hipError_t e = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking);
    if (e != hipSuccess) return bail(set_error(MTS_ERR_HIP, std::string("stream: ") + hipGetErrorString(e)));
    int rc;
    const int64_t np = n->nparam;
    if ((rc = n->alloc(&n->P, np)) || (rc = n->alloc(&n->G, np)) || (rc = n->alloc(&n->Mo, np)) ||
        (rc = n->alloc(&n->Vo, np)))
        return bail(rc);
    // tensors: channels and level
    const int* c = n->c;
    const int tc[mts_net_s::NT][2] = {{3, 0},        {c[0], 0}, {c[0], 0},         {c[0], 1}, {c[1], 1},
                                      {c[1], 1},     {c[1], 2}, {c[2], 2},         {c[2], 2}, {c[2], 3},
                                      {c[3], 3},     {c[3], 3}, {c[3] + c[2], 2},  {c[2], 2}, {c[2], 2},
                                      {c[2] + c[1], 1}, {c[1], 1}, {c[1], 1},      {c[1] + c[0], 0}, {c[0], 0},
                                      {c[0], 0}};
    int64_t maxe = 0;
    for (int t = 0; t < mts_net_s::NT; t++) {
        Tens& T = n->T[t];
        T.C = tc[t][0];
        T.level = tc[t][1];
        const int64_t ne = (int64_t)max_batch * (max_h >> T.level) * (max_w >> T.level) * T.C;
        const bool cat = t == mts_net_s::C0 || t == mts_net_s::C1 || t == mts_net_s::C2;
        const bool pooled = t == mts_net_s::P0 || t == mts_net_s::P1 || t == mts_net_s::P2;
        if (!cat) maxe = std::max(maxe, ne);
        if ((!cat && (rc = n->alloc(&T.a, ne))) || ((cat || pooled) && (rc = n->alloc(&T.g, ne)))) return bail(rc);
    }
    const int64_t P0 = (int64_t)max_batch * max_h * max_w;
    int64_t pn = 0;
    for (const ConvL& l : n->L) {  // packed weights and weight-gradient partials of each layer
        n->wf.push_back(n->wp_n);
        n->wp_n += conv_pack_elems(l.cin, l.cout, l.ksz);
        n->wb.push_back(n->wp_n);
        n->wp_n += conv_pack_elems(l.cout, l.cin, l.ksz);
        n->wpart.push_back(pn);
        pn += ((int64_t)l.ksz * l.ksz * l.cin + 1) * l.cout * wg_cap(l.cin, l.cout, l.ksz);
    }
    if ((rc = n->alloc(&n->out, P0 * 2)) || (rc = n->alloc(&n->gb[0], maxe)) || (rc = n->alloc(&n->gb[1], maxe)) ||
        (rc = n->alloc(&n->Wp, n->wp_n)) || (rc = n->alloc(&n->part, pn)) || (rc = n->alloc(&n->loss, 2)) ||
        (rc = n->alloc(&n->red, (P0 + LOSS_CHUNK - 1) / LOSS_CHUNK * 2)))
        return bail(rc);
    // He-normal weights, zero biases, zero Adam moments
    std::vector<float> h(np, 0.0f);
    std::mt19937_64 rng(seed);
    for (const ConvL& l : n->L) {
        std::normal_distribution<float> nd(0.0f, std::sqrt(2.0f / (float)(l.cin * l.ksz * l.ksz)));
        const float sc = l.relu ? 1.0f : 0.1f;  // small head: the first predictions stay near zero
        for (int64_t i = 0; i < (int64_t)l.ksz * l.ksz * l.cout * l.cin; i++) h[l.woff + i] = sc * nd(rng);
    }
    if ((e = hipMemcpy(n->P, h.data(), np * 4, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemset(n->Mo, 0, np * 4)) != hipSuccess || (e = hipMemset(n->Vo, 0, np * 4)) != hipSuccess ||
        (e = hipMemset(n->G, 0, np * 4)) != hipSuccess)
        return bail(set_error(MTS_ERR_HIP, std::string("init: ") + hipGetErrorString(e)));
    n->refresh_bf16();
    if ((e = hipStreamSynchronize(n->stream)) != hipSuccess)
        return bail(set_error(MTS_ERR_HIP, std::string("init: ") + hipGetErrorString(e)));
    *out = n;
    return MTS_OK;
}

int mts_net_destroy(mts_net n) {
    delete n;
    return MTS_OK;
}

int mts_net_flops(mts_net n, int B, int H, int W, double* fwd) {
    if (int rc = check_net(n)) return rc;
    if (!fwd || B <= 0 || H <= 0 || W <= 0) return set_error(MTS_ERR_ARG, "bad argument");
    double f = 0.0;
    for (size_t i = 0; i < n->L.size(); i++) {
        const ConvL& l = n->L[i];
        const int lv = layer_level(i);
        f += 2.0 * B * (double)(H >> lv) * (double)(W >> lv) * l.cin * l.cout * l.ksz * l.ksz;
    }
    *fwd = f;
    return MTS_OK;
}

int mts_net_param_count(mts_net n, int64_t* count) {
    if (int rc = check_net(n)) return rc;
    if (!count) return set_error(MTS_ERR_ARG, "null argument");
    *count = n->nparam;
    return MTS_OK;
}

int mts_net_get_params(mts_net n, float* host) {
    if (int rc = check_net(n)) return rc;
    if (!host) return set_error(MTS_ERR_ARG, "null argument");
    NET_TRY(hipMemcpyAsync(host, n->P, n->nparam * 4, hipMemcpyDeviceToHost, n->stream));
    NET_TRY(hipStreamSynchronize(n->stream));
    return MTS_OK;
}

int mts_net_set_params(mts_net n, const float* host) {
    if (int rc = check_net(n)) return rc;
    if (!host) return set_error(MTS_ERR_ARG, "null argument");
    NET_TRY(hipMemcpyAsync(n->P, host, n->nparam * 4, hipMemcpyHostToDevice, n->stream));
    n->refresh_bf16();
    NET_TRY(hipStreamSynchronize(n->stream));
    return MTS_OK;
}

int mts_net_get_grads(mts_net n, float* host) {
    if (int rc = check_net(n)) return rc;
    if (!host) return set_error(MTS_ERR_ARG, "null argument");
    NET_TRY(hipMemcpyAsync(host, n->G, n->nparam * 4, hipMemcpyDeviceToHost, n->stream));
    NET_TRY(hipStreamSynchronize(n->stream));
    return MTS_OK;
}

int mts_net_forward(mts_net n, const float* in, int B, int H, int W, float* out) {
    if (int rc = check_net(n)) return rc;
    if (!in || B <= 0 || B > n->maxB || H <= 0 || W <= 0 || H > n->maxH || W > n->maxW || H % 8 || W % 8 ||
        (int64_t)H * W * B > (int64_t)n->maxH * n->maxW * n->maxB)
        return set_error(MTS_ERR_ARG, "input shape exceeds the network's buffers or is not a multiple of 8");
    n->B = B;
    n->H = H;
    n->W = W;
    hipStream_t st = n->stream;
    auto& T = n->T;
    const int64_t p0 = n->npix(0);
    hipLaunchKernelGGL(k_f2bf, dim3(nblk(p0 * 3)), dim3(256), 0, st, in, T[mts_net_s::X0].a, p0 * 3);
    typedef mts_net_s S;
    auto pool = [&](int a, int b) {
        const Tens& x = T[a];
        hipLaunchKernelGGL(k_pool, dim3(nblk(n->npix(x.level + 1) * x.C / 8)), dim3(256), 0, st, x.a, T[b].a, B,
                           H >> x.level, W >> x.level, x.C);
    };
    int rc = 0;
    auto conv = [&](int li, int x, int y) { rc = rc ? rc : n->conv_fwd(li, n->input(T[x]), T[y].a, nullptr); };
    auto conv_cat = [&](int li, int lo, int skip, int y) {
        rc = rc ? rc : n->conv_fwd(li, n->input(T[lo], T[skip]), T[y].a, nullptr);
    };
    conv(0, S::X0, S::E0A);
    conv(1, S::E0A, S::E0);
    pool(S::E0, S::P0);
    conv(2, S::P0, S::E1A);
    conv(3, S::E1A, S::E1);
    pool(S::E1, S::P1);
    conv(4, S::P1, S::E2A);
    conv(5, S::E2A, S::E2);
    pool(S::E2, S::P2);
    conv(6, S::P2, S::E3A);
    conv(7, S::E3A, S::E3);
    conv_cat(8, S::E3, S::E2, S::D2A);
    conv(9, S::D2A, S::D2);
    conv_cat(10, S::D2, S::E1, S::D1A);
    conv(11, S::D1A, S::D1);
    conv_cat(12, S::D1, S::E0, S::D0A);
    conv(13, S::D0A, S::D0);
    rc = rc ? rc : n->conv_fwd(14, n->input(T[S::D0]), nullptr, n->out);
    NET_TRY((hipError_t)rc);
    if (out) NET_TRY(hipMemcpyAsync(out, n->out, p0 * 2 * 4, hipMemcpyDeviceToDevice, st));
    NET_TRY(hipGetLastError());
    NET_TRY(hipStreamSynchronize(st));
    return MTS_OK;
}

int mts_net_backward(mts_net n, const float* target, const float* mask, float* loss_host) {
    if (int rc = check_net(n)) return rc;
    if (!target || !mask || n->B == 0) return set_error(MTS_ERR_ARG, "run mts_net_forward first");
    hipStream_t st = n->stream;
    auto& T = n->T;
    typedef mts_net_s S;
    const int B = n->B, H = n->H, W = n->W;
    const int64_t p0 = n->npix(0);
    const int nlc = (int)((p0 + LOSS_CHUNK - 1) / LOSS_CHUNK);
    hipLaunchKernelGGL(k_loss_part, dim3(nlc), dim3(256), 0, st, n->out, target, mask, p0, n->red);
    hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(64), 0, st, n->red, nlc, n->loss);
    hipLaunchKernelGGL(k_loss_grad, dim3(nblk(p0)), dim3(256), 0, st, n->out, target, mask, p0, n->loss, n->gb[0]);
    // head, then decoder, then encoder (reverse order of the forward pass);
    // k: which of the gradient operands is the current one
    int rc = 0, k = 0;
    // a layer whose input is an activation: its gradient is the next operand
    auto conv = [&](int li, int x) {
        rc = rc ? rc : n->conv_bwd(li, n->input(T[x]), k, T[x].a, nullptr);
        k ^= 1;
    };
    auto conv_cat = [&](int li, int lo, int skip, int cat) {  // then the upsampled part's operand
        rc = rc ? rc : n->conv_bwd(li, n->input(T[lo], T[skip]), k, nullptr, T[cat].g);
        k ^= 1;
        const Tens &x = T[lo], &s = T[skip];
        hipLaunchKernelGGL(k_grad_lo, dim3(nblk(n->npix(x.level) * x.C / 8)), dim3(256), 0, st, T[cat].g, x.a, n->gb[k], B,
                           H >> s.level, W >> s.level, x.C, s.C);
    };
    auto conv_pool = [&](int li, int pooled, int x, int lo, int cat) {  // then the operand of the pooled tensor x
        rc = rc ? rc : n->conv_bwd(li, n->input(T[pooled]), k, nullptr, T[pooled].g);
        k ^= 1;
        const Tens& t = T[x];
        hipLaunchKernelGGL(k_grad_skip, dim3(nblk(n->npix(t.level) * t.C / 8)), dim3(256), 0, st, T[cat].g, T[pooled].g, t.a,
                           n->gb[k], B, H >> t.level, W >> t.level, T[lo].C, t.C);
    };
    conv(14, S::D0);
    conv(13, S::D0A);
    conv_cat(12, S::D1, S::E0, S::C0);
    conv(11, S::D1A);
    conv_cat(10, S::D2, S::E1, S::C1);
    conv(9, S::D2A);
    conv_cat(8, S::E3, S::E2, S::C2);
    conv(7, S::E3A);
    conv_pool(6, S::P2, S::E2, S::E3, S::C2);
    conv(5, S::E2A);
    conv_pool(4, S::P1, S::E1, S::D2, S::C1);
    conv(3, S::E1A);
    conv_pool(2, S::P0, S::E0, S::D1, S::C0);
    conv(1, S::E0A);
    rc = rc ? rc : n->conv_bwd(0, n->input(T[S::X0]), k, nullptr, nullptr);
    n->sum_grads();
    NET_TRY((hipError_t)rc);
    NET_TRY(hipGetLastError());
    float l2[2];
    NET_TRY(hipMemcpyAsync(l2, n->loss, 8, hipMemcpyDeviceToHost, st));
    NET_TRY(hipStreamSynchronize(st));
    if (loss_host) *loss_host = l2[0];
    return MTS_OK;
}

int mts_net_adam(mts_net n, float lr, float beta1, float beta2, float eps, int step) {
    if (int rc = check_net(n)) return rc;
    if (step < 1) return set_error(MTS_ERR_ARG, "Adam step counts from 1");
    const float c1 = 1.0f - std::pow(beta1, (float)step), c2 = 1.0f - std::pow(beta2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(n->nparam)), dim3(256), 0, n->stream, n->P, n->G, n->Mo, n->Vo, n->nparam, lr,
                       beta1, beta2, eps, c1, c2);
    n->refresh_bf16();
    NET_TRY(hipGetLastError());
    NET_TRY(hipStreamSynchronize(n->stream));
    return MTS_OK;
}

// C = A B on dense host matrices (A: M x K, B: K x N, row-major, rounded to
// BF16 on the device) as the layers compute it: a 1x1 convolution of M pixels
// with K input and N output channels (K padded with zeros to whole vectors).
int mts_net_gemm_check(const float* A, const float* Bm, int M, int N, int K, float* C) {
    if (!A || !Bm || !C || M <= 0 || N <= 0 || K <= 0 || (int64_t)M * N > (1 << 24) || (int64_t)M * K > (1 << 24) ||
        (int64_t)K * N > (1 << 24))
        return set_error(MTS_ERR_ARG, "bad GEMM check shape");
    const int Kp = (K + 7) / 8 * 8;
    std::vector<float> a, w;  // A padded; B as weights [N][Kp]
    try {
        a.assign((size_t)M * Kp, 0.0f);
        w.assign((size_t)N * Kp, 0.0f);
    } catch (...) {
        return set_error(MTS_ERR_OOM, "host allocation");
    }
    for (int m = 0; m < M; m++) std::copy(A + (size_t)m * K, A + (size_t)(m + 1) * K, &a[(size_t)m * Kp]);
    for (int k = 0; k < K; k++)
        for (int n = 0; n < N; n++) w[(size_t)n * Kp + k] = Bm[(size_t)k * N + n];
    mts_net_s d;  // owns the buffers and the stream
    float *dA, *dW, *dC;
    bf16 *hA, *hW;
    NET_TRY(hipStreamCreateWithFlags(&d.stream, hipStreamNonBlocking));
    const int64_t nw = conv_pack_elems(Kp, N, 1);
    int rc;
    if ((rc = d.alloc(&dA, a.size())) || (rc = d.alloc(&dW, w.size())) || (rc = d.alloc(&dC, (size_t)M * N)) ||
        (rc = d.alloc(&hA, a.size())) || (rc = d.alloc(&hW, nw)))
        return rc;
    NET_TRY(hipMemcpyAsync(dA, a.data(), a.size() * 4, hipMemcpyHostToDevice, d.stream));
    NET_TRY(hipMemcpyAsync(dW, w.data(), w.size() * 4, hipMemcpyHostToDevice, d.stream));
    hipLaunchKernelGGL(k_f2bf, dim3(nblk((int64_t)a.size())), dim3(256), 0, d.stream, dA, hA, (int64_t)a.size());
    PackJobs J{};
    J.j[0] = PackJob{0, 0, Kp, N, 1, 0};
    hipLaunchKernelGGL(k_pack, dim3(nblk(nw), 1), dim3(256), 0, d.stream, dW, hW, J);
    ConvArgs c{};
    c.in = ConvIn{hA, nullptr, Kp, 0, 0, 1, M};
    c.Cin = Kp;
    c.Cout = N;
    c.ksz = 1;
    c.sgn = 1;
    c.Wf = hW;
    c.Yf = dC;
    NET_TRY((hipError_t)launch_conv(c, 1, d.stream));
    NET_TRY(hipGetLastError());
    NET_TRY(hipMemcpyAsync(C, dC, (size_t)M * N * 4, hipMemcpyDeviceToHost, d.stream));
    NET_TRY(hipStreamSynchronize(d.stream));
    return MTS_OK;
}

int mts_net_stream(mts_net n, void** stream) {
    if (int rc = check_net(n)) return rc;
    if (!stream) return set_error(MTS_ERR_ARG, "null argument");
    *stream = (void*)n->stream;
    return MTS_OK;
}

}  // extern "C"
