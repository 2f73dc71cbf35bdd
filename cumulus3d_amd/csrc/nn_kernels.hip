// nn_kernels.hip — kernels of the learned initialiser: a small U-Net in bf16 with fp32
// accumulation on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16), its backward pass, Adam,
// the training loss against plain-PatchStereo labels and the plane-sweep input features.
//
// Convolutions are implicit GEMMs over NHWC tensors: a workgroup stages a tile of pixels with its
// halo in LDS, from where its four waves read the pixels of every tap as one MFMA operand; the weights, packed in the order the lanes take them, come from L2 as the other.
// The weight gradient reduces over pixels, the MFMA's K dimension, through transposing LDS reads.
#include "nn_kernels.hpp"

#include <algorithm>

namespace c3d {
namespace nn {

typedef short s16x8 __attribute__((__vector_size__(16)));
typedef short s16x4 __attribute__((__vector_size__(8)));
typedef float f32x4 __attribute__((__vector_size__(16)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ f32x4 mfma(s16x8 a, s16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Pixel index of (gy, gx) of an image of H x W in a tensor of that size, or (up) in one of half the
// size that is upsampled to it by repetition.
__device__ __forceinline__ size_t source_pixel(int img, int gy, int gx, int H, int W, int up) {
    return up ? (size_t)(img * (H / 2) + gy / 2) * (W / 2) + gx / 2 : (size_t)(img * H + gy) * W + gx;
}

// ---------------------------------------------------------------- convolution (forward / data gradient)

// A workgroup computes 16 x 4R pixels x 16 NT output channels: wave w the rows w R .. w R + R - 1. It
// stages the tile and its halo, all input channels (groups of 32 one after another, so that the 64
// lanes read 64 bytes a pixel without bank conflicts). The weights are the MFMA's first operand, so
// that a lane ends with four channels of one pixel and stores them at once; those of the next step
// are loaded while a step's are used. Every output accumulates tap by tap and 32 channels at a
// time in the same order, so R and NT change no result.
//
// What bounds it: the layers are small (0.3 to 15 GFLOP), so the latency of the staging and the
// stores count as much as the matrix cores; at R = 4, NT = 4 these could be kept half busy by LDS
// and fully by L1. Reading each tap's pixels from L1 instead, 16 or 64 pixels a wave, left them at
// 130 TFLOP/s: the forward pass of 6 images of 480 x 272 took 1.48 ms of convolutions, now 0.60 (350
// TFLOP/s), a training step of 8 images 3.70, now 1.25.
template <int KS, int R, int NT>
__global__ __launch_bounds__(256) void k_conv(ConvArgs a) {
    constexpr int HALO = KS / 2, TAPS = KS * KS;
    constexpr int TW = 16 + 2 * HALO, TH = 4 * R + 2 * HALO, NPX = TW * TH;
    constexpr int NLD = (NPX * 4 + 255) / 256;  // 16-byte loads a thread per 32 channels
    extern __shared__ __attribute__((aligned(16))) uint16_t tile[];  // [cin / 32][NPX][32]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int tx = (a.W + 15) / 16, ty = (a.H + 4 * R - 1) / (4 * R);
    const int img = (int)(blockIdx.x / (unsigned)(tx * ty)), rest = (int)(blockIdx.x % (unsigned)(tx * ty));
    const int y0 = rest / tx * (4 * R), x0 = rest % tx * 16;
    const int ct0 = blockIdx.y * NT;
    const int nc = a.cin / 32;
    {
        int pix[NLD], pix2[NLD];  // the pixel of each of this thread's loads in x and x2, -1 outside the image
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
            const int e = threadIdx.x + 256 * j, p = e >> 2;
            const int gy = y0 + p / TW - HALO, gx = x0 + p % TW - HALO;
            const bool in = e < NPX * 4 && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W;
            pix[j] = in ? (int)source_pixel(img, gy, gx, a.H, a.W, a.up) : -1;
            pix2[j] = in ? (int)source_pixel(img, gy, gx, a.H, a.W, 0) : -1;
        }
#pragma unroll 2
        for (int c = 0; c < nc; ++c) {
            const bool first = c * 32 < a.c1;  // channels of x, else of x2
            const uint16_t* src = (first ? a.x + c * 32 : a.x2 + (c * 32 - a.c1)) + (threadIdx.x & 3) * 8;
            const int xs = first ? a.c1 : a.cin - a.c1;
            s16x8 v[NLD];
#pragma unroll
            for (int j = 0; j < NLD; ++j) {
                const int p = first ? pix[j] : pix2[j];
                v[j] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if (p >= 0) v[j] = *(const s16x8*)(src + (size_t)p * xs);
            }
#pragma unroll
            for (int j = 0; j < NLD; ++j)
                if ((int)threadIdx.x + 256 * j < NPX * 4) *(s16x8*)&tile[(size_t)c * NPX * 32 + (threadIdx.x + 256 * j) * 8] = v[j];
        }
    }
    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[r][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint16_t* w = a.w + (size_t)ct0 * 512 + lane * 8;
    s16x8 wn[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wn[n] = *(const s16x8*)(w + n * 512);
    __syncthreads();
    int left = TAPS * nc;
    for (int dy = 0; dy < KS; ++dy)
        for (int dx = 0; dx < KS; ++dx) {
            const uint16_t* t = tile + ((wave * R + dy) * TW + r16 + dx) * 32 + kg * 8;
#pragma unroll 1
            for (int c = 0; c < nc; ++c, t += NPX * 32) {
                s16x8 X[R], wc[NT];
#pragma unroll
                for (int r = 0; r < R; ++r) X[r] = *(const s16x8*)(t + r * TW * 32);
#pragma unroll
                for (int n = 0; n < NT; ++n) wc[n] = wn[n];
                if (--left > 0) {
                    w += (size_t)a.ctiles * 512;
#pragma unroll
                    for (int n = 0; n < NT; ++n) wn[n] = *(const s16x8*)(w + n * 512);
                }
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r][n] = mfma(wc[n], X[r], acc[r][n]);
            }
        }
    // lane holds pixel r16 of each row and channels 4 kg .. 4 kg + 3 of each 16
    const int x = x0 + r16;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int co = (ct0 + n) * 16 + 4 * kg;
        const f32x4 b = a.bias ? *(const f32x4*)(a.bias + co) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = y0 + wave * R + r;
            if (x >= a.W || y >= a.H) continue;
            const size_t p = (size_t)(img * a.H + y) * a.W + x;
            f32x4 v = acc[r][n] + b;
            if (a.y32) {
                *(f32x4*)(a.y32 + p * a.y32s + co) = v;
            } else {
                s16x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = (short)f2bf(a.relu ? fmaxf(v[j], 0.f) : v[j]);
                *(s16x4*)(a.y + p * a.ys + co) = o;
            }
        }
    }
}

template <int KS, int R, int NT>
static void launch_conv_rows(const ConvArgs& a, unsigned blocks, unsigned ny, size_t lds, hipStream_t s) {
    hipLaunchKernelGGL((k_conv<KS, R, NT>), dim3(blocks, ny), dim3(256), lds, s, a);
}

// Taller tiles stage less halo and use each weight for more pixels; smaller ones are taken where a
// launch would otherwise have fewer than two workgroups per CU, or one CU's LDS no room for two.
template <int KS, int NT>
static void launch_conv(const ConvArgs& a, hipStream_t s) {
    const unsigned tx = (unsigned)((a.W + 15) / 16), ny = (unsigned)(a.cout / (16 * NT));
    auto blocks = [&](int rows) { return (unsigned)a.nimg * tx * (unsigned)((a.H + rows - 1) / rows); };
    auto lds = [&](int rows) { return (size_t)(16 + 2 * (KS / 2)) * (rows + 2 * (KS / 2)) * a.cin * sizeof(uint16_t); };
    auto good = [&](int rows) { return blocks(rows) * ny >= 512 && lds(rows) <= 80 * 1024; };
    if (good(16)) launch_conv_rows<KS, 4, NT>(a, blocks(16), ny, lds(16), s);
    else if (good(8)) launch_conv_rows<KS, 2, NT>(a, blocks(8), ny, lds(8), s);
    else launch_conv_rows<KS, 1, NT>(a, blocks(4), ny, lds(4), s);
}

// cout: 16 or a multiple of 32; 16 NT channels a workgroup
hipError_t conv(const ConvArgs& a, hipStream_t s) {
    if (a.cin % 32 != 0 || a.c1 % 32 != 0 || a.cin > 256 || (a.cout != 16 && a.cout % 32 != 0) || (a.ksize != 1 && a.ksize != 3)) return hipErrorInvalidValue;
    if (a.ksize == 1) {
        if (a.cout == 16) launch_conv<1, 1>(a, s);
        else launch_conv<1, 2>(a, s);
    } else if (a.cout % 64 == 0) {
        launch_conv<3, 4>(a, s);
    } else if (a.cout % 96 == 0) {
        launch_conv<3, 6>(a, s);
    } else if (a.cout % 32 == 0) {
        launch_conv<3, 2>(a, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- weight gradient

// A workgroup takes 32 input x 32 output channels, all taps, and every gridDim.z-th tile of 32 x 16
// pixels: it stages the tile's dz and x (with halo) in LDS, and each of its four waves goes down four
// rows of it. Per staged row of x a wave reads its 32 pixels at the three horizontal taps once and
// multiplies them with the dz of the (up to three) rows that reach it; ds_read_b64_tr_b16 gives a lane
// four pixels of one channel, as the MFMA wants them, from rows of channels. The waves' sums are
// added in LDS and stored in a slice per workgroup; k_wgrad_sum adds the slices in order, so that
// the result does not depend on the order of the workgroups.
//
// What bounds it: staging and LDS. A training step on 8 images of 480 x 272 spends 1.87 ms on its 12
// layers, the sums of the slices among it. One wave per tap that staged both operands transposed,
// two bytes a store, and added 4,096-pixel sums with atomics took 3.61 ms.
constexpr int WG_TW = 32, WG_TH = 16, WG_ROWS = 4;

__device__ __forceinline__ s16x8 tr_read(const uint16_t* p) {  // pixels p, p + 1 .. p + 3 and p + 4 .. p + 7
    typedef short v4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4* lds4;
    const v4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * 32));
    return s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

template <int KS>
__global__ __launch_bounds__(256) void k_wgrad(WgradArgs a, float* slices) {
    constexpr int HALO = KS / 2, TAPS = KS * KS;
    constexpr int XW = WG_TW + 2 * HALO, XH = WG_TH + 2 * HALO;
    constexpr int NX = XW * XH * 32, NZ = WG_TW * WG_TH * 32;
    constexpr int SUMS = TAPS * 4 * 256;  // fp32 sums of one wave
    constexpr int BYTES = (NX + NZ) * 2 > 2 * SUMS * 4 ? (NX + NZ) * 2 : 2 * SUMS * 4;
    __shared__ __attribute__((aligned(16))) unsigned char lds[BYTES];
    uint16_t* sx = (uint16_t*)lds;  // [row][pixel][32]
    uint16_t* sz = sx + NX;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i16 = lane & 15, kg = lane >> 4;
    const int ci0 = blockIdx.x * 32, co0 = blockIdx.y * 32;
    const int tx = (a.W + WG_TW - 1) / WG_TW, ty = (a.H + WG_TH - 1) / WG_TH;
    const int tiles = a.nimg * tx * ty;
    const uint16_t* xp = ci0 < a.c1 ? a.x + ci0 : a.x2 + (ci0 - a.c1);
    const int xs = ci0 < a.c1 ? a.c1 : a.cin - a.c1;
    const int up = ci0 < a.c1 ? a.up : 0;
    f32x4 acc[TAPS][2][2];
#pragma unroll
    for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[t][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the 16 lanes of a group read 4 pixels x 16 channels: lane i16 supplies pixel i16 / 4, channels
    // 4 (i16 % 4) .. + 3 of the group's pixels 8 kg .. 8 kg + 3
    const int tr = (8 * kg + i16 / 4) * 32 + 4 * (i16 % 4);
    for (int tile = blockIdx.z; tile < tiles; tile += gridDim.z) {
        const int img = tile / (tx * ty), rest = tile % (tx * ty);
        const int y0 = rest / tx * WG_TH, x0 = rest % tx * WG_TW;
        if (tile != (int)blockIdx.z) __syncthreads();  // the previous tile is used up
        for (int e = threadIdx.x; e < NX / 8; e += 256) {
            const int p = e >> 2, gy = y0 + p / XW - HALO, gx = x0 + p % XW - HALO;
            s16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
            if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W) v = *(const s16x8*)(xp + source_pixel(img, gy, gx, a.H, a.W, up) * xs + (e & 3) * 8);
            *(s16x8*)&sx[e * 8] = v;
        }
        for (int e = threadIdx.x; e < NZ / 8; e += 256) {
            const int p = e >> 2, gy = y0 + p / WG_TW, gx = x0 + p % WG_TW;
            s16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
            if (gy < a.H && gx < a.W) v = *(const s16x8*)(a.dz + ((size_t)(img * a.H + gy) * a.W + gx) * a.cout + co0 + (e & 3) * 8);
            *(s16x8*)&sz[e * 8] = v;
        }
        __syncthreads();
        s16x8 Z[KS][2];  // dz of the last KS rows
#pragma unroll
        for (int r = 0; r < WG_ROWS + 2 * HALO; ++r) {
            const int row = wave * WG_ROWS + r;  // staged row of x
            if (r < WG_ROWS) {
#pragma unroll
                for (int i = 0; i < 2; ++i) Z[r % KS][i] = tr_read(&sz[row * WG_TW * 32 + tr + i * 16]);
            }
#pragma unroll
            for (int dx = 0; dx < KS; ++dx) {
                s16x8 X[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) X[j] = tr_read(&sx[(row * XW + dx) * 32 + tr + j * 16]);
#pragma unroll
                for (int dy = 0; dy < KS; ++dy) {
                    if (r - dy < 0 || r - dy >= WG_ROWS) continue;  // row r of x is tap dy of the dz row r - dy
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[dy * KS + dx][i][j] = mfma(Z[(r - dy) % KS][i], X[j], acc[dy * KS + dx][i][j]);
                }
            }
        }
    }
    // waves 2 and 3 into 0 and 1, then 1 into 0
    float* part = (float*)lds;
    auto give = [&](int slot) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) *(f32x4*)&part[slot * SUMS + (t * 4 + q) * 256 + lane * 4] = acc[t][q >> 1][q & 1];
    };
    auto take = [&](int slot) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[t][q >> 1][q & 1] += *(const f32x4*)&part[slot * SUMS + (t * 4 + q) * 256 + lane * 4];
    };
    __syncthreads();
    if (wave >= 2) give(wave - 2);
    __syncthreads();
    if (wave < 2) take(wave);
    __syncthreads();
    if (wave == 1) give(0);
    __syncthreads();
    if (wave != 0) return;
    take(0);
    // lane holds output channels 4 kg .. + 3 and input channel i16 of each 16 x 16
    float* o = slices + (size_t)blockIdx.z * a.cout * TAPS * a.cin;
#pragma unroll
    for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    o[((size_t)(co0 + i * 16 + 4 * kg + q) * TAPS + t) * a.cin + ci0 + j * 16 + i16] = acc[t][i][j][q];
}

__global__ __launch_bounds__(256) void k_wgrad_sum(const float* slices, int n, long long count, float* dw) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    float s = 0.f;
#pragma unroll 8
    for (int k = 0; k < n; ++k) s += slices[(size_t)k * count + i];
    dw[i] = s;
}

// Slices: enough workgroups for four per CU, at most one per tile and WG_SLICE_FLOATS floats in all.
int wgrad_slices(const WgradArgs& a) {
    const long long tiles = (long long)a.nimg * ((a.W + WG_TW - 1) / WG_TW) * ((a.H + WG_TH - 1) / WG_TH);
    const long long blocks = (long long)(a.cin / 32) * (a.cout / 32);
    const long long weights = (long long)a.cout * a.ksize * a.ksize * a.cin;
    return (int)std::max<long long>(1, std::min(std::min(tiles, (1024 + blocks - 1) / blocks), WG_SLICE_FLOATS / weights));
}

// cin, c1 and cout: multiples of 32; slices: wgrad_slices(a) x the layer's weights
hipError_t wgrad(const WgradArgs& a, float* slices, hipStream_t s) {
    if (a.cin % 32 || a.c1 % 32 || a.cout % 32 || (a.ksize != 1 && a.ksize != 3)) return hipErrorInvalidValue;
    const int n = wgrad_slices(a);
    const dim3 grid((unsigned)(a.cin / 32), (unsigned)(a.cout / 32), (unsigned)n);
    if (a.ksize == 3) hipLaunchKernelGGL(k_wgrad<3>, grid, dim3(256), 0, s, a, slices);
    else hipLaunchKernelGGL(k_wgrad<1>, grid, dim3(256), 0, s, a, slices);
    const long long count = (long long)a.cout * a.ksize * a.ksize * a.cin;
    hipLaunchKernelGGL(k_wgrad_sum, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, slices, n, count, a.dw);
    return hipGetLastError();
}

// dz = bf16(da * (a > 0)) and db[c] += sum_p dz[p][c]; without `da`, dz is given and only summed. One
// workgroup takes DZ_CHUNK pixels, a thread 8 channels of every (2048 / c)th of them; the workgroup's
// sums are added up in LDS before one atomic per channel. Bound by HBM: 8 bytes a value. As two
// passes, with one value a thread and every thread of the second walking 1,024 pixels two bytes at a
// time, they took 3.36 ms of a training step on 8 images of 480 x 272, now 0.46.
constexpr int DZ_CHUNK = 1024;

template <bool RELU>
__global__ __launch_bounds__(256) void k_dz(const float* da, const uint16_t* a, uint16_t* dz, int c, long long npix, float* db) {
    __shared__ float sum[256 * 8];
    const int groups = c / 8, g = threadIdx.x % groups, pstep = 256 / groups;
    const long long p0 = (long long)blockIdx.x * DZ_CHUNK, p1 = min(npix, p0 + DZ_CHUNK);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if ((int)threadIdx.x < pstep * groups)
        for (long long p = p0 + threadIdx.x / groups; p < p1; p += pstep) {
            const size_t i = (size_t)p * c + g * 8;
            s16x8 z;
            if constexpr (RELU) {
                const s16x8 av = *(const s16x8*)(a + i);
                const f32x4 d0 = *(const f32x4*)(da + i), d1 = *(const f32x4*)(da + i + 4);
#pragma unroll
                for (int j = 0; j < 8; ++j) z[j] = (short)f2bf(bf2f((uint16_t)av[j]) > 0.f ? (j < 4 ? d0[j & 3] : d1[j & 3]) : 0.f);
                *(s16x8*)(dz + i) = z;
            } else {
                z = *(const s16x8*)(dz + i);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += bf2f((uint16_t)z[j]);
        }
#pragma unroll
    for (int j = 0; j < 8; ++j) sum[threadIdx.x * 8 + j] = acc[j];
    __syncthreads();
    for (int ch = threadIdx.x; ch < c; ch += 256) {
        float s = 0.f;
        for (int q = 0; q < pstep; ++q) s += sum[(q * groups + ch / 8) * 8 + (ch & 7)];
        atomicAdd(&db[ch], s);
    }
}

// c: a multiple of 32, at most 2048; da and a null: dz is given
hipError_t dz_grad(const float* da, const uint16_t* a, uint16_t* dz, int c, long long npix, float* db, hipStream_t s) {
    if (c % 32 != 0 || c > 2048 || (da == nullptr) != (a == nullptr)) return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)((npix + DZ_CHUNK - 1) / DZ_CHUNK);
    if (da) hipLaunchKernelGGL(k_dz<true>, dim3(blocks), dim3(256), 0, s, da, a, dz, c, npix, db);
    else hipLaunchKernelGGL(k_dz<false>, dim3(blocks), dim3(256), 0, s, da, a, dz, c, npix, db);
    return hipGetLastError();
}

// ---------------------------------------------------------------- elementwise and resampling

__global__ void k_pool(const uint16_t* x, int xs, int c, int nimg, int H, int W, uint16_t* y, int ys) {
    const int Ho = H / 2, Wo = W / 2;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nimg * Ho * Wo * c;
    if (i >= n) return;
    const int ch = (int)(i % c);
    const long long q = i / c;
    const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho), b = (int)(q / ((long long)Wo * Ho));
    const long long base = ((long long)b * H + 2 * yo) * W + 2 * xo;
    const float v = bf2f(x[base * xs + ch]) + bf2f(x[(base + 1) * xs + ch]) + bf2f(x[(base + W) * xs + ch]) +
                    bf2f(x[(base + W + 1) * xs + ch]);
    y[q * ys + ch] = f2bf(0.25f * v);
}

hipError_t pool(const uint16_t* x, int xs, int c, int nimg, int H, int W, uint16_t* y, int ys, hipStream_t s) {
    const long long n = (long long)nimg * (H / 2) * (W / 2) * c;
    hipLaunchKernelGGL(k_pool, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, xs, c, nimg, H, W, y, ys);
    return hipGetLastError();
}

__global__ void k_pool_grad(const float* dy, int dys, int c, int nimg, int H, int W, float* dx, int dxs) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nimg * H * W * c;
    if (i >= n) return;
    const int ch = (int)(i % c);
    const long long p = i / c;
    const int x = (int)(p % W), y = (int)((p / W) % H), b = (int)(p / ((long long)W * H));
    const int Ho = H / 2, Wo = W / 2;
    const long long q = ((long long)b * Ho + y / 2) * Wo + x / 2;
    dx[p * dxs + ch] += 0.25f * dy[q * dys + ch];
}

hipError_t pool_grad(const float* dy, int dys, int c, int nimg, int H, int W, float* dx, int dxs, hipStream_t s) {
    const long long n = (long long)nimg * H * W * c;
    hipLaunchKernelGGL(k_pool_grad, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, dy, dys, c, nimg, H, W, dx, dxs);
    return hipGetLastError();
}

__global__ void k_upsample_grad(const float* dy, int dys, int yoff, int c, int nimg, int H, int W, float* dx, int dxs) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nimg * H * W * c;
    if (i >= n) return;
    const int ch = (int)(i % c);
    const long long q = i / c;
    const int x = (int)(q % W), y = (int)((q / W) % H), b = (int)(q / ((long long)W * H));
    const int W2 = 2 * W;
    const long long p = ((long long)b * 2 * H + 2 * y) * W2 + 2 * x;
    const float g = dy[p * dys + yoff + ch] + dy[(p + 1) * dys + yoff + ch] + dy[(p + W2) * dys + yoff + ch] +
                    dy[(p + W2 + 1) * dys + yoff + ch];
    dx[q * dxs + ch] += g;
}

hipError_t upsample_grad(const float* dy, int dys, int yoff, int c, int nimg, int H, int W, float* dx, int dxs, hipStream_t s) {
    const long long n = (long long)nimg * H * W * c;
    hipLaunchKernelGGL(k_upsample_grad, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, dy, dys, yoff, c, nimg, H, W, dx, dxs);
    return hipGetLastError();
}

__global__ void k_add_channels(const float* dy, int dys, int off, int c, long long npix, float* dx, int dxs) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= npix * c) return;
    const long long p = i / c;
    const int ch = (int)(i - p * c);
    dx[p * dxs + ch] += dy[p * dys + off + ch];
}

hipError_t add_channels(const float* dy, int dys, int off, int c, long long npix, float* dx, int dxs, hipStream_t s) {
    const long long n = npix * c;
    hipLaunchKernelGGL(k_add_channels, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, dy, dys, off, c, npix, dx, dxs);
    return hipGetLastError();
}

__global__ void k_fill(float* p, float v, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t fill(float* p, float v, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

// A convolution's weights in the order k_conv reads them: for each tap, 32 input channels and 16
// output channels the 64 lanes' 8 values (lane = 16 (ci % 32 / 8) + co % 16).
__device__ __forceinline__ size_t packed(int ci, int t, int co, int cin, int cout) {
    return ((((size_t)t * (cin / 32) + ci / 32) * (cout / 16) + co / 16) * 64 + (ci % 32 / 8) * 16 + co % 16) * 8 + ci % 8;
}

__global__ void k_weights_bf16(const float* w32, int cout, int taps, int cin, uint16_t* w, uint16_t* wt) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)cout * taps * cin;
    if (i >= n) return;
    const int ci = (int)(i % cin);
    const int t = (int)((i / cin) % taps);
    const int co = (int)(i / ((long long)cin * taps));
    const uint16_t b = f2bf(w32[i]);
    w[packed(ci, t, co, cin, cout)] = b;
    // data gradient: the taps flipped, input and output channels exchanged
    wt[packed(co, taps - 1 - t, ci, cout, cin)] = b;
}

hipError_t weights_bf16(const float* w32, int cout, int taps, int cin, uint16_t* w, uint16_t* wt, hipStream_t s) {
    const long long n = (long long)cout * taps * cin;
    hipLaunchKernelGGL(k_weights_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w32, cout, taps, cin, w, wt);
    return hipGetLastError();
}

// ---------------------------------------------------------------- loss

__device__ __forceinline__ float sigm(float x) { return 1.f / (1.f + __expf(-x)); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// The four sums leave a workgroup in one atomic each, from at most LOSS_BLOCKS workgroups: atomics of
// every wave on the same four words took 0.83 ms of a training step on 8 images of 480 x 272
// (0.04 now).
constexpr int LOSS_BLOCKS = 512;

__global__ __launch_bounds__(256) void k_loss(LossArgs a) {
    __shared__ float part[4][4];
    const long long HW = (long long)a.H * a.W;
    const long long P = a.nimg * HW;
    float ld = 0.f, ln = 0.f, lc = 0.f, cnt = 0.f;
    for (long long p = (long long)blockIdx.x * 256 + threadIdx.x; p < P; p += (long long)gridDim.x * 256) {
        float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        const int b = (int)(p / HW);
        const int rem = (int)(p - (long long)b * HW);
        const int y = rem / a.W, x = rem - y * a.W;
        const float* o = a.out + p * 32;
        const float* lb = a.label + p * 4;
        if (y < a.Hv && x < a.Wv && lb[0] > 0.f) {
            const float ia = 1.f / a.range[2 * b + 1], ib = 1.f / a.range[2 * b];
            const float s0 = sigm(o[0]);
            const float id = ia + s0 * (ib - ia);
            const float idt = 1.f / lb[0];
            const float e = id - idt;
            ld += fabsf(e) / (ib - ia);
            g[0] = (e > 0.f ? 1.f : (e < 0.f ? -1.f : 0.f)) * s0 * (1.f - s0);
            const float vx = o[1], vy = o[2], vz = o[3];
            const float nv = sqrtf(vx * vx + vy * vy + vz * vz + 1e-6f);
            const float nx = vx / nv, ny = vy / nv, nz = vz / nv;
            const float dot = nx * lb[1] + ny * lb[2] + nz * lb[3];
            ln += 1.f - dot;
            g[1] = -a.w_normal * (lb[1] - dot * nx) / nv;
            g[2] = -a.w_normal * (lb[2] - dot * ny) / nv;
            g[3] = -a.w_normal * (lb[3] - dot * nz) / nv;
            const float c = sigm(o[4]);
            const float tgt = fabsf(1.f / id - lb[0]) <= a.conf_tol * lb[0] ? 1.f : 0.f;
            lc += -(tgt * __logf(fmaxf(c, 1e-7f)) + (1.f - tgt) * __logf(fmaxf(1.f - c, 1e-7f)));
            g[4] = a.w_conf * (c - tgt);
            cnt += 1.f;
        }
        uint16_t* d = a.dout + p * 32;
#pragma unroll
        for (int k = 0; k < 5; ++k) d[k] = f2bf(g[k]);
    }
    ld = wave_sum(ld);
    ln = wave_sum(ln);
    lc = wave_sum(lc);
    cnt = wave_sum(cnt);
    if ((threadIdx.x & 63) == 0) {
        float* q = part[threadIdx.x >> 6];
        q[0] = ld;
        q[1] = ln;
        q[2] = lc;
        q[3] = cnt;
    }
    __syncthreads();
    if (threadIdx.x < 4) atomicAdd(&a.sums[threadIdx.x], part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x]);
}

hipError_t loss(const LossArgs& a, hipStream_t s) {
    const long long P = (long long)a.nimg * a.H * a.W;
    hipLaunchKernelGGL(k_loss, dim3((unsigned)std::min<long long>((P + 255) / 256, LOSS_BLOCKS)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------- Adam

__global__ void k_adam(float* w, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps, float b1t,
                       float b2t, const float* count) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] / fmaxf(count[0], 1.f);
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / b1t) / (sqrtf(vi / b2t) + eps);
}

hipError_t adam(float* w, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps, float b1t,
                float b2t, const float* count, hipStream_t s) {
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w, g, m, v, n, lr, b1, b2, eps, b1t, b2t, count);
    return hipGetLastError();
}

// ---------------------------------------------------------------- plane-sweep features

// Channels 0..31: mean over the sources of |I_ref - I_src(H_k x)| / 255 for fronto-parallel planes
// at 32 inverse depths evenly spaced (bin centres) between 1/dmax and 1/dmin; 1 where no source
// sees the pixel. Channel 32: I_ref / 255. Channels 33..63 and the padding pixels: 0.
__device__ __forceinline__ float bilin_u8(const uint8_t* g, int w, int h, float u, float v, bool& inside) {
    const float xf = floorf(u), yf = floorf(v);
    const int x0 = (int)xf, y0 = (int)yf;
    inside = u >= 0.f && v >= 0.f && u <= (float)(w - 1) && v <= (float)(h - 1);
    if (!inside) return 0.f;
    const int x1 = min(x0 + 1, w - 1), y1 = min(y0 + 1, h - 1);
    const float ax = u - xf, ay = v - yf;
    const float p00 = g[y0 * w + x0], p10 = g[y0 * w + x1], p01 = g[y1 * w + x0], p11 = g[y1 * w + x1];
    const float top = p00 + ax * (p10 - p00), bot = p01 + ax * (p11 - p01);
    return top + ay * (bot - top);
}

// One thread per pixel; its 64 bf16 channels leave in eight 16-byte stores.
__global__ __launch_bounds__(256) void k_sweep(SweepArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.H * a.W) return;
    const int y = i / a.W, x = i - y * a.W;
    s16x8* f = (s16x8*)(a.feat + (long long)i * 64);
    const bool in = x < a.rw && y < a.rh;
    const float ir = in ? (float)a.ref[y * a.rw + x] : 0.f;
    const float rx = (x - a.rk[2]) / a.rk[0], ry = (y - a.rk[3]) / a.rk[1];
    const float ia = 1.f / a.dmax, ib = 1.f / a.dmin;
    for (int k0 = 0; k0 < 32; k0 += 8) {
        s16x8 o = {0, 0, 0, 0, 0, 0, 0, 0};
        if (in) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int k = k0 + q;
                const float d = 1.f / (ia + (k + 0.5f) / 32.f * (ib - ia));
                const float X = rx * d, Y = ry * d, Z = d;
                float cost = 0.f;
                int n = 0;
                for (int s = 0; s < a.nsrc; ++s) {
                    const float* R = a.r[s];
                    const float xs = R[0] * X + R[1] * Y + R[2] * Z + a.t[s][0];
                    const float ys = R[3] * X + R[4] * Y + R[5] * Z + a.t[s][1];
                    const float zs = R[6] * X + R[7] * Y + R[8] * Z + a.t[s][2];
                    if (!(zs > 1e-6f)) continue;
                    const float u = a.sk[s][0] * xs / zs + a.sk[s][2], v = a.sk[s][1] * ys / zs + a.sk[s][3];
                    bool inside;
                    const float is = bilin_u8(a.src[s], a.sw[s], a.sh[s], u, v, inside);
                    if (!inside) continue;
                    cost += fabsf(ir - is);
                    n++;
                }
                o[q] = (short)f2bf(n > 0 ? cost / (255.f * n) : 1.f);
            }
        }
        f[k0 / 8] = o;
    }
    f[4] = s16x8{in ? (short)f2bf(ir / 255.f) : (short)0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 5; q < 8; ++q) f[q] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
}

hipError_t sweep(const SweepArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_sweep, dim3((unsigned)((a.H * a.W + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------- network output -> predictions
//
// Bound by the transfer to the host. With the predictions formed on the host from the padded 128-byte
// head output of each pixel, features and prediction of 6 images of 480 x 272 took 13.9 to 32.8 ms, by
// process (a host vector of 100 MB a call); formed here, 40 bytes a pixel cross at most, and both take
// 2.7 to 3.7 ms together (the convolutions' share of the gain is 0.9).

__global__ __launch_bounds__(256) void k_predict(PredictArgs a) {
    const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
    if (p >= a.npix) return;
    const float4 q = *(const float4*)(a.out + p * 32);
    const float q4 = a.out[p * 32 + 4];
    const int b = (int)(p / a.per);
    const float ia = 1.f / a.range[2 * b + 1], ib = 1.f / a.range[2 * b];
    if (a.depth) a.depth[p] = 1.f / (ia + 1.f / (1.f + expf(-q.x)) * (ib - ia));
    if (a.normal) {
        const float nv = sqrtf(q.y * q.y + q.z * q.z + q.w * q.w + 1e-6f);
        a.normal[3 * p] = q.y / nv;
        a.normal[3 * p + 1] = q.z / nv;
        a.normal[3 * p + 2] = q.w / nv;
    }
    if (a.conf) a.conf[p] = 1.f / (1.f + expf(-q4));
    if (a.head) {
        float* h = a.head + 5 * p;
        h[0] = q.x;
        h[1] = q.y;
        h[2] = q.z;
        h[3] = q.w;
        h[4] = q4;
    }
}

hipError_t predict(const PredictArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_predict, dim3((unsigned)((a.npix + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------- network output -> PatchStereo planes

__global__ void k_init_planes(InitPlanesArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.w * a.h) return;
    const int y = i / a.w, x = i - y * a.w;
    // the full-resolution pixel centre in quarter-resolution pixels (two halvings of the pyramid,
    // c <- (c + 0.5) / 2 - 0.5)
    const float u = (x + 0.5f) * 0.25f - 0.5f, v = (y + 0.5f) * 0.25f - 0.5f;
    const float uc = fminf(fmaxf(u, 0.f), (float)(a.qw - 1)), vc = fminf(fmaxf(v, 0.f), (float)(a.qh - 1));
    const int x0 = (int)floorf(uc), y0 = (int)floorf(vc);
    const int x1 = min(x0 + 1, a.qw - 1), y1 = min(y0 + 1, a.qh - 1);
    const float ax = uc - x0, ay = vc - y0;
    const float ia = 1.f / a.dmax, ib = 1.f / a.dmin;
    auto inv = [&](int qx, int qy) { return ia + sigm(a.out[((long long)qy * a.W + qx) * 32]) * (ib - ia); };
    const float top = inv(x0, y0) + ax * (inv(x1, y0) - inv(x0, y0));
    const float bot = inv(x0, y1) + ax * (inv(x1, y1) - inv(x0, y1));
    const float id = top + ay * (bot - top);
    const int qx = min(max((int)roundf(uc), 0), a.qw - 1), qy = min(max((int)roundf(vc), 0), a.qh - 1);
    const float* o = a.out + ((long long)qy * a.W + qx) * 32;
    float4 pl = make_float4(0.f, 0.f, 0.f, 0.f);
    if (sigm(o[4]) >= a.conf_min) {
        const float nv = sqrtf(o[1] * o[1] + o[2] * o[2] + o[3] * o[3] + 1e-6f);
        float nx = o[1] / nv, ny = o[2] / nv, nz = o[3] / nv;
        const float rx = (x - a.k[2]) / a.k[0], ry = (y - a.k[3]) / a.k[1];
        if (nx * rx + ny * ry + nz > 0.f) {
            nx = -nx;
            ny = -ny;
            nz = -nz;
        }
        pl = make_float4(nx, ny, nz, 1.f / id);
    }
    a.plane[i] = pl;
}

hipError_t init_planes(const InitPlanesArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_init_planes, dim3((unsigned)((a.w * a.h + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace nn
}  // namespace c3d
