// pm_device.hpp — device-side data layout and arithmetic of the gfx950 PatchStereo kernels.
//
// Layout in HBM (one session):
//   gray   all view-level images, u8 row-major, no padding (reference patch loads)
//   quad   per view-level, a (w+3) x (h+3) table: entry (x0, y0) for x0 in [-2, w], y0 in [-2, h] holds
//          the bilinear 2x2 neighbourhood p(x0,y0), p(x0+1,y0), p(x0,y0+1), p(x0+1,y0+1) with 0 outside
//          the image, so that one load gives all four texels of a source sample and clamping the
//          integer sample position into the table reproduces "0 outside" exactly
//          (patchmatch.cu:169-192 software bilinear). Two forms of the table, one per namespace of
//          window kernels (pm_windows.hip is compiled for each): 4-byte entries of the four bytes, and
//          8-byte entries of the row starts and row differences as half floats (exact), which save
//          the four instructions that form them; which one a launch takes is run_quad8's rule.
//   plane  float4 (nx, ny, nz, d) per pixel, row-major per view, views of a batch back to back
//          (ViewState packed as in patchmatch.rs:327-348); cost f32, best view u8, count u8 alike.
//
// Arithmetic: every operation is written out (explicit fmaf where an FMA is intended; the library
// is compiled with -ffp-contract=off) in the order the CPU oracle uses, with IEEE division and
// square root, the polynomial exp / sin-cos below and a seeded reciprocal for the per-sample
// projective divide, so that the device and the CPU oracle agree bit for bit.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#ifndef C3D_QUAD_BYTES
#define C3D_QUAD_BYTES 4
#endif

namespace c3d {

constexpr int MAXSRC = 32;
constexpr int MAX_WR = 20;  // largest window radius (patchmatch.rs:292-294)
constexpr float INF_ERR = 1e30f;

struct LevelDesc {
    int w, h;
    int qpitch;      // quad row pitch (w + 3)
    int pad0;
    long long qoff;  // index of quad entry (0, 0) (the 2-texel border precedes it)
    long long goff;  // byte offset of the u8 image
    float fx, fy, cx, cy;
    float ifx, ify;   // 1 / fx, 1 / fy
    int plain, pad1;  // k lies where a pixel's (u - c) / f may go through div_exact
};

struct PairRec {
    int src;
    float r[9], t[3], c[3];
};

struct LevelPair {
    float A[9];
    float b[3];
};

struct ViewDesc {
    unsigned long long key;
    float dmin, dmax;
    int nsrc, pad0;
};

struct BatchItem {
    long long off;  // first pixel of this view in the batch state buffers
    int view, w, h;
    int low_off;    // upsampling: first pixel of the low-resolution input in the prior buffer
};

struct KParams {
    unsigned long long seed;
    const uint8_t* gray;
    const void* quad;  // entries of 4 or 8 bytes: the table of the launched kernels' namespace
    const LevelDesc* lv;
    const PairRec* pairs;
    const LevelPair* lpairs;
    const ViewDesc* views;
    const BatchItem* batch;
    const float* snap;
    const long long* snap_off;
    float4* plane;
    float* cost;
    uint8_t* bview;
    uint8_t* count;
    const float4* prior;
    int nitems, nlevels, level, geometric;
    int run_id, t, color, random_init;
    int topk, n1, n2, use_prior;
    float tau_good, tau_bad, inv2beta2, prev_w;
    float inv2s, inv2c255, vmin255, weak_var255;
    float cos_tri_min, inv2inc, lambda, gmax;
    float eps, phi, up_inv2s, up_inv2c;
    float cos_filter_tri, q_min, ncc_norm, inv2ncc;
    float filter_gmax;
    // first flattened tile of each batch item for the launch's tile shape, tile_pre[nitems] = all
    // tiles (null: locate_tile searches the items linearly)
    const int* tile_pre;
    int wv_stride;  // LDS floats per source in the per-thread view-weight table
    int ntiles;     // total workgroups of the launch
    int max_nsrc;   // largest source count of the batch (sizes the LDS view-weight table)
    int wr;         // window radius (read by the kernels compiled for any radius)
};

// ---------------------------------------------------------------- work distribution

// Workgroups are dealt round-robin to the 8 XCDs (each with its own L2). Runs of XCD_RUN
// consecutive logical tiles go to one XCD, so that neighbouring tiles share their source footprints
// in that L2, and the runs are dealt to the XCDs in turn, so that every XCD gets its share of the
// costly and of the cheap parts of each view. (One contiguous eighth of the tiles per XCD left
// XCDs idle while the one with the costliest eighth finished: 1.7 of 2 wave slots per SIMD were
// taken on average.) In the half step a run is a square of 8 x 8 blocks (HALF_BAND), 128 x 64 pixels,
// with one-row workgroups; with 2 and 4 rows a run's 64 workgroups are 8 blocks high and 16 and 32 wide.
// The kernels of 64 x 4 and 128 x 4 pixel tiles (evaluation, read-out, upsampling, median) take runs of
// 64 tiles row by row; runs were compared on the half step only.
// Each round of 8 runs starts at another XCD, scattered by a multiplicative hash: without it a width
// of a whole or half number of rounds gives each XCD the same columns of every view. Measured against
// runs of 16 tiles of one row: half step of 9 views of 1920 x 1080 with 6 sources 17.91 -> 17.72 ms; 2
// such views from a random start, 3 iterations 31.1 -> 30.15 ms; 9 views of up to 1283 x 717,
// geometric, 24.5 -> 24.05 ms; 12 views of 960 x 540 over 3 scales 218.6 -> 217.0 ms (234 ms without
// the scattering). Runs of 32 tiles, 4 x 8 or 8 x 4, gained less (17.92 and 17.86 ms; 30.9 and 31.2 ms).
// Windows whose weights are formed again wait less for L2 and more for the last XCD: they keep runs of
// 16 of one row (3 views of 641 x 479, window (5, 1): 12.25 against 12.6 ms).
// The tiles after the last whole round keep their order.
constexpr int XCD_RUN = 64;
constexpr int XCD_RUN_ROW = 16;
constexpr int HALF_BAND = 8;
template <int RUN = XCD_RUN>
__device__ __forceinline__ int xcd_tile(int bid, int n) {
    const int nx = 8;
    if (bid >= n - n % (nx * RUN)) return bid;
    const int k = bid / nx, round = k / RUN;
    const int x = (bid + (int)((uint32_t)round * 0x9E3779B1u >> 29)) % nx;
    return (round * nx + x) * RUN + k % RUN;
}

// Tile tl of an item of tx x ty tiles: row by row, or (band > 1) column by column in bands of that many
// rows.
__device__ __forceinline__ void tile_origin(int tl, int tx, int ty, int tw, int th, int band, int& x0, int& y0) {
    const int b = tl / (band * tx), r = tl - b * band * tx, rows = min(band, ty - b * band);
    x0 = r / rows * tw;
    y0 = (b * band + r % rows) * th;
}

// Finds the batch item of flattened tile `t` for tiles of tw x th pixels; returns the item and
// the tile's pixel origin, or false when t is past the last item.
__device__ __forceinline__ bool locate_tile(const KParams& P, int t, int tw, int th, BatchItem& it, int& x0, int& y0,
                                            int band = 1, int* item = nullptr) {
    for (int i = 0; i < P.nitems; ++i) {
        BatchItem b = P.batch[i];
        int tx = (b.w + tw - 1) / tw, ty = (b.h + th - 1) / th;
        int n = tx * ty;
        if (t < n) {
            it = b;
            if (item) *item = i;
            tile_origin(t, tx, ty, tw, th, band, x0, y0);
            return true;
        }
        t -= n;
    }
    return false;
}

// locate_tile through the launch's tile offsets (P.tile_pre, built for the same tw x th): a binary
// search over the items instead of a linear one. The last item whose first tile is at or before t
// holds it (items without tiles share their successor's offset and are passed over).
__device__ __forceinline__ bool locate_tile_pre(const KParams& P, int t, int tw, int th, BatchItem& it, int& x0, int& y0, int band) {
    const int* pre = P.tile_pre;
    if (t >= pre[P.nitems]) return false;
    int lo = 0, hi = P.nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    it = P.batch[lo];
    const int tl = t - pre[lo];
    const int tx = (it.w + tw - 1) / tw;
    tile_origin(tl, tx, (it.h + th - 1) / th, tw, th, band, x0, y0);
    return true;
}

// The tile's item and pixel origin through P.tile_pre when the launch provides it (built for the
// same tw x th), else by the linear search.
__device__ __forceinline__ bool find_tile(const KParams& P, int t, int tw, int th, BatchItem& it, int& x0, int& y0, int band = 1) {
    return P.tile_pre ? locate_tile_pre(P, t, tw, th, it, x0, y0, band) : locate_tile(P, t, tw, th, it, x0, y0, band);
}

// ---------------------------------------------------------------- tile shapes

// Waves per half-step workgroup ("rows": one row of blocks each): a compile-time variant (1, 2 or
// 4), picked per session by the tile autotuner (c3d_pm_autotune). One is the default: a wave's slot
// on its SIMD is refilled as soon as that wave ends, where a 4-wave workgroup holds its slots (and
// its LDS) until its slowest wave is done, and the waves' work differs through the data-dependent
// early exits. On the other hand 4-wave workgroups take less LDS a wave (the margins of the staged
// pixels are shared; a one-wave workgroup holds 12,096 bytes and 256 a source). Jobs from random
// planes are often faster with them, which is what the tuner is for.
constexpr int HALF_SPAN = 128;   // pixel span of one row of 64 active pixels (k_eval of one colour)
// A wave of the half step takes a block of half_bw x half_bh pixels, half of them active: 16 x 8, or
// 8 x 8, 8 x 4 and 8 x 2 with two, four and eight lanes per pixel. What
// a wave costs is what its costliest lane costs, window by window, and pixels of a compact block
// agree better on it (which sources see them, when a candidate is given up) than 64 pixels along
// 128 of one row: 3.4 % fewer VALU instructions for the same pixels. The block's samples also share
// more source lines (a third of the L1 misses of the row), a ragged width wastes less, and the
// staged tile is 2.9 instead of 6.1 KB. 9 views of 1920 x 1080 with 6 sources: half step
// 23.5 -> 22.2 ms; 2 such views, 3 iterations from a random start: 35.3 -> 31.9 ms; one of
// 160 x 96: 0.69 -> 0.61 ms.
__host__ __device__ constexpr int half_bw(int tpp) { return tpp == 1 ? 16 : 8; }
__host__ __device__ constexpr int half_bh(int tpp) { return tpp <= 2 ? 8 : 16 / tpp; }

// Active pixel p of a wave's block as (column of active pixels, row): four neighbouring lanes take a
// 2 x 2 group, so that lanes next to each other sample next to each other in the source, whichever
// way it is turned against the reference.
template <int TPP>
__device__ __forceinline__ void block_pixel(int p, int& col, int& row) {
    col = (p & 1) | ((p >> 1) & 2);
    row = (p >> 1) & 1;
    if (TPP == 1) {
        col |= (p >> 2) & 4;
        row |= ((p >> 2) & 2) | ((p >> 3) & 4);
    } else {
        row |= (p >> 2) & 6;
    }
}

// Pitch of the staged reference rows: the block with its margins, rounded up to 8 modulo 16, with
// which the 64 lanes of a block read 64 different LDS banks.
__host__ __device__ constexpr int half_pitch(int tpp, int wr) { return ((half_bw(tpp) + 2 * wr + 7) / 16) * 16 + 8; }
constexpr int PIX_TW = 64;       // eval/filter tiles: 64 x 4 pixels
constexpr int PIX_TH = 4;

// ---------------------------------------------------------------- random numbers (kernel.rs:248-259)

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float rnd(unsigned long long& s) {
    s += 0x9e3779b97f4a7c15ULL;
    unsigned long long z = mix64(s);
    return ((float)(z >> 40) + 1.0f) * (1.0f / 16777216.0f);
}
__device__ __forceinline__ unsigned long long rng_state(unsigned long long seed, unsigned long long key, int level, int run,
                                                        int t, int half, unsigned long long pixel) {
    unsigned long long tag = ((unsigned long long)level << 48) ^ ((unsigned long long)run << 32) ^
                             ((unsigned long long)t << 16) ^ (unsigned long long)half;
    return mix64(seed ^ mix64(key ^ mix64(tag)) ^ pixel);
}

// ---------------------------------------------------------------- elementary functions

// exp: Cody-Waite reduction, degree-7 Taylor polynomial, scale by 2^n; 0 below -86, +inf above
// 88, NaN kept. Branch-free: the polynomial runs on the argument clamped to [-86, 88] and the
// special values are selected afterwards (same results as testing first).
__device__ __forceinline__ float c3d_expf(float x) {
    const float xc = fminf(fmaxf(x, -86.0f), 88.0f);
    float n = rintf(xc * 1.44269504088896341f);
    float r = fmaf(-n, 0.693145751953125f, xc);
    r = fmaf(-n, 1.42860677e-06f, r);
    float p = 1.98412698e-04f;
    p = fmaf(p, r, 1.38888889e-03f);
    p = fmaf(p, r, 8.33333333e-03f);
    p = fmaf(p, r, 4.16666667e-02f);
    p = fmaf(p, r, 1.66666667e-01f);
    p = fmaf(p, r, 0.5f);
    p = fmaf(p, r, 1.0f);
    p = fmaf(p, r, 1.0f);
    int ni = (int)n;
    float e = p * __int_as_float((ni + 127) << 23);
    e = x > -86.0f ? e : 0.0f;
    e = x > 88.0f ? __builtin_inff() : e;
    return x != x ? x : e;
}

// c3d_expf(-t) for t >= 0 (or NaN) in 15 instead of 25 operations: no upper bound to keep, the lower one
// by the last select alone, and the power of two applied by exponent (p 2^n is normal, so exact).
__device__ __forceinline__ float expf_down(float t) {
    const float n = rintf(-t * 1.44269504088896341f);
    float r = fmaf(-n, 0.693145751953125f, -t);
    r = fmaf(-n, 1.42860677e-06f, r);
    float p = 1.98412698e-04f;
    p = fmaf(p, r, 1.38888889e-03f);
    p = fmaf(p, r, 8.33333333e-03f);
    p = fmaf(p, r, 4.16666667e-02f);
    p = fmaf(p, r, 1.66666667e-01f);
    p = fmaf(p, r, 0.5f);
    p = fmaf(p, r, 1.0f);
    p = fmaf(p, r, 1.0f);
    return t >= 86.0f ? 0.0f : __builtin_amdgcn_ldexpf(p, (int)n);
}

// sin and cos: quadrant reduction, Taylor polynomials on |r| <= pi/4.
__device__ __forceinline__ void c3d_sincosf(float x, float& so, float& co) {
    float k = rintf(x * 0.636619772367581343f);
    float r = fmaf(-k, 1.57079625129699707f, x);
    r = fmaf(-k, 7.54978941586159635e-08f, r);
    r = fmaf(-k, 5.39030252995776476e-15f, r);
    float r2 = r * r;
    float ps = 2.75573192e-06f;
    ps = fmaf(r2, ps, -1.98412698e-04f);
    ps = fmaf(r2, ps, 8.33333333e-03f);
    ps = fmaf(r2, ps, -1.66666667e-01f);
    float s = fmaf(r * r2, ps, r);
    float pc = -2.75573192e-07f;
    pc = fmaf(r2, pc, 2.48015873e-05f);
    pc = fmaf(r2, pc, -1.38888889e-03f);
    pc = fmaf(r2, pc, 4.16666667e-02f);
    pc = fmaf(r2, pc, -0.5f);
    float c = fmaf(r2, pc, 1.0f);
    int q = ((int)k) & 3;
    if (q == 0) { so = s; co = c; }
    else if (q == 1) { so = c; co = -s; }
    else if (q == 2) { so = -s; co = -c; }
    else { so = -c; co = s; }
}

// Reciprocal of the projective divide of one source sample: bit-pattern seed (relative error
// below 2^-4.3), one third-order step r(1 + e + e^2) and one Newton step r(1 + e), e = 1 - z r,
// leaving 2^-25.8 before the last rounding: within 1 ulp of 1/z for positive normal z (0.78 ulp
// at most over a binade), reproducible on any IEEE machine, 6 full-rate VALU operations. The
// hardware estimate v_rcp_f32 plus one Newton step would be the correctly rounded quotient, but
// v_rcp_f32 issues at a quarter of the rate and measured slower (26.65 against 27.21 ms per half
// step on 7 x 1920x1080 with 6 sources).
__device__ __forceinline__ float rcp_seed(float z) { return __uint_as_float(0x7EF311C3u - __float_as_uint(z)); }
__device__ __forceinline__ float rcp_sample(float z) {
    float r = rcp_seed(z);
    float e = fmaf(-z, r, 1.0f);
    r = fmaf(r, fmaf(e, e, e), r);
    e = fmaf(-z, r, 1.0f);
    r = fmaf(r, e, r);
    return r;
}

// Correctly rounded 1/x, a/b and square root from the hardware estimates and FMA residuals (Newton's
// step, and Markstein's: q + (a - b q) y rounds to a/b when y is the rounded 1/b and q within an ulp),
// the same bits as IEEE division and sqrtf in 3, 3 and 5 instructions; the compiler's sequences,
// which also serve the ends of the exponent range, take 10, 10 and 13. inv_exact and sqrt_exact equal
// the IEEE results on every mantissa of one and of two binades (measured on the device). For
// arguments and results between 2^-100 and 2^100 (and a = 0); callers keep IEEE division for the rest.
// An infinite numerator or quotient gives NaN, not infinity.
__device__ __forceinline__ float inv_exact(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}
__device__ __forceinline__ float div_exact(float a, float b, float inv_b) {
    const float q = a * inv_b;
    return fmaf(fmaf(-b, q, a), inv_b, q);
}
__device__ __forceinline__ float sqrt_exact(float x) {
    const float r = __builtin_amdgcn_rsqf(x);
    const float s = x * r;
    return fmaf(fmaf(-s, s, x), 0.5f * r, s);
}
constexpr float EXACT_LO = 0x1p-100f, EXACT_HI = 0x1p100f;

// ---------------------------------------------------------------- vectors

struct f3 {
    float x, y, z;
};
__device__ __forceinline__ f3 mk3(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ float dot3(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross3(f3 a, f3 b) {
    return mk3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ f3 nrm3(f3 a) {
    float d = dot3(a, a);
    float l = 1.0f / sqrtf(d > 1e-30f ? d : 1e-30f);
    return mk3(a.x * l, a.y * l, a.z * l);
}
__device__ __forceinline__ f3 xyz(float4 h) { return mk3(h.x, h.y, h.z); }
__device__ __forceinline__ float4 mk4(f3 n, float d) { return make_float4(n.x, n.y, n.z, d); }

// patchmatch.cu:386
__device__ __forceinline__ f3 pixel_ray(const LevelDesc& R, int x, int y) {
    return mk3(((float)x - R.cx) / R.fx, ((float)y - R.cy) / R.fy, 1.0f);
}

// ---------------------------------------------------------------- reference window

template <int WR, int WSTEP>
struct Win {
    static constexpr int WN = (2 * WR) / WSTEP + 1;
    static constexpr int WN2 = WN * WN;
    static constexpr int LAST = -WR + (WN - 1) * WSTEP;  // last sample offset
    static constexpr bool HELD = WN2 <= 49;              // registers hold the weights
};

// Weighted statistics of the reference patch (patchmatch.cu:199-223): bilateral weights w_k in
// registers, weighted mean and two-pass variance in gray levels. The window values I_k themselves
// are re-read from the reference accessor (LDS) where the covariance needs them.
template <int WR, int WSTEP>
struct RefWin {
    float ic, mu, W, iW, var;
    float w[Win<WR, WSTEP>::HELD ? Win<WR, WSTEP>::WN2 : 1];
};

// Reference image accessors: 0 outside the image.
struct RefGlobal {
    const uint8_t* p;
    int w, h;
    __device__ __forceinline__ float at(int x, int y) const {
        if (x < 0 || y < 0 || x >= w || y >= h) return 0.0f;
        return (float)p[(size_t)y * w + x];
    }
};

template <int TW>
struct RefTile {
    const float* s;
    int x0, y0;
    __device__ __forceinline__ float at(int x, int y) const { return s[(y - y0) * TW + (x - x0)]; }
};

__device__ __forceinline__ float bilateral_weight(const KParams& P, float ic, float v, int dx, int dy) {
    float d = ic - v;
    float sp = (float)(dx * dx + dy * dy) * P.inv2s;
    return expf_down(fmaf(d * d, P.inv2c255, sp));
}

// ref_stats where the weights are not held: formed again where they are used, row by row, the same values.
template <int WR, int WSTEP, class REF>
__device__ __forceinline__ void ref_stats_rows(const KParams& P, const REF& ref, int x, int y, RefWin<WR, WSTEP>& rw) {
    constexpr int WN = Win<WR, WSTEP>::WN;
    rw.ic = ref.at(x, y);
    float W = 0.0f, S = 0.0f;
#pragma unroll 1
    for (int a = 0; a < WN; ++a) {
        const int dy = -WR + a * WSTEP;
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int dx = -WR + b * WSTEP;
            const float v = ref.at(x + dx, y + dy), w = bilateral_weight(P, rw.ic, v, dx, dy);
            W += w;
            S = fmaf(w, v, S);
        }
    }
    const float mu = S / W;
    float V = 0.0f;
#pragma unroll 1
    for (int a = 0; a < WN; ++a) {
        const int dy = -WR + a * WSTEP;
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int dx = -WR + b * WSTEP;
            const float v = ref.at(x + dx, y + dy), dk = v - mu;
            V = fmaf(bilateral_weight(P, rw.ic, v, dx, dy) * dk, dk, V);
        }
    }
    rw.mu = mu;
    rw.W = W;
    rw.iW = 1.0f / W;
    rw.var = V / W;
}

template <int WR, int WSTEP, class REF>
__device__ __forceinline__ void ref_stats(const KParams& P, const REF& ref, int x, int y, RefWin<WR, WSTEP>& rw) {
    constexpr int WN = Win<WR, WSTEP>::WN;
    if constexpr (!Win<WR, WSTEP>::HELD) {
        ref_stats_rows<WR, WSTEP>(P, ref, x, y, rw);
        return;
    }
    rw.ic = ref.at(x, y);
    float W = 0.0f, S = 0.0f;
#pragma unroll
    for (int a = 0; a < WN; ++a) {
        const int dy = -WR + a * WSTEP;
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int dx = -WR + b * WSTEP;
            const int k = a * WN + b;
            float v = ref.at(x + dx, y + dy);
            float d = rw.ic - v;
            float sp = (float)(dx * dx + dy * dy) * P.inv2s;
            float w = expf_down(fmaf(d * d, P.inv2c255, sp));
            rw.w[k] = w;
            W += w;
            S = fmaf(w, v, S);
        }
    }
    float mu = S / W;
    float V = 0.0f;
#pragma unroll
    for (int a = 0; a < WN; ++a) {
        const int dy = -WR + a * WSTEP;
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int dx = -WR + b * WSTEP;
            const int k = a * WN + b;
            float dk = ref.at(x + dx, y + dy) - mu;
            float wd = rw.w[k] * dk;
            V = fmaf(wd, dk, V);
        }
    }
    rw.mu = mu;
    rw.W = W;
    rw.iW = 1.0f / W;
    rw.var = V / W;
}

// ---------------------------------------------------------------- homography and cost

// Plane-induced homography (patchmatch.cu:225-242) translated to the pixel: H maps the window offset
// (dx, dy, 1) of pixel (x, y), H = (A + b n^T K^-1 / delta) T(x, y). Its third column is
// A (x, y, 1)^T + b / d exactly (n^T K^-1 (x, y, 1)^T / delta = 1 / d), free of the cancellation of
// the untranslated form for strongly slanted planes.
__device__ __forceinline__ bool homography(const LevelDesc& R, const LevelPair& L, float ifx, float ify, float x, float y, float d,
                                           f3 n, float* H) {
    f3 ray = mk3((x - R.cx) * ifx, (y - R.cy) * ify, 1.0f);
    float delta = d * dot3(n, ray);
    if (!(delta < -1e-12f)) return false;
    float id, invd;
    if (fmaxf(-delta, fabsf(d)) < EXACT_HI && fabsf(d) > EXACT_LO) {
        id = inv_exact(delta);
        invd = inv_exact(d);
    } else {
        id = 1.0f / delta;
        invd = 1.0f / d;
    }
    float u0 = n.x * ifx, u1 = n.y * ify;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        float br = L.b[r] * id;
        H[r * 3 + 0] = L.A[r * 3 + 0] + br * u0;
        H[r * 3 + 1] = L.A[r * 3 + 1] + br * u1;
        H[r * 3 + 2] = fmaf(L.A[r * 3 + 0], x, fmaf(L.A[r * 3 + 1], y, L.A[r * 3 + 2])) + L.b[r] * invd;
    }
    return true;
}

// Bilinear interpolation of one quad entry at the fractions (ax, ay): top = p00 + ax (p10 - p00),
// bot = p01 + ax (p11 - p01), top + ay (bot - top), each an FP32 FMA. The two row starts and the two
// row differences are packed half floats (integers of magnitude below 2^11, exact), and each row is
// one mixed FMA on them: the same value as the FP32 formula. From a 4-byte entry p00 | p10 << 8 |
// p01 << 16 | p11 << 24 they take a byte permute each that sets the exponent byte 0x64 above each
// texel, which reads 1024 + p exactly, and a packed subtraction each; an 8-byte entry holds them.
// Everything from here on is compiled once per entry size, and so has a namespace per entry size.
#if C3D_QUAD_BYTES == 8
inline namespace entry8 {
#else
inline namespace entry4 {
#endif
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t quad_entry4(uint32_t p00, uint32_t p10, uint32_t p01, uint32_t p11) {
    return p00 | (p10 << 8) | (p01 << 16) | (p11 << 24);
}
__device__ __forceinline__ uint2 quad_entry8(uint32_t p00, uint32_t p10, uint32_t p01, uint32_t p11) {
    const half2_t p = {(_Float16)(int)p00, (_Float16)(int)p01};
    const half2_t d = {(_Float16)((int)p10 - (int)p00), (_Float16)((int)p11 - (int)p01)};
    return make_uint2(__builtin_bit_cast(uint32_t, p), __builtin_bit_cast(uint32_t, d));
}
#if C3D_QUAD_BYTES == 8
typedef uint2 QuadEntry;
__device__ __forceinline__ void quad_rows(QuadEntry q, half2_t& p, half2_t& d) {
    p = __builtin_bit_cast(half2_t, q.x);
    d = __builtin_bit_cast(half2_t, q.y);
}
#else
typedef uint32_t QuadEntry;
__device__ __forceinline__ void quad_rows(QuadEntry q, half2_t& p, half2_t& d) {
    const half2_t l = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, q, 0x04020400u));  // (1024 + p00, 1024 + p01)
    const half2_t h = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, q, 0x04030401u));  // (1024 + p10, 1024 + p11)
    d = h - l;
    p = l - (half2_t){(_Float16)1024.0f, (_Float16)1024.0f};
}
#endif
__device__ __forceinline__ float quad_lerp(QuadEntry q, float ax, float ay) {
    half2_t p, d;
    quad_rows(q, p, d);
    const float top = fmaf(ax, (float)d.x, (float)p.x);
    const float bot = fmaf(ax, (float)d.y, (float)p.y);
    return fmaf(ay, bot - top, top);
}

// The quad table of a source as the samples use it: `base` is the table's first entry (x0, y0) =
// (-2, -2); the byte offset of an entry, QB ((y0 + 2) qpitch + (x0 + 2)), is formed exactly in FP32
// (multiples of QB below 2^24 QB) from the clamped floor of the sample position, and the load uses
// the uniform base plus a 32-bit offset.
constexpr float QB = (float)sizeof(QuadEntry);
struct QuadTable {
    const QuadEntry* base;
    float pitch, off, w, h;
};
__device__ __forceinline__ QuadTable quad_table(const KParams& P, const LevelDesc& S) {
    const float pitch = QB * (float)S.qpitch;
    return QuadTable{(const QuadEntry*)P.quad + (S.qoff - 2LL * S.qpitch - 2), pitch, 2.0f * pitch + 2.0f * QB, (float)S.w, (float)S.h};
}
__device__ __forceinline__ QuadEntry quad_load(const QuadTable& t, float xc, float yc) {
    return *(const QuadEntry*)((const char*)t.base + (uint32_t)fmaf(yc, t.pitch, fmaf(xc, QB, t.off)));
}
// one source sample in gray levels: the entry and the fractions
__device__ __forceinline__ QuadEntry quad_fetch(const QuadTable& t, float u, float v, float& ax, float& ay) {
    const float xf = floorf(u), yf = floorf(v);
    ax = u - xf;
    ay = v - yf;
    return quad_load(t, __builtin_amdgcn_fmed3f(xf, -2.0f, t.w), __builtin_amdgcn_fmed3f(yf, -2.0f, t.h));
}
__device__ __forceinline__ float quad_sample(const QuadTable& t, float u, float v) {
    float ax, ay;
    const QuadEntry q = quad_fetch(t, u, v, ax, ay);
    return quad_lerp(q, ax, ay);
}

// Gathers kept in flight by the window loop: this default serves the cost-probe kernel; the
// evaluation and read-out keep five (three waves per SIMD) and the half step picks its own per
// build. Measured on 7 x 1920x1080, 6 sources, with 4-row half-step workgroups: 4 -> 502.8 ms,
// 6 -> 500.8 ms, 8 -> 500.8 ms per job (photometric half steps 2.9 ms faster, geometric ones
// 2.8 ms slower), 12 spills; the compiler's own batches of eight gathers drained to zero before
// the next batch gave 512.9 ms.
constexpr int WINDOW_PIPE = 8;

// Window sums of one hypothesis x source (H translated to the pixel). A sample whose projective
// depth z is not above 1e-8 contributes the value 0 (patchmatch.cu:271-276). CHECK = false when all
// four window corners have z > 1e-8: z is monotone in each offset (every step is a correctly
// rounded affine operation), so then every sample does. With CHECK the sample is computed anyway
// (any position is clamped into the quad table) and replaced by a select.
// AHEAD: the reference value of a sample is read from LDS with the sample's gather, PIPE samples
// before it is used, instead of at its use. The half step's windows take it (one fewer wait on
// LDS per sample; it fits their registers); the evaluation and read-out, held to three waves
// per SIMD, would spill with it.
template <int WR, int WSTEP, bool CHECK, int PIPE, bool AHEAD, class REF>
__device__ __forceinline__ void window_sums(const RefWin<WR, WSTEP>& rw, const REF& ref, int x, int y, const QuadTable& qt,
                                            const float* H, float& Ss, float& SSs, float& IS) {
    constexpr int WN = Win<WR, WSTEP>::WN;
    constexpr int N = WN * WN;
    Ss = 0.f;
    SSs = 0.f;
    IS = 0.f;
    // A rolling pipeline over the row-major samples: the gather of sample k + PIPE is issued before
    // sample k is used up, so PIPE gathers stay in flight. The sums take the samples in row-major
    // order.
    float fx[N], fy[N], rv[N];
    QuadEntry qv[N];
    float rz = 0.f, ru = 0.f, rt = 0.f;  // the issued row's projective terms at dx = 0
    auto xoff = [](int k) { return -WR + (k % WN) * WSTEP; };
    auto yoff = [](int k) { return -WR + (k / WN) * WSTEP; };
    auto row = [&](int k) {
        const float oy = (float)yoff(k);
        rz = fmaf(H[7], oy, H[8]);
        ru = fmaf(H[1], oy, H[2]);
        rt = fmaf(H[4], oy, H[5]);
    };
    auto issue = [&](int k) {
        if (k % WN == 0) row(k);
        if constexpr (AHEAD) rv[k] = ref.at(x + xoff(k), y + yoff(k));
        const float ox = (float)xoff(k);
        const float r = rcp_sample(fmaf(H[6], ox, rz));
        qv[k] = quad_fetch(qt, fmaf(H[0], ox, ru) * r, fmaf(H[3], ox, rt) * r, fx[k], fy[k]);
    };
#pragma unroll
    for (int k = 0; k < PIPE && k < N; ++k) issue(k);
#pragma unroll
    for (int k = 0; k < N; ++k) {
        // the operations of issue(n) and those on sample k in turn: written one after the other,
        // the compiler needs more registers and spills at three waves per SIMD (half step 21.4
        // instead of 20.0 ms on 9 views of 1920 x 1080); at two waves the order makes no difference
        const int n = k + PIPE < N ? k + PIPE : N - 1;
        const bool more = k + PIPE < N;
        float zz, r, e, u, v, xf, yf;
        if (more) {
            if (n % WN == 0) row(n);
            if constexpr (AHEAD) rv[n] = ref.at(x + xoff(n), y + yoff(n));
            zz = fmaf(H[6], (float)xoff(n), rz);
        }
        if (more) {
            r = rcp_seed(zz);
            e = fmaf(-zz, r, 1.0f);
        }
        half2_t p, d;
        quad_rows(qv[k], p, d);
        if (more) {
            e = fmaf(e, e, e);
            r = fmaf(r, e, r);
        }
        const float top = fmaf(fx[k], (float)d.x, (float)p.x);
        if (more) e = fmaf(-zz, r, 1.0f);
        const float bot = fmaf(fx[k], (float)d.y, (float)p.y);
        if (more) u = fmaf(H[0], (float)xoff(n), ru);
        const float dv = bot - top;
        if (more) r = fmaf(r, e, r);
        float sv = fmaf(fy[k], dv, top);
        if (CHECK) sv = fmaf(H[6], (float)xoff(k), fmaf(H[7], (float)yoff(k), H[8])) > 1e-8f ? sv : 0.0f;
        if (more) v = fmaf(H[3], (float)xoff(n), rt);
        const float sp = sv - rw.ic;
        if (more) u = u * r;
        const float ws = rw.w[k] * sp;
        if (more) {
            v = v * r;
            xf = floorf(u);
        }
        Ss += ws;
        if (more) yf = floorf(v);
        SSs = fmaf(ws, sp, SSs);
        if (more) fx[n] = u - xf;
        IS = fmaf(ws, AHEAD ? rv[k] : ref.at(x + xoff(k), y + yoff(k)), IS);
        if (more) {
            xf = __builtin_amdgcn_fmed3f(xf, -2.0f, qt.w);
            fy[n] = v - yf;
            yf = __builtin_amdgcn_fmed3f(yf, -2.0f, qt.h);
            qv[n] = quad_load(qt, xf, yf);
        }
    }
}

// window_sums as a loop over the rows, each in groups of CH samples whose gathers are issued together,
// that forms the bilateral weights again; same values and order. Two uses:
// Windows of more than 49 samples (the quality profile's (5, 1)), whose weights registers cannot
// hold: with the window known at compile time the offsets are constants, the reference reads carry
// theirs as immediates and the samples in front of the source need no check. 2 iterations of 3 views
// with 3 sources against the kernels of any radius: 641 x 479 13.3 -> 12.1 ms, geometric 16.4 ->
// 11.5 ms, 1281 x 959 46.8 -> 37.5 ms. Half of a sample's VALU instructions are its weight.
// Whole rows at three waves per SIMD; two waves measured 12.8 ms, four (spills) 12.4 ms, half
// rows at four 13.0 ms.
// Windows with CHECK. Windows that need the check are rare (0.4 to 2 % of a wave's windows have
// such a lane, over runs on 1920 x 1080 and 960 x 540 views). A second unrolled copy of the window
// beside the first one costs registers all the same (the compiler hoists what the two have in
// common above the branch: 247 VGPRs instead of 192 in the photometric half step) and drains the
// first gathers there. Groups of one sample measured 2 % slower on one 960 x 540 view, of six
// 3 % slower on 9 views of 1920 x 1080 (spills).
template <int WR, int WSTEP, bool CHECK, int CH, class REF>
__device__ __forceinline__ void window_rows(const KParams& P, const RefWin<WR, WSTEP>& rw, const REF& ref, int x, int y,
                                                   const QuadTable& qt, const float* H,
                                                   float& Ss, float& SSs, float& IS) {
    constexpr int WN = Win<WR, WSTEP>::WN;
    Ss = 0.f;
    SSs = 0.f;
    IS = 0.f;
#pragma unroll 1
    for (int a = 0; a < WN; ++a) {
        const int dy = -WR + a * WSTEP;
        const float oy = (float)dy;
        const float rz = fmaf(H[7], oy, H[8]), ru = fmaf(H[1], oy, H[2]), rv = fmaf(H[4], oy, H[5]);
#pragma unroll 1
        for (int b0 = 0; b0 < WN; b0 += CH) {
            float fx[CH], fy[CH], zs[CH];
            QuadEntry qv[CH];
#pragma unroll
            for (int g = 0; g < CH; ++g) {
                const float ox = (float)(-WR + (b0 + g) * WSTEP);
                zs[g] = fmaf(H[6], ox, rz);
                const float r = rcp_sample(zs[g]);
                qv[g] = quad_fetch(qt, fmaf(H[0], ox, ru) * r, fmaf(H[3], ox, rv) * r, fx[g], fy[g]);
            }
#pragma unroll
            for (int g = 0; g < CH; ++g) {
                if (WN % CH != 0 && b0 + g >= WN) break;
                const int dx = -WR + (b0 + g) * WSTEP;
                const float sv = !CHECK || zs[g] > 1e-8f ? quad_lerp(qv[g], fx[g], fy[g]) : 0.0f;
                const float iv = ref.at(x + dx, y + dy);
                const float sp = sv - rw.ic;
                const float ws = bilateral_weight(P, rw.ic, iv, dx, dy) * sp;
                Ss += ws;
                SSs = fmaf(ws, sp, SSs);
                IS = fmaf(ws, iv, IS);
            }
        }
    }
}

// Bilateral-weighted NCC cost 1 - rho, 2 on failure (patchmatch.cu:244-290); the covariance is
// sum(w s' I)/W - mu mean(s') with s' the shifted source samples.
// COPY: windows with a sample behind the source take an unrolled copy of the window (short latency,
// many registers) instead of the loop.
template <int WR, int WSTEP, int PIPE = WINDOW_PIPE, bool AHEAD = false, bool COPY = false, class REF>
__device__ __forceinline__ float ncc_cost(const KParams& P, const RefWin<WR, WSTEP>& rw, const REF& ref, const LevelDesc& S,
                                          const float* H, int x, int y) {
    float z = H[8];
    if (!(z > 1e-8f)) return 2.0f;
    const float iz = z < EXACT_HI ? inv_exact(z) : 1.0f / z;
    const float u = H[2] * iz;
    const float v = H[5] * iz;
    // inside the source (a NaN position is not)
    if (!(__builtin_amdgcn_fmed3f(u, 0.f, (float)(S.w - 1)) == u && __builtin_amdgcn_fmed3f(v, 0.f, (float)(S.h - 1)) == v)) return 2.0f;
    if (rw.var < P.vmin255) return 2.0f;
    const QuadTable qt = quad_table(P, S);
    constexpr float lo = (float)(-WR), hi = (float)Win<WR, WSTEP>::LAST;
    const float za = fmaf(H[7], lo, H[8]), zb = fmaf(H[7], hi, H[8]);
    const bool all_front = fmaf(H[6], lo, za) > 1e-8f && fmaf(H[6], hi, za) > 1e-8f && fmaf(H[6], lo, zb) > 1e-8f &&
                           fmaf(H[6], hi, zb) > 1e-8f;
    float Ss, SSs, IS;
    if constexpr (!Win<WR, WSTEP>::HELD) {
        if (all_front) window_rows<WR, WSTEP, false, Win<WR, WSTEP>::WN>(P, rw, ref, x, y, qt, H, Ss, SSs, IS);
        else window_rows<WR, WSTEP, true, 3>(P, rw, ref, x, y, qt, H, Ss, SSs, IS);
    } else if (all_front) {
        window_sums<WR, WSTEP, false, PIPE, AHEAD>(rw, ref, x, y, qt, H, Ss, SSs, IS);
    } else if constexpr (COPY) {
        window_sums<WR, WSTEP, true, PIPE, AHEAD>(rw, ref, x, y, qt, H, Ss, SSs, IS);
    } else {
        window_rows<WR, WSTEP, true, 3>(P, rw, ref, x, y, qt, H, Ss, SSs, IS);
    }
    const float iW = rw.iW;
    float mus = Ss * iW;
    float vars = fmaf(-mus, mus, SSs * iW);
    if (vars < P.vmin255) return 2.0f;
    float cov = fmaf(-rw.mu, mus, IS * iW);
    // both variances lie between vmin255 and 255^2; a quotient below the exact range vanishes from 1 - rho
    const float sd = sqrt_exact(rw.var * vars);
    float cc = 1.0f - div_exact(cov, sd, inv_exact(sd));
    return fminf(fmaxf(cc, 0.0f), 2.0f);
}

// ---------------------------------------------------------------- windows of any radius

// Windows without a compiled-in build (any radius up to 20, step 1 or 2; the kernels
// instantiated with WR = 0 read the radius from KParams::wr): the bilateral weight of a sample is
// recomputed where it is used, as the reference does for windows above 36 samples
// (patchmatch.cu:47,153-165). Every operation and its order match the register-resident path, so
// both give identical results for the same radius.
struct RefWinDyn {
    float ic, mu, W, iW, var;
    int wr;
};

struct RefTileDyn {
    const float* s;
    int x0, y0, pitch;
    __device__ __forceinline__ float at(int x, int y) const { return s[(y - y0) * pitch + (x - x0)]; }
};

template <int WR, int WSTEP>
using RefWinT = typename std::conditional<(WR > 0), RefWin<WR, WSTEP>, RefWinDyn>::type;

template <int WSTEP, class REF>
__device__ void ref_stats_dyn(const KParams& P, const REF& ref, int x, int y, int wr, RefWinDyn& rw) {
    const int wn = (2 * wr) / WSTEP + 1;
    rw.ic = ref.at(x, y);
    rw.wr = wr;
    float W = 0.0f, S = 0.0f;
    for (int a = 0; a < wn; ++a) {
        const int dy = -wr + a * WSTEP;
        for (int b = 0; b < wn; ++b) {
            const int dx = -wr + b * WSTEP;
            float v = ref.at(x + dx, y + dy);
            float w = bilateral_weight(P, rw.ic, v, dx, dy);
            W += w;
            S = fmaf(w, v, S);
        }
    }
    float mu = S / W;
    float V = 0.0f;
    for (int a = 0; a < wn; ++a) {
        const int dy = -wr + a * WSTEP;
        for (int b = 0; b < wn; ++b) {
            const int dx = -wr + b * WSTEP;
            float v = ref.at(x + dx, y + dy);
            float dk = v - mu;
            float wd = bilateral_weight(P, rw.ic, v, dx, dy) * dk;
            V = fmaf(wd, dk, V);
        }
    }
    rw.mu = mu;
    rw.W = W;
    rw.iW = 1.0f / W;
    rw.var = V / W;
}

constexpr int DYN_GROUP = 6;
template <int WSTEP, class REF>
__device__ float ncc_cost_dyn(const KParams& P, const RefWinDyn& rw, const REF& ref, const LevelDesc& S, const float* H, int x,
                              int y) {
    float z = H[8];
    if (!(z > 1e-8f)) return 2.0f;
    const float iz = z < EXACT_HI ? inv_exact(z) : 1.0f / z;
    const float u = H[2] * iz;
    const float v = H[5] * iz;
    // inside the source (a NaN position is not)
    if (!(__builtin_amdgcn_fmed3f(u, 0.f, (float)(S.w - 1)) == u && __builtin_amdgcn_fmed3f(v, 0.f, (float)(S.h - 1)) == v)) return 2.0f;
    if (rw.var < P.vmin255) return 2.0f;
    const QuadTable qt = quad_table(P, S);
    const int wr = rw.wr, wn = (2 * wr) / WSTEP + 1;
    float Ss = 0.f, SSs = 0.f, IS = 0.f;
    for (int a = 0; a < wn; ++a) {
        const int dyi = -wr + a * WSTEP;
        const float oy = (float)dyi;
        const float rz = fmaf(H[7], oy, H[8]);
        const float ru = fmaf(H[1], oy, H[2]);
        const float rv = fmaf(H[4], oy, H[5]);
        // G samples from b0 on: their gathers are issued before the first is used (the barrier keeps
        // the compiler from waiting for each in turn). Groups of six at three waves per SIMD against the
        // loop over single samples at two, 2 iterations of 3 views with 3 sources: 641 x 479 window
        // (7, 2) 8.0 -> 7.65 ms, geometric 10.3 -> 8.5 ms; (5, 1) 13.3 -> 12.5 and 16.4 -> 13.0 ms;
        // 1281 x 959 (5, 1) 46.8 -> 41.5 ms. Groups of four: 13.1, 13.5 and 43.4 ms for the last three.
        auto group = [&](int b0, auto g) {
            constexpr int G = decltype(g)::value;
            QuadEntry qs[G];
            float fx[G], fy[G], zs[G];
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const float ox = (float)(-wr + (b0 + i) * WSTEP);
                zs[i] = fmaf(H[6], ox, rz);
                const float r = rcp_sample(zs[i]);
                qs[i] = quad_fetch(qt, fmaf(H[0], ox, ru) * r, fmaf(H[3], ox, rv) * r, fx[i], fy[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int dxi = -wr + (b0 + i) * WSTEP;
                const float sv = zs[i] > 1e-8f ? quad_lerp(qs[i], fx[i], fy[i]) : 0.0f;
                const float iv = ref.at(x + dxi, y + dyi);
                const float sp = sv - rw.ic;
                const float ws = bilateral_weight(P, rw.ic, iv, dxi, dyi) * sp;
                Ss += ws;
                SSs = fmaf(ws, sp, SSs);
                IS = fmaf(ws, iv, IS);
            }
        };
        int b = 0;
#pragma unroll 1
        for (; b + DYN_GROUP <= wn; b += DYN_GROUP) group(b, std::integral_constant<int, DYN_GROUP>{});
        const int rest = wn - b;
        if (rest == 1) group(b, std::integral_constant<int, 1>{});
        else if (rest == 2) group(b, std::integral_constant<int, 2>{});
        else if (rest == 3) group(b, std::integral_constant<int, 3>{});
        else if (rest == 4) group(b, std::integral_constant<int, 4>{});
        else if (rest == 5) group(b, std::integral_constant<int, 5>{});
    }
    const float iW = rw.iW;
    float mus = Ss * iW;
    float vars = fmaf(-mus, mus, SSs * iW);
    if (vars < P.vmin255) return 2.0f;
    float cov = fmaf(-rw.mu, mus, IS * iW);
    // both variances lie between vmin255 and 255^2; a quotient below the exact range vanishes from 1 - rho
    const float sd = sqrt_exact(rw.var * vars);
    float cc = 1.0f - div_exact(cov, sd, inv_exact(sd));
    return fminf(fmaxf(cc, 0.0f), 2.0f);
}

// Dispatch between the register-resident window (WR > 0) and the window of any radius (WR = 0).
template <int WR, int WSTEP, class REF>
__device__ __forceinline__ void ref_stats_any(const KParams& P, const REF& ref, int x, int y, int wr, RefWinT<WR, WSTEP>& rw) {
    if constexpr (WR > 0) ref_stats<WR, WSTEP>(P, ref, x, y, rw);
    else ref_stats_dyn<WSTEP>(P, ref, x, y, wr, rw);
}

template <int WR, int WSTEP, int PIPE = WINDOW_PIPE, bool AHEAD = false, bool COPY = false, class REF>
__device__ __forceinline__ float ncc_cost_any(const KParams& P, const RefWinT<WR, WSTEP>& rw, const REF& ref, const LevelDesc& S,
                                              const float* H, int x, int y) {
    if constexpr (WR > 0) return ncc_cost<WR, WSTEP, PIPE, AHEAD, COPY>(P, rw, ref, S, H, x, y);
    else return ncc_cost_dyn<WSTEP>(P, rw, ref, S, H, x, y);
}

// Forward-backward reprojection error through the source depth snapshot (patchmatch.cu:292-314).
// geo_error in two halves: geo_fetch projects the pixel at depth d into the source and issues the
// load of the source's snapshot depth at the nearest pixel; geo_finish back-projects it and
// returns the reprojection distance. A caller can put other work between the two, so that the
// load's latency is hidden; geo_finish(geo_fetch(...)) is geo_error exactly.
struct GeoFetch {
    float u, v, dj;
    bool ok;  // false: the result is INF_ERR
};

__device__ __forceinline__ GeoFetch geo_fetch(const KParams& P, const LevelDesc& R, const LevelDesc& S, const PairRec& pr, int x,
                                              int y, float d) {
    GeoFetch g{0.f, 0.f, 0.f, false};
    long long off = P.snap_off[pr.src];
    if (off < 0) return g;
    f3 X = mk3(((float)x - R.cx) / R.fx * d, ((float)y - R.cy) / R.fy * d, d);
    float xj = pr.r[0] * X.x + pr.r[1] * X.y + pr.r[2] * X.z + pr.t[0];
    float yj = pr.r[3] * X.x + pr.r[4] * X.y + pr.r[5] * X.z + pr.t[1];
    float zj = pr.r[6] * X.x + pr.r[7] * X.y + pr.r[8] * X.z + pr.t[2];
    if (!(zj > 1e-8f)) return g;
    float u, v;
    if (zj < EXACT_HI) {  // an overflow is outside the source as NaN too
        const float iz = inv_exact(zj);
        u = div_exact(S.fx * xj, zj, iz) + S.cx;
        v = div_exact(S.fy * yj, zj, iz) + S.cy;
    } else {
        u = S.fx * xj / zj + S.cx;
        v = S.fy * yj / zj + S.cy;
    }
    float uf = floorf(u + 0.5f), vf = floorf(v + 0.5f);
    if (!(uf >= 0.f && vf >= 0.f && uf < (float)S.w && vf < (float)S.h)) return g;
    g.dj = P.snap[off + (long long)vf * S.w + (long long)uf];
    g.u = u;
    g.v = v;
    g.ok = true;
    return g;
}

__device__ __forceinline__ float geo_finish(const LevelDesc& R, const LevelDesc& S, const PairRec& pr, int x, int y, const GeoFetch& g) {
    if (!g.ok) return INF_ERR;
    const float dj = g.dj, u = g.u, v = g.v;
    if (!(dj > 0.f)) return INF_ERR;
    f3 Yj;
    if (S.plain) Yj = mk3(div_exact(u - S.cx, S.fx, S.ifx) * dj, div_exact(v - S.cy, S.fy, S.ify) * dj, dj);
    else Yj = mk3((u - S.cx) / S.fx * dj, (v - S.cy) / S.fy * dj, dj);
    f3 q = mk3(Yj.x - pr.t[0], Yj.y - pr.t[1], Yj.z - pr.t[2]);
    float Yx = pr.r[0] * q.x + pr.r[3] * q.y + pr.r[6] * q.z;
    float Yy = pr.r[1] * q.x + pr.r[4] * q.y + pr.r[7] * q.z;
    float Yz = pr.r[2] * q.x + pr.r[5] * q.y + pr.r[8] * q.z;
    if (!(Yz > 1e-8f)) return INF_ERR;
    const float nx = R.fx * Yx, ny = R.fy * Yy;
    float ex, ey;
    // numerators below 2^100 over a divisor above 1e-8: quotients below 2^127
    if (fmaxf(Yz, fmaxf(fabsf(nx), fabsf(ny))) < EXACT_HI) {
        const float iz = inv_exact(Yz);
        ex = div_exact(nx, Yz, iz) + R.cx - (float)x;
        ey = div_exact(ny, Yz, iz) + R.cy - (float)y;
    } else {
        ex = nx / Yz + R.cx - (float)x;
        ey = ny / Yz + R.cy - (float)y;
    }
    return sqrtf(ex * ex + ey * ey);
}

__device__ __forceinline__ float geo_error(const KParams& P, const LevelDesc& R, const LevelDesc& S, const PairRec& pr, int x, int y,
                                           float d) {
    return geo_finish(R, S, pr, x, y, geo_fetch(P, R, S, pr, x, y, d));
}

// (photometric cost, truncated geometric error) of one hypothesis x one source (patchmatch.cu:316-324)
// In geometric runs the snapshot depth is fetched before the NCC window and used after it.
template <int WR, int WSTEP, int PIPE = WINDOW_PIPE, class REF>
__device__ __forceinline__ float pair_cost(const KParams& P, const RefWinT<WR, WSTEP>& rw, const REF& ref, const LevelDesc& R,
                                           const LevelDesc& S, const PairRec& pr, const LevelPair& lp, int x, int y, float4 h,
                                           float* geo) {
    float H[9];
    float c = 2.0f;
    GeoFetch gf{0.f, 0.f, 0.f, false};
    if (P.geometric) gf = geo_fetch(P, R, S, pr, x, y, h.w);
    if (homography(R, lp, R.ifx, R.ify, (float)x, (float)y, h.w, xyz(h), H))
        c = ncc_cost_any<WR, WSTEP, PIPE>(P, rw, ref, S, H, x, y);
    if (P.geometric) *geo = fminf(geo_finish(R, S, pr, x, y, gf), P.gmax);
    return c;
}

// ---------------------------------------------------------------- random hypotheses

// patchmatch.cu:347-361
__device__ __forceinline__ f3 random_normal(unsigned long long& st, f3 ray) {
    f3 n = mk3(0.f, 0.f, -1.f);
    for (int k = 0; k < 64; ++k) {
        float v1 = 2.f * rnd(st) - 1.f;
        float v2 = 2.f * rnd(st) - 1.f;
        float s = v1 * v1 + v2 * v2;
        if (s < 1.f && s > 0.f) {
            float r = 2.f * sqrtf(1.f - s);
            n = mk3(v1 * r, v2 * r, 1.f - 2.f * s);
            break;
        }
    }
    if (dot3(n, ray) > 0.f) n = mk3(-n.x, -n.y, -n.z);
    return n;
}

// patchmatch.cu:363-366
__device__ __forceinline__ float random_depth(unsigned long long& st, float dmin, float dmax) {
    float a = 1.f / dmax, b = 1.f / dmin;
    return 1.f / (a + rnd(st) * (b - a));
}

// patchmatch.cu:368-384
__device__ __forceinline__ f3 perturb_normal(unsigned long long& st, f3 n, f3 ray, float phi) {
    f3 a = random_normal(st, mk3(0.f, 0.f, 0.f));
    f3 ax = cross3(a, n);
    float l2 = dot3(ax, ax);
    float ang = rnd(st) * phi;
    if (l2 < 1e-12f) return n;
    ax = nrm3(ax);
    f3 bn = cross3(ax, n);
    for (int k = 0; k < 4; ++k) {
        float sa, ca;
        c3d_sincosf(ang, sa, ca);
        f3 m = mk3(n.x * ca + bn.x * sa, n.y * ca + bn.y * sa, n.z * ca + bn.z * sa);
        if (dot3(m, ray) < 0.f) return nrm3(m);
        ang *= 0.5f;
    }
    return n;
}

// triangulation x incidence x resolution prior (patchmatch.cu:388-422); r = window radius
__device__ __forceinline__ float view_prior(const KParams& P, const LevelDesc& R, const PairRec& pr, const float* H, bool hok, int x,
                                            int y, float4 h, float r) {
    if (!hok) return 0.f;
    f3 ray = pixel_ray(R, x, y);
    f3 X = mk3(ray.x * h.w, ray.y * h.w, h.w);
    f3 S = mk3(pr.c[0] - X.x, pr.c[1] - X.y, pr.c[2] - X.z);
    float ls = sqrtf(dot3(S, S)), lx = sqrtf(dot3(X, X));
    if (ls <= 0.f || lx <= 0.f) return 0.f;
    float cost = -dot3(S, X) / (ls * lx);
    float tri = 1.f;
    if (cost > P.cos_tri_min) {
        float s = 1.f - (1.f - cost) / (1.f - P.cos_tri_min);
        tri = fminf(fmaxf(1.f - s * s, 0.f), 1.f);
    }
    float cphi = dot3(S, xyz(h)) / ls;
    float xi = 1.f - fmaxf(0.f, cphi);
    float inc = c3d_expf(-xi * xi * P.inv2inc);
    const float cxs[4] = {-r, -r, r, r};
    const float cys[4] = {-r, r, r, -r};
    float px[4], py[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float z = H[6] * cxs[k] + H[7] * cys[k] + H[8];
        if (!(z > 1e-8f)) return 0.f;
        px[k] = (H[0] * cxs[k] + H[1] * cys[k] + H[2]) / z;
        py[k] = (H[3] * cxs[k] + H[4] * cys[k] + H[5]) / z;
    }
    float area = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) area += px[k] * py[(k + 1) & 3] - px[(k + 1) & 3] * py[k];
    area = 0.5f * fabsf(area);
    float aref = (2.f * r + 1.f) * (2.f * r + 1.f);
    if (!(area > 0.f)) return 0.f;
    float res = fminf(area / aref, aref / area);
    return tri * inc * res;
}

// ---------------------------------------------------------------- run start

// The plane a run starts from (mode 1: initialised where random_init says so, patchmatch.cu:668-677).
__device__ __forceinline__ float4 eval_init_plane(const KParams& P, const ViewDesc& vd, const LevelDesc& R, int x, int y, int pix,
                                                  long long base, int mode) {
    float4 h = P.plane[base + pix];
    // random_init 1: every pixel (patchmatch.cu:668-676); 2: pixels without a positive depth
    if (mode == 1 && (P.random_init == 1 || (P.random_init == 2 && !(h.w > 0.f)))) {
        unsigned long long st = rng_state(P.seed, vd.key, P.level, P.run_id, 0xFFFF, 0, (unsigned long long)pix);
        float d = random_depth(st, vd.dmin, vd.dmax);
        f3 n = random_normal(st, pixel_ray(R, x, y));
        h = mk4(n, d);
        P.plane[base + pix] = h;
    }
    return h;
}

}  // namespace entry4 / entry8
}  // namespace c3d
