// pm_kernels.hip — gfx950 PatchStereo kernels without a matching window (run start, upsampling, median
// filter, restorer, threshold, pyramid, state transfers), the tile counts and their launchers.
// The kernels follow the rules of the reference's crates/cuda/src/kernels/patchmatch.cu (cited per
// kernel); the window kernels are in pm_windows.hip.
#include "pm_device.hpp"
#include "pm_kernels.hpp"

namespace c3d {

// The batch item holding pixel g of the flattened batch, by a binary search over the items' pixel
// offsets (stored in increasing order); false for a pixel outside every item. Per-pixel passes use
// it instead of locate_tile: a few loads per thread, where a workgroup's linear search over the
// items for its tile costs more than a light pass itself on a 108-view batch.
__device__ __forceinline__ bool locate_pixel(const KParams& P, long long g, BatchItem& it, int& item, int& pix) {
    int lo = 0, hi = P.nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (P.batch[mid].off <= g) lo = mid;
        else hi = mid - 1;
    }
    it = P.batch[lo];
    item = lo;
    if (g < it.off || g - it.off >= (long long)it.w * it.h) return false;
    pix = (int)(g - it.off);
    return true;
}

// The window-free part of a run start for every pixel: random initialisation by random_init and
// the best-view reset (patchmatch.cu:668-677). Stored costs are not touched. One thread per pixel
// of the flattened batch.
__global__ __launch_bounds__(256) void k_eval_init(KParams P, long long npix) {
    const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
    if (g >= npix) return;
    BatchItem it;
    int item, pix;
    if (!locate_pixel(P, g, it, item, pix)) return;
    const int y = pix / it.w, x = pix - y * it.w;
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    const ViewDesc vd = P.views[it.view];
    eval_init_plane(P, vd, R, x, y, pix, it.off, 1);
    P.bview[it.off + pix] = 255;
}

// ================================================================ plane records in LDS
//
// Both scale-change kernels below transfer a neighbour's plane onto a pixel's own viewing ray.
// The neighbour q (plane normal n_q, depth d_q on its ray r_q) holds the plane n_q . X = c_q with
// c_q = d_q (n_q . r_q), so the depth it gives pixel p is c_q / (n_q . r_p) (patchmatch.cu:405-412
// transfer, same f32 operations and order). A workgroup therefore stages, once, the records
// (n_q, c_q) of every neighbour its pixels can reach; c_q is NaN for a missing neighbour (outside
// the image, or d_q not > 0), which every later test rejects exactly as the explicit checks would.

__device__ __forceinline__ float4 plane_record(float4 q, f3 ray_q) {
    const f3 n = xyz(q);
    const float c = q.w > 0.f ? q.w * dot3(n, ray_q) : __int_as_float(0x7fc00000);
    return mk4(n, c);
}

// ================================================================ joint bilateral upsampling
// Output rules of pm_upsample (patchmatch.cu:739-801, upsample.rs:104-175): every low-resolution
// neighbour in the 5 x 5 block around the pixel's position at the lower scale whose transferred depth
// is positive and finite contributes exp(-ds/(2 sigma_s^2) - (I_p - I_q)^2/(2 sigma_c^2)) in scan
// order; with no weight the nearest such neighbour (first in scan order on ties) is taken; the
// normal is normalised and turned towards the camera.
//
// A 64 x 4 pixel tile reaches the low-resolution columns [x0/2 - 2, x0/2 + 33] and rows
// [y0/2 - 2, y0/2 + 3]: 36 x 6 plane records and gray levels are staged in LDS by the whole
// workgroup, so each of the 25 taps of a pixel is two LDS reads instead of a float4 and a byte
// gather from global memory with its own transfer arithmetic.
constexpr int UP_CW = PIX_TW / 2 + 4;  // 36 staged low-resolution columns
constexpr int UP_CH = PIX_TH / 2 + 4;  // 6 staged rows

__global__ __launch_bounds__(256) void k_upsample(KParams P) {
    __shared__ float4 rec[UP_CH * UP_CW];
    __shared__ float lgray[UP_CH * UP_CW];
    BatchItem it;
    int px0, py0;
    if (!find_tile(P, xcd_tile(blockIdx.x, P.ntiles), PIX_TW, PIX_TH, it, px0, py0)) return;  // uniform per workgroup
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    const LevelDesc L = P.lv[it.view * P.nlevels + P.level - 1];
    const float4* low = P.prior + it.low_off;
    const int qxa = px0 / 2 - 2, qya = py0 / 2 - 2;  // first staged low-resolution column and row
    for (int k = threadIdx.x; k < UP_CH * UP_CW; k += 256) {
        const int qx = qxa + k % UP_CW, qy = qya + k / UP_CW;
        float4 r = make_float4(0.f, 0.f, 0.f, __int_as_float(0x7fc00000));
        float g = 0.f;
        if (qx >= 0 && qx < L.w && qy >= 0 && qy < L.h) {
            r = plane_record(low[qy * L.w + qx], pixel_ray(L, qx, qy));
            g = (float)P.gray[L.goff + (size_t)qy * L.w + qx] * (1.0f / 255.0f);
        }
        rec[k] = r;
        lgray[k] = g;
    }
    __syncthreads();
    const int x = px0 + (threadIdx.x & 63), y = py0 + (threadIdx.x >> 6);
    if (x >= it.w || y >= it.h) return;
    const f3 rp = pixel_ray(R, x, y);
    const float ip = (float)P.gray[R.goff + (size_t)y * R.w + x] * (1.0f / 255.0f);
    const float px = ((float)x - 0.5f) * 0.5f, py = ((float)y - 0.5f) * 0.5f;
    const int qx0 = (int)roundf(px), qy0 = (int)roundf(py);
    float sw = 0.f, sd = 0.f, snx = 0.f, sny = 0.f, snz = 0.f;
    float nd = 1e30f, ndep = 0.f;
    f3 nn = mk3(0.f, 0.f, 0.f);
#pragma unroll
    for (int dy = -2; dy <= 2; ++dy) {
        const int qy = qy0 + dy;
        const int row = (qy - qya) * UP_CW - qxa;
#pragma unroll
        for (int dx = -2; dx <= 2; ++dx) {
            const int qx = qx0 + dx;
            const float4 r = rec[row + qx];
            const f3 nq = xyz(r);
            const float den = dot3(nq, rp);
            const float d = r.w / den;
            if (!(den < -1e-6f) || !(d > 0.f) || !isfinite(d)) continue;
            const float ds = ((float)qx - px) * ((float)qx - px) + ((float)qy - py) * ((float)qy - py);
            if (ds < nd) {
                nd = ds;
                ndep = d;
                nn = nq;
            }
            const float iq = lgray[row + qx];
            const float wgt = c3d_expf(-ds * P.up_inv2s - (ip - iq) * (ip - iq) * P.up_inv2c);
            sw += wgt;
            sd += wgt * d;
            snx += wgt * nq.x;
            sny += wgt * nq.y;
            snz += wgt * nq.z;
        }
    }
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    const bool weighted = sw > 1e-12f;
    if (weighted || nd < 1e29f) {
        const float d = weighted ? sd / sw : ndep;
        f3 nv = weighted ? mk3(snx, sny, snz) : nn;
        if (dot3(nv, nv) > 1e-24f) {
            nv = nrm3(nv);
            if (dot3(nv, rp) >= 0.f) nv = mk3(-nv.x, -nv.y, -nv.z);
            o = mk4(nv, d);
        }
    }
    P.plane[it.off + y * it.w + x] = o;
}

// ================================================================ 5 x 5 median plane filter
// Output rule of pm_median (patchmatch.cu:803-849, upsample.rs:177-260): a pixel with a positive
// depth takes, among the neighbours of its 5 x 5 block (clipped to the image) whose plane transfers
// to a positive finite depth on its ray, the lower median of those depths, ties ordered by pixel
// index; its output is that neighbour's normal with the transferred depth. Other pixels keep their
// plane.
//
// The 64 x 4 tile and its 2-pixel halo (68 x 8 records) are staged in LDS. Each pixel then holds
// its 25 candidate depths in registers (a rejected one as +inf) and picks the median by rank:
// candidate k has rank #{j > k : d_j < d_k} + #{j < k : d_j <= d_k} (slot order is pixel-index
// order, so this is the index tie-break), and the candidate of rank (count - 1) / 2 is the median.
// No data-dependent branches or register indexing: every lane does the same 600 comparisons.
constexpr int MED_CW = PIX_TW + 4;
constexpr int MED_CH = PIX_TH + 4;

__global__ __launch_bounds__(256) void k_median(KParams P) {
    __shared__ float4 rec[MED_CH * MED_CW];
    BatchItem it;
    int px0, py0;
    if (!find_tile(P, xcd_tile(blockIdx.x, P.ntiles), PIX_TW, PIX_TH, it, px0, py0)) return;  // uniform per workgroup
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    const float4* in = P.prior + it.off;
    const int w = it.w, h = it.h;
    const int xa = px0 - 2, ya = py0 - 2;
    for (int k = threadIdx.x; k < MED_CH * MED_CW; k += 256) {
        const int qx = xa + k % MED_CW, qy = ya + k / MED_CW;
        float4 r = make_float4(0.f, 0.f, 0.f, __int_as_float(0x7fc00000));
        if (qx >= 0 && qx < w && qy >= 0 && qy < h) r = plane_record(in[qy * w + qx], pixel_ray(R, qx, qy));
        rec[k] = r;
    }
    __syncthreads();
    const int x = px0 + (threadIdx.x & 63), y = py0 + (threadIdx.x >> 6);
    if (x >= w || y >= h) return;
    const float4 self = in[y * w + x];
    float4 out = self;
    if (self.w > 0.f) {
        const f3 rp = pixel_ray(R, x, y);
        const int base = (y - ya - 2) * MED_CW + (x - xa - 2);
        float d[25];
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < 25; ++k) {
            const float4 r = rec[base + (k / 5) * MED_CW + k % 5];
            const float den = dot3(xyz(r), rp);
            const float t = r.w / den;
            const bool ok = den < -1e-6f && t > 0.f && isfinite(t);
            d[k] = ok ? t : __int_as_float(0x7f800000);
            cnt += ok ? 1 : 0;
        }
        if (cnt > 0) {
            const int m = (cnt - 1) / 2;
            int pick = 0;
#pragma unroll
            for (int k = 0; k < 25; ++k) {
                int rank = 0;
#pragma unroll
                for (int j = 0; j < 25; ++j) {
                    if (j < k) rank += d[j] <= d[k] ? 1 : 0;
                    if (j > k) rank += d[j] < d[k] ? 1 : 0;
                }
                pick = (rank == m && d[k] < __int_as_float(0x7f800000)) ? k : pick;
            }
            float dm = d[0];
#pragma unroll
            for (int k = 1; k < 25; ++k) dm = pick == k ? d[k] : dm;
            const float4 r = rec[base + (pick / 5) * MED_CW + pick % 5];
            out = make_float4(r.x, r.y, r.z, dm);
        }
    }
    P.plane[it.off + y * w + x] = out;
}

// ================================================================ small device-side helpers

// depth channel of the planes -> snapshot buffer (same pixel layout)
__global__ void k_extract_depth(const float4* plane, float* out, long long n) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = plane[i].w;
}

// read-out threshold: depth/normal kept where depth > 0 and count >= need (densify.rs:446-454)
__global__ __launch_bounds__(256) void k_threshold(KParams P, const uint8_t* need_per_item, float4* out, long long npix) {
    const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
    if (g >= npix) return;
    BatchItem it;
    int item, pix;
    if (!locate_pixel(P, g, it, item, pix)) return;
    const long long p = it.off + pix;
    float4 h = P.plane[p];
    if (!(h.w > 0.f && P.count[p] >= need_per_item[item])) h = make_float4(0.f, 0.f, 0.f, 0.f);
    out[p] = h;
}

// detail restorer merge (densify.rs:396-409): the photometric plane replaces the upsampled one where
// the upsampled depth is not positive or c_init - c_photo > xi; the merged state carries cost 2 (the
// upsampled ViewState is ViewState::new, kernel.rs:154-159).
__global__ void k_restore(float4* plane, const float4* up, const float* c_init, float* cost, float xi, long long n) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float4 u = up[i];
    if (!(u.w <= 0.f || c_init[i] - cost[i] > xi)) plane[i] = u;
    cost[i] = 2.0f;
}

// one step of the gray pyramid (build_pyramid and blur3, crates/dense/src/upsample.rs:45-99): the
// 3-tap Gaussian (edge clamp, rows first, then columns) at the four pixels of the 2x2 cell, their
// mean, rounded half away from zero and clamped to 8 bits. Every sum runs in the reference's order.
__global__ void k_pyramid_step(const uint8_t* src, int w, int h, uint8_t* dst, float g0, float g1, float g2) {
    const int nw = w / 2, nh = h / 2;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nw * nh) return;
    const int x = i % nw, y = i / nw;
    const float g[3] = {g0, g1, g2};
    float b[4];
#pragma unroll
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
            const int X = 2 * x + dx, Y = 2 * y + dy;
            const int xa = X - 1 < 0 ? 0 : X - 1, xb = X + 1 > w - 1 ? w - 1 : X + 1;
            float a = 0.0f;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                int yy = Y + k - 1;
                yy = yy < 0 ? 0 : (yy > h - 1 ? h - 1 : yy);
                const uint8_t* r = src + (size_t)yy * w;
                float t = 0.0f;
                t += g0 * (float)r[xa];
                t += g1 * (float)r[X];
                t += g2 * (float)r[xb];
                a += g[k] * t;
            }
            b[dy * 2 + dx] = a;
        }
    const float v = 0.25f * (b[0] + b[1] + b[2] + b[3]);
    const float r = roundf(v);
    dst[i] = (uint8_t)(r < 0.f ? 0.f : (r > 255.f ? 255.f : r));
}

// The quad tables of one view-level, the 8-byte one if there is one: entry (x0, y0), x0 in [-2, w],
// y0 in [-2, h].
__global__ void k_quad_build(const uint8_t* g, int w, int h, uint32_t* q4, uint2* q8) {
    int i = blockIdx.x * 256 + threadIdx.x;
    int qp = w + 3;
    if (i >= qp * (h + 3)) return;
    int y0 = i / qp - 2, x0 = i % qp - 2;
    auto at = [&](int x, int y) -> uint32_t {
        return (x >= 0 && y >= 0 && x < w && y < h) ? (uint32_t)g[(size_t)y * w + x] : 0u;
    };
    const uint32_t p00 = at(x0, y0), p10 = at(x0 + 1, y0), p01 = at(x0, y0 + 1), p11 = at(x0 + 1, y0 + 1);
    q4[i] = quad_entry4(p00, p10, p01, p11);
    if (q8) q8[i] = quad_entry8(p00, p10, p01, p11);
}

// ================================================================ launchers

bool half_shape_ok(int rows, int tpp) { return ((rows == 1 || rows == 2) && tpp == 1) || (rows == 4 && (tpp == 1 || tpp == 2)); }

int half_tiles(const BatchItem* items, int n, int rows, int tpp) {
    const int bw = half_bw(tpp), bh = half_bh(tpp) * rows;
    int t = 0;
    for (int i = 0; i < n; ++i) t += ((items[i].w + bw - 1) / bw) * ((items[i].h + bh - 1) / bh);
    return t;
}
// Lanes per pixel of a batch when the caller asks for no shape. A launch of few waves lasts as long as
// one wave does, which is the windows of its pixels one after another: more lanes per pixel make a
// wave shorter, and cost what every lane repeats of its pixel's own work. Eight or four lanes are
// taken while the launch stays within one round of two waves per SIMD (2048), two within three rounds.
// One view with 3 sources, 2 iterations, states in and out, with 8 / 4 / 2 / 1 lanes per pixel:
// 160 x 96 0.40 / 0.51 / 0.61 / 0.92 ms (before: 0.96), 320 x 180 0.68 / 0.63 / 0.70 / 1.04,
// 480 x 270 1.16 / 1.00 / 0.90 / 1.13, 760 x 428 2.56 / 2.00 / 1.68 / 1.73, 960 x 540
// 3.91 / 2.95 / 2.38 / 2.35.
int half_lanes(const BatchItem* items, int n) {
    if (half_tiles(items, n, 1, 8) <= 2048) return 8;
    if (half_tiles(items, n, 1, 4) <= 2048) return 4;
    return half_tiles(items, n, 1, 2) <= 6144 ? 2 : 1;
}
int span_tiles(const BatchItem* items, int n) {
    int t = 0;
    for (int i = 0; i < n; ++i) t += ((items[i].w + HALF_SPAN - 1) / HALF_SPAN) * ((items[i].h + PIX_TH - 1) / PIX_TH);
    return t;
}
int pix_tiles(const BatchItem* items, int n) {
    int t = 0;
    for (int i = 0; i < n; ++i) t += ((items[i].w + PIX_TW - 1) / PIX_TW) * ((items[i].h + PIX_TH - 1) / PIX_TH);
    return t;
}

const KernelSet* kernel_set(int wr, int wstep, bool any_radius, int quad_bytes) {
    return quad_bytes == 8 ? quad8::kernel_set(wr, wstep, any_radius) : quad4::kernel_set(wr, wstep, any_radius);
}

hipError_t launch_quad_build(const uint8_t* g, int w, int h, uint32_t* q4, uint2* q8, hipStream_t s) {
    int n = (w + 3) * (h + 3);
    hipLaunchKernelGGL(k_quad_build, dim3((n + 255) / 256), dim3(256), 0, s, g, w, h, q4, q8);
    return hipGetLastError();
}

// The per-sample reciprocal of the window loops, applied to n given values (c3d_pm_sample_reciprocal).
__global__ __launch_bounds__(256) void k_sample_reciprocal(const float* z, float* r, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) r[i] = rcp_sample(z[i]);
}

hipError_t launch_sample_reciprocal(const float* z, float* r, long long n, hipStream_t s) {
    hipLaunchKernelGGL(k_sample_reciprocal, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, z, r, n);
    return hipGetLastError();
}

// a depth array and a 3-float normal array merged into planes (nx, ny, nz, d) (state uploads)
__global__ __launch_bounds__(256) void k_merge_planes(const float* depth, const float* normal, float4* plane, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) plane[i] = make_float4(normal[3 * i], normal[3 * i + 1], normal[3 * i + 2], depth[i]);
}

hipError_t launch_merge_planes(const float* depth, const float* normal, float4* plane, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_merge_planes, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, depth, normal, plane, n);
    return hipGetLastError();
}

// planes (nx, ny, nz, d) split into a depth array and a 3-float normal array (result downloads)
__global__ __launch_bounds__(256) void k_split_planes(const float4* plane, float* depth, float* normal, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        const float4 q = plane[i];
        depth[i] = q.w;
        normal[3 * i] = q.x;
        normal[3 * i + 1] = q.y;
        normal[3 * i + 2] = q.z;
    }
}

hipError_t launch_split_planes(const float4* plane, float* depth, float* normal, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_split_planes, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, plane, depth, normal, n);
    return hipGetLastError();
}

// npix: the pixels of the batch (the end of its last item)
hipError_t launch_eval_init(const KParams& P, long long npix, hipStream_t s) {
    if (npix <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_eval_init, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s, P, npix);
    return hipGetLastError();
}

hipError_t launch_upsample(const KParams& P, hipStream_t s) {
    hipLaunchKernelGGL(k_upsample, dim3(P.ntiles), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t launch_median(const KParams& P, hipStream_t s) {
    hipLaunchKernelGGL(k_median, dim3(P.ntiles), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t launch_extract_depth(const float4* plane, float* out, long long n, hipStream_t s) {
    hipLaunchKernelGGL(k_extract_depth, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, plane, out, n);
    return hipGetLastError();
}
hipError_t launch_restore(float4* plane, const float4* up, const float* c_init, float* cost, float xi, long long n,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_restore, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, plane, up, c_init, cost, xi, n);
    return hipGetLastError();
}
hipError_t launch_pyramid_step(const uint8_t* src, int w, int h, uint8_t* dst, const float g[3], hipStream_t s) {
    const int n = (w / 2) * (h / 2);
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pyramid_step, dim3((n + 255) / 256), dim3(256), 0, s, src, w, h, dst, g[0], g[1], g[2]);
    return hipGetLastError();
}
// Tile offsets of the batch items for tiles of tw x th pixels: pre[i] = tiles of the items before
// i, pre[n] = all tiles. One lane sums the counts in item order (a few hundred items at most).
__global__ void k_tile_prefix(const BatchItem* batch, int n, int tw, int th, int* pre) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    int acc = 0;
    for (int i = 0; i < n; ++i) {
        const BatchItem b = batch[i];
        pre[i] = acc;
        acc += ((b.w + tw - 1) / tw) * ((b.h + th - 1) / th);
    }
    pre[n] = acc;
}

// pre: n + 1 ints; the half step's tiles for (rows, lanes per pixel) are half_bw x (half_bh rows)
hipError_t launch_half_tile_prefix(const BatchItem* batch, int n, int rows, int tpp, int* pre, hipStream_t s) {
    hipLaunchKernelGGL(k_tile_prefix, dim3(1), dim3(64), 0, s, batch, n, half_bw(tpp), half_bh(tpp) * rows, pre);
    return hipGetLastError();
}
// the 64 x 4 tiles of k_eval (all pixels) and k_filter (pix_tiles)
hipError_t launch_pix_tile_prefix(const BatchItem* batch, int n, int* pre, hipStream_t s) {
    hipLaunchKernelGGL(k_tile_prefix, dim3(1), dim3(64), 0, s, batch, n, PIX_TW, PIX_TH, pre);
    return hipGetLastError();
}
// the 128 x 4 spans of k_eval over the pixels of one colour (span_tiles)
hipError_t launch_span_tile_prefix(const BatchItem* batch, int n, int* pre, hipStream_t s) {
    hipLaunchKernelGGL(k_tile_prefix, dim3(1), dim3(64), 0, s, batch, n, HALF_SPAN, PIX_TH, pre);
    return hipGetLastError();
}

// npix: the pixels of the batch (the end of its last item)
hipError_t launch_threshold(const KParams& P, const uint8_t* need, float4* out, long long npix, hipStream_t s) {
    if (npix <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_threshold, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s, P, need, out, npix);
    return hipGetLastError();
}

}  // namespace c3d
