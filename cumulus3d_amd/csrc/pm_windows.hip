// pm_windows.hip — the gfx950 PatchStereo kernels with a matching window (run-start and state evaluation,
// red-black half step, read-out filter, cost probe), the quad tables they sample and their launchers.
// Compiled twice, for quad entries of 4 and of 8 bytes (C3D_QUAD_BYTES), into namespaces quad4 and
// quad8; the results are the same.
//
// The kernels follow the rules of crates/dense/src/kernel.rs:36-74 as implemented by the reference's
// crates/cuda/src/kernels/patchmatch.cu (cited per kernel). Work decomposition (MI355X-specific):
//   * wave64 = the 64 active pixels (red-black: every other pixel) of a block of 16 x 8 pixels; 1, 2 or
//     4 waves per workgroup, block below block (autotuned); a workgroup stages its reference pixels
//     with the window's margin in LDS once;
//   * all views of a batch share one flattened 1-D grid of tiles (no empty blocks for smaller
//     views), remapped so that consecutive tiles run on the same XCD and share its L2;
//   * the per-thread view weights of the refinement live in LDS, everything else in VGPRs; the
//     hypothesis and source loops stay rolled so that one inlined NCC body serves all hypotheses.
#include "pm_device.hpp"
#include "pm_kernels.hpp"

#if C3D_QUAD_BYTES == 8
#define C3D_QUAD_NS quad8
#else
#define C3D_QUAD_NS quad4
#endif

namespace c3d {
namespace C3D_QUAD_NS {

// The run-start evaluation and the read-out keep five source gathers in flight through a window
// and, for register-held windows of at most 36 samples, ask for three waves per SIMD: 117-141
// VGPRs for the (5, 2) window, no spills. (The depth was chosen on an earlier window loop, which took
// 156-158 VGPRs with five and 180-187, two waves per SIMD, with eight.)
constexpr int EVAL_PIPE = 5;
template <int WR, int WSTEP>
constexpr int eval_waves() {
    return (WR > 0 && Win<(WR > 0 ? WR : 1), WSTEP>::WN2 <= 36) ? 3 : 1;
}

// region offsets for the up direction (patchmatch.cu:424-436)
__constant__ int V_OFF[7][2] = {{0, -1}, {-1, -2}, {1, -2}, {-2, -3}, {2, -3}, {-3, -4}, {3, -4}};

__device__ __forceinline__ void rot_dir(int dir, int dx, int dy, int& ox, int& oy) {
    ox = dx;
    oy = dy;
    for (int k = 0; k < dir; ++k) {
        int t = ox;
        ox = -oy;
        oy = t;
    }
}

template <int N>
__device__ __forceinline__ float4 pick4(const float4 (&a)[N], int i) {
    float4 r = a[0];
#pragma unroll
    for (int q = 1; q < N; ++q)
        if (q == i) r = a[q];
    return r;
}

// Reference tile accessor: compile-time pitch for the fixed windows, runtime pitch for WR = 0.
template <int WR, int TW>
using TileRefT = typename std::conditional<(WR > 0), RefTile<TW>, RefTileDyn>::type;

template <int WR, int TW>
__device__ __forceinline__ TileRefT<WR, TW> tile_ref(const float* tile, int x0, int y0, int pitch) {
    if constexpr (WR > 0) return RefTile<TW>{tile, x0, y0};
    else return RefTileDyn{tile, x0, y0, pitch};
}

// (photometric cost, truncated geometric error) of one hypothesis x one source with the pixel's
// reciprocal focal lengths hoisted (patchmatch.cu:316-324)
template <int WR, int WSTEP, bool GEO, int PIPE, bool AHEAD, bool COPY, class REF>
__device__ __forceinline__ float pair_cost_h(const KParams& P, const RefWinT<WR, WSTEP>& rw, const REF& ref, const LevelDesc& R,
                                             const LevelDesc& S, const PairRec& pr, const LevelPair& lp, float ifx, float ify, int x,
                                             int y, float4 h, float& geo) {
    float H[9];
    float c = 2.0f;
    // geometric runs: the snapshot depth is fetched before the NCC window and used after it
    GeoFetch gf{0.f, 0.f, 0.f, false};
    if constexpr (GEO) gf = geo_fetch(P, R, S, pr, x, y, h.w);
    if (homography(R, lp, ifx, ify, (float)x, (float)y, h.w, xyz(h), H)) c = ncc_cost_any<WR, WSTEP, PIPE, AHEAD, COPY>(P, rw, ref, S, H, x, y);
    geo = GEO ? fminf(geo_finish(R, S, pr, x, y, gf), P.gmax) : 0.f;
    return c;
}

// ================================================================ half step (patchmatch.cu:439-657)
// GEO: geometric-consistency run (the geometric term is compiled in only there).
// TPP: lanes per pixel (1, 2, 4 or 8). The lanes of a pixel (neighbours) keep their own copies of the
// pixel's state and split its NCC windows: lane j of them costs the step-2 hypotheses and the
// refinement candidates of index j modulo TPP, and the costs are exchanged; every decision is then
// taken on all of them from the same values in the same order, so the results are those of one
// lane per pixel.
// FEW: the build for launches of up to few_waves() waves, at two waves per SIMD, with more gathers in
// flight and the unrolled copy of the window (see ncc_cost). Its waves are a quarter shorter by
// themselves, and a launch of a few rounds ends with its last waves: one view of 960 x 540 (4,080
// waves) takes 2.35 instead of 2.51 ms for 2 iterations with 3 sources, 1920 x 1080 (16,200) 7.33
// instead of 7.52. Two such views (32,400) tie, and from there the three waves per SIMD of the
// other build win: 9 views of 1920 x 1080 with 6 sources 22.2 -> 20.0 ms a half step. What binds it
// is the issue of VALU instructions, which three waves keep busier (3.8 instead of 4.2 cycles an
// instruction; 2.4 of 3 wave slots taken on average). Geometric launches cross over earlier: 12 views
// of 480 x 270 (12,648 waves) with 4 sources take 11.4 ms for 3 iterations in the FEW build and 10.9
// in the other, 1280 x 720 (7,200) 6.2 ms in either, where the photometric ones take 4.8 and 5.1.
constexpr int few_waves(bool geo) { return geo ? 8192 : 16384; }
template <int WR, int WSTEP>
constexpr int half_waves(bool few) {
    if (WR == 0 || !Win<(WR > 0 ? WR : 1), WSTEP>::HELD) return 3;  // rows or groups of samples (window_rows, ncc_cost_dyn)
    return (!few && WR > 0 && Win<(WR > 0 ? WR : 1), WSTEP>::WN2 <= 36) ? 3 : 2;
}

template <int WR, int WSTEP, bool GEO, int ROWS, int TPP, bool FEW>
__global__ __launch_bounds__(ROWS * 64) __attribute__((amdgpu_waves_per_eu(half_waves<WR, WSTEP>(FEW), half_waves<WR, WSTEP>(FEW))))
void k_half(KParams P) {
    constexpr int NT = ROWS * 64;
    constexpr int BW = half_bw(TPP), BH = half_bh(TPP) * ROWS;  // pixels of the workgroup's block
    // source gathers in flight in the window loop: four for three waves per SIMD (the 168 VGPRs of
    // that and two spilled, 12 bytes of scratch a lane; deeper spills more and measures no faster),
    // six for two waves (221-237 VGPRs), fewer for the 49 register-held weights of a 7 x 7 window
    constexpr int PIPE = Win<(WR > 0 ? WR : 1), WSTEP>::WN2 > 36 ? 3 : (FEW ? 6 : 4);
    // the reference value of a window sample is read with its gather (see window_sums)
    constexpr bool AHEAD = Win<(WR > 0 ? WR : 1), WSTEP>::WN2 <= 36;
    constexpr int TW = half_pitch(TPP, WR);
    constexpr int TH = BH + 2 * WR;
    __shared__ float tile_s[WR > 0 ? TW * TH : 1];
    // per-thread hypothesis table: the 9 candidates of step 2, then the refinement candidates
    __shared__ float4 hyp_lds[9 * NT];
    // dynamic LDS: [reference tile (WR = 0 only)] [per-thread view weights]
    extern __shared__ float dyn_lds[];
    const int wr = WR > 0 ? WR : P.wr;
    const int twd = WR > 0 ? TW : half_pitch(TPP, wr), thd = BH + 2 * wr;
    float* tile = WR > 0 ? tile_s : dyn_lds;
    float* wv_lds = WR > 0 ? dyn_lds : dyn_lds + twd * thd;

    BatchItem it;
    int px0, py0;
    constexpr bool HELD = WR > 0 && Win<(WR > 0 ? WR : 1), WSTEP>::HELD;
    if (!find_tile(P, xcd_tile<HELD ? XCD_RUN : XCD_RUN_ROW>(blockIdx.x, P.ntiles), BW, BH, it, px0, py0, HELD ? HALF_BAND / ROWS : 1)) return;
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    const int w = it.w, h = it.h;
    {
        const uint8_t* g = P.gray + R.goff;
        const int tx0 = px0 - wr, ty0 = py0 - wr;
        for (int i = threadIdx.x; i < twd * thd; i += NT) {
            int ty = i / twd, tx = i - ty * twd;
            int gx = tx0 + tx, gy = ty0 + ty;
            tile[i] = (gx >= 0 && gy >= 0 && gx < w && gy < h) ? (float)g[(size_t)gy * w + gx] : 0.0f;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int sub = lane & (TPP - 1);  // this lane's share of the pixel's windows
    int col, row;
    block_pixel<TPP>(lane / TPP, col, row);
    const int y = py0 + half_bh(TPP) * (int)(threadIdx.x >> 6) + row;
    const int x = px0 + 2 * col + ((y + P.color) & 1);
    if (x >= w || y >= h) return;  // both lanes of a pixel leave together

    const auto ref = tile_ref<WR, TW>(tile, px0 - wr, py0 - wr, twd);
    const ViewDesc vd = P.views[it.view];
    const int nsrc = vd.nsrc;
    const PairRec* prs = P.pairs + (size_t)it.view * MAXSRC;
    const LevelPair* lps = P.lpairs + ((size_t)it.view * P.nlevels + P.level) * MAXSRC;
    const long long base = it.off;
    const int pix = y * w + x;
    float4* pl = P.plane + base;
    const float* co = P.cost + base;
    const f3 ray = pixel_ray(R, x, y);
    const float ifx = R.ifx, ify = R.ify;
    float* wv = wv_lds + threadIdx.x;
    float4* hyp = hyp_lds + threadIdx.x;  // hyp[i * NT]

    // 1. candidates: current + best of 8 regions (patchmatch.cu:477-511). The 72 neighbour costs
    //    are loaded unconditionally (out-of-image offsets read the pixel's own cost and are ignored).
    const float4 hyp0 = pl[pix];
    hyp[0] = hyp0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int dir = r & 3;
        const bool strip = r >= 4;
        const int cnt = strip ? 11 : 7;
        float best = 1e30f;
        int bq = -1, bx = 0, by = 0;
#pragma unroll
        for (int k = 0; k < 11; ++k) {
            if (k >= cnt) break;
            int dx, dy;
            if (strip) rot_dir(dir, 0, -(3 + 2 * k), dx, dy);
            else rot_dir(dir, V_OFF[k][0], V_OFF[k][1], dx, dy);
            const int qx = x + dx, qy = y + dy;
            const bool inb = qx >= 0 && qy >= 0 && qx < w && qy < h;
            const int qi = inb ? qy * w + qx : pix;
            const float cq = co[qi];
            if (inb && cq < best) {
                best = cq;
                bq = qi;
                bx = qx;
                by = qy;
            }
        }
        float4 hr = hyp0;
        if (bq >= 0) {
            float4 q = pl[bq];
            f3 n = xyz(q);
            f3 rq = pixel_ray(R, bx, by);
            float den = dot3(n, ray);
            if (den < -1e-6f && q.w > 0.f) {
                float d = q.w * dot3(n, rq) / den;
                if (d > 0.f && isfinite(d)) hr = mk4(n, d);
            }
        }
        hyp[(1 + r) * NT] = hr;
    }

    // 2. view selection and aggregation (patchmatch.cu:513-594)
    RefWinT<WR, WSTEP> rw;
    ref_stats_any<WR, WSTEP>(P, ref, x, y, wr, rw);
    const int vprev = P.bview[base + pix];
    // Aggregated costs: over the adopted sources (weight w2 > 0), or, while none is adopted, the
    // prior-weighted costs over all sources that the fallback takes. One array holds both in turn:
    // the first adopted source restarts it, and the fallback is then never used.
    float agg[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) agg[i] = 0.f;
    float den = 0.f, wbest = 0.f, denf = 0.f;
    int vbest = 255;
#pragma nounroll
    for (int j = 0; j < nsrc; ++j) {
        const PairRec& pr = prs[j];
        const LevelDesc S = P.lv[pr.src * P.nlevels + P.level];
        const LevelPair& lp = lps[j];
        float prior;
        {
            float H[9];
            bool ok = homography(R, lp, ifx, ify, (float)x, (float)y, hyp0.w, xyz(hyp0), H);
            prior = view_prior(P, R, pr, H, ok, x, y, hyp0, (float)wr);
        }
        wv[j * P.wv_stride] = 0.f;
        if (!(prior > 0.f)) continue;
        float m[9];  // photometric cost, then the term the aggregation takes: with lambda times the geometric error
        int good = 0, bad = 0;
        float conf = 0.f;
        auto vote = [&](float mi) {
            if (mi < P.tau_good) {
                good++;
                conf += c3d_expf(-mi * mi * P.inv2beta2);
            }
            if (mi > P.tau_bad) bad++;
        };
#pragma unroll
        for (int q = 0; q < 9; ++q) m[q] = 0.f;
        if constexpr (TPP == 1) {
#pragma nounroll
            for (int i = 0; i < 9; ++i) {
                float gi;
                const float mi = pair_cost_h<WR, WSTEP, GEO, PIPE, AHEAD, FEW>(P, rw, ref, R, S, pr, lp, ifx, ify, x, y, hyp[i * NT], gi);
                if (i > 0) vote(mi);
                const float ti = mi + P.lambda * gi;
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if (q == i) m[q] = ti;
            }
        } else {
            float gg[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) gg[q] = 0.f;
#pragma nounroll
            for (int i = sub; i < 9; i += TPP) {
                float gi;
                const float mi = pair_cost_h<WR, WSTEP, GEO, PIPE, AHEAD, FEW>(P, rw, ref, R, S, pr, lp, ifx, ify, x, y, hyp[i * NT], gi);
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if (q == i) {
                        m[q] = mi;
                        gg[q] = gi;
                    }
            }
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                m[q] = __shfl(m[q], lane - sub + (q & (TPP - 1)));
                if constexpr (GEO) gg[q] = __shfl(gg[q], lane - sub + (q & (TPP - 1)));
                if (q > 0) vote(m[q]);
                m[q] = m[q] + P.lambda * gg[q];
            }
        }
        bool adopt = good > P.n1 && bad < P.n2;
        bool isprev = j == vprev;
        float wp = adopt ? (isprev ? 2.f : 1.f) * conf / (float)good : (isprev ? P.prev_w : 0.f);
        float w2 = wp * prior;
        wv[j * P.wv_stride] = w2 > 0.f ? w2 : -prior;
        const bool adopted = w2 > 0.f;
        if (adopted && !(den > 0.f)) {
#pragma unroll
            for (int i = 0; i < 9; ++i) agg[i] = 0.f;
        }
        if (adopted || !(den > 0.f)) {
            const float wa = adopted ? w2 : prior;
#pragma unroll
            for (int i = 0; i < 9; ++i) agg[i] += wa * m[i];
        }
        denf += prior;
        if (adopted) {
            den += w2;
            if (w2 > wbest) {
                wbest = w2;
                vbest = j;
            }
        }
    }
    int bi9 = 0;
    const bool fallback = !(den > 0.f) && denf > 0.f;
    if (fallback) {
        for (int j = 0; j < nsrc; ++j) wv[j * P.wv_stride] = -wv[j * P.wv_stride];
        den = denf;
    }
    if (den > 0.f) {
#pragma unroll
        for (int i = 0; i < 9; ++i) agg[i] = agg[i] / den;
    } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) agg[i] = 2.f;
    }
    float bcost = agg[0];
#pragma unroll
    for (int i = 1; i < 9; ++i)
        if (agg[i] < bcost) {
            bi9 = i;
            bcost = agg[i];
        }
    float4 best = hyp[bi9 * NT];

    // 3. refinement: 6 hypotheses, plus the coarse prior at weak texture (patchmatch.cu:596-653)
    unsigned long long st = rng_state(P.seed, vd.key, P.level, P.run_id, P.t, P.color, (unsigned long long)pix);
    float d_r = random_depth(st, vd.dmin, vd.dmax);
    f3 n_r = random_normal(st, ray);
    float u = 2.f * rnd(st) - 1.f;
    float inv = best.w > 0.f ? (1.f / best.w) * (1.f + u * P.eps) : -1.f;
    float d_p = inv > 0.f ? 1.f / inv : d_r;
    if (!(best.w > 0.f)) best.w = d_r;
    f3 n0 = xyz(best);
    f3 n_p = perturb_normal(st, n0, ray, P.phi);
    float4* cand = hyp;  // the hypothesis table is free again
    cand[0] = mk4(n0, d_r);
    cand[NT] = mk4(n_r, best.w);
    cand[2 * NT] = mk4(n_r, d_r);
    cand[3 * NT] = mk4(n0, d_p);
    cand[4 * NT] = mk4(n_p, best.w);
    cand[5 * NT] = mk4(n_p, d_p);
    int ncand = 6;
    if (P.use_prior && rw.var < P.weak_var255) {
        float4 q = P.prior[base + pix];
        if (q.w > 0.f && dot3(xyz(q), ray) < 0.f) {
            cand[6 * NT] = q;
            ncand = 7;
        }
    }
    // A candidate's cost is a sum of non-negative terms (weights > 0, costs in [0, 2], geometric
    // errors in [0, gmax], lambda >= 0) divided by den: its partial sums only grow, so once
    // nm / den reaches bcost the candidate cannot be accepted and its remaining sources are
    // skipped. The accepted planes and costs are unchanged.
    // With several lanes per pixel each lane costs its candidates against the step-2 best (a
    // candidate that reaches it cannot be accepted later either, the best only decreasing), then
    // all of them accept in candidate order from the exchanged costs: a skipped candidate's is its
    // partial sum, at or above the step-2 best (which has no upper bound: it grows with lambda gmax).
    const bool early = P.lambda >= 0.f && (!GEO || P.gmax >= 0.f);
    float ccs[7];
#pragma unroll
    for (int q = 0; q < 7; ++q) ccs[q] = 0.f;  // each is set by the lane that costs it
#pragma nounroll
    for (int c = sub; c < ncand; c += TPP) {
        const float4 hc = cand[c * NT];
        float cc = 2.f;
        if (den > 0.f) {
            float nm = 0.f;
#pragma nounroll
            for (int j = 0; j < nsrc; ++j) {
                float wj = wv[j * P.wv_stride];
                if (!(wj > 0.f)) continue;
                const PairRec& pr = prs[j];
                const LevelDesc S = P.lv[pr.src * P.nlevels + P.level];
                float g;
                float m = pair_cost_h<WR, WSTEP, GEO, PIPE, AHEAD, FEW>(P, rw, ref, R, S, pr, lps[j], ifx, ify, x, y, hc, g);
                nm += wj * (m + P.lambda * g);
                if (early && nm / den >= bcost) break;
            }
            cc = nm / den;
        }
        if constexpr (TPP == 1) {
            if (cc < bcost) {
                bcost = cc;
                best = hc;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 7; ++q)
                if (q == c) ccs[q] = cc;
        }
    }
    if constexpr (TPP > 1) {
#pragma unroll
        for (int q = 0; q < 7; ++q) ccs[q] = __shfl(ccs[q], lane - sub + (q & (TPP - 1)));
#pragma unroll
        for (int q = 0; q < 7; ++q)
            if (q < ncand && ccs[q] < bcost) {
                bcost = ccs[q];
                best = cand[q * NT];
            }
    }
    if (sub == 0) {
        pl[pix] = best;
        P.cost[base + pix] = bcost;
        P.bview[base + pix] = (uint8_t)vbest;
    }
}

// Stages the reference rows of a 64 x 4 pixel tile (plus the window margin) in LDS.
__device__ __forceinline__ void stage_pix_tile(float* tile, const uint8_t* g, int w, int h, int px0, int py0, int wr) {
    const int TW = PIX_TW + 2 * wr, TH = PIX_TH + 2 * wr;
    const int tx0 = px0 - wr, ty0 = py0 - wr;
    for (int i = threadIdx.x; i < TW * TH; i += 256) {
        int ty = i / TW, tx = i - ty * TW;
        int gx = tx0 + tx, gy = ty0 + ty;
        tile[i] = (gx >= 0 && gy >= 0 && gx < w && gy < h) ? (float)g[(size_t)gy * w + gx] : 0.0f;
    }
}

// ================================================================ run start / evaluation (patchmatch.cu:659-692)
//
// A run starts with pm_eval: random initialisation (mode 1, by random_init), the top-K cost of
// every pixel's plane and the best view reset. When the run then has at least one iteration, the
// costs of the pixels of colour 0 are dead: the first half step (colour 0) recomputes and rewrites
// every colour-0 pixel without reading its stored cost (its candidate step reads only the 72
// neighbours of the opposite colour), and nothing else reads them in between. So such a run starts
// with k_eval_init over every pixel (the initialisation and best-view reset, no window) and
// k_eval<ONE = true> for the pixels of colour 1 only, with the half step's one-colour lane
// mapping, which does half the window work. Runs of no iterations and c3d_pm_evaluate keep the
// whole evaluation (ONE = false).
// top-K mean of the plane's per-source costs (patchmatch.cu:326-345), 2 for a non-positive depth
template <int WR, int WSTEP, class REF>
__device__ __forceinline__ float eval_cost(const KParams& P, const ViewDesc& vd, const LevelDesc& R, const PairRec* prs,
                                           const LevelPair* lps, const REF& ref, int wr, int x, int y, float4 h) {
    if (!(h.w > 0.f)) return 2.f;
    RefWinT<WR, WSTEP> rw;
    ref_stats_any<WR, WSTEP>(P, ref, x, y, wr, rw);
    float b0 = 1e30f, b1 = 1e30f, b2 = 1e30f;
#pragma nounroll
    for (int j = 0; j < vd.nsrc; ++j) {
        const PairRec& pr = prs[j];
        const LevelDesc S = P.lv[pr.src * P.nlevels + P.level];
        float gq = 0.f;
        float cc = pair_cost<WR, WSTEP, EVAL_PIPE>(P, rw, ref, R, S, pr, lps[j], x, y, h, &gq);
        if (P.geometric) cc = cc + P.lambda * gq;
        if (cc < b0) {
            b2 = b1;
            b1 = b0;
            b0 = cc;
        } else if (cc < b1) {
            b2 = b1;
            b1 = cc;
        } else if (cc < b2) {
            b2 = cc;
        }
    }
    int k = P.topk < vd.nsrc ? P.topk : vd.nsrc;
    float s = b0;
    if (k >= 2) s += b1;
    if (k >= 3) s += b2;
    return k > 0 ? s / (float)k : 2.0f;
}

// ONE = false: every pixel of 64 x 4 tiles, initialisation (mode 1) and cost. ONE = true: the
// pixels of colour P.color of 128 x 4 spans (one lane per pixel, as the half step), cost only
// (k_eval_init has initialised them).
template <int WR, int WSTEP, bool ONE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(eval_waves<WR, WSTEP>()))) void k_eval(KParams P, int mode) {
    constexpr int SPAN = ONE ? HALF_SPAN : PIX_TW;
    constexpr int TW = SPAN + 2 * WR;
    __shared__ float tile_s[WR > 0 ? TW * (PIX_TH + 2 * WR) : 1];
    extern __shared__ float dyn_lds[];
    const int wr = WR > 0 ? WR : P.wr;
    float* tile = WR > 0 ? tile_s : dyn_lds;
    BatchItem it;
    int px0, py0;
    if (!find_tile(P, xcd_tile(blockIdx.x, P.ntiles), SPAN, PIX_TH, it, px0, py0)) return;
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    {
        const uint8_t* g = P.gray + R.goff;
        const int twd = SPAN + 2 * wr, thd = PIX_TH + 2 * wr;
        const int tx0 = px0 - wr, ty0 = py0 - wr;
        for (int i = threadIdx.x; i < twd * thd; i += 256) {
            int ty = i / twd, tx = i - ty * twd;
            int gx = tx0 + tx, gy = ty0 + ty;
            tile[i] = (gx >= 0 && gy >= 0 && gx < it.w && gy < it.h) ? (float)g[(size_t)gy * it.w + gx] : 0.0f;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, y = py0 + (threadIdx.x >> 6);
    const int x = ONE ? px0 + 2 * lane + ((y + P.color) & 1) : px0 + lane;
    if (x >= it.w || y >= it.h) return;
    const ViewDesc vd = P.views[it.view];
    const PairRec* prs = P.pairs + (size_t)it.view * MAXSRC;
    const LevelPair* lps = P.lpairs + ((size_t)it.view * P.nlevels + P.level) * MAXSRC;
    const int pix = y * it.w + x;
    const long long base = it.off;
    const float4 h = ONE ? P.plane[base + pix] : eval_init_plane(P, vd, R, x, y, pix, base, mode);
    const auto ref = tile_ref<WR, TW>(tile, px0 - wr, py0 - wr, SPAN + 2 * wr);
    P.cost[base + pix] = eval_cost<WR, WSTEP>(P, vd, R, prs, lps, ref, wr, x, y, h);
    if (!ONE && mode == 1) P.bview[base + pix] = 255;
}

// ================================================================ final read-out (patchmatch.cu:694-737)
template <int WR, int WSTEP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(eval_waves<WR, WSTEP>()))) void k_filter(KParams P) {
    constexpr int TW = PIX_TW + 2 * WR;
    __shared__ float tile_s[WR > 0 ? TW * (PIX_TH + 2 * WR) : 1];
    extern __shared__ float dyn_lds[];
    const int wr = WR > 0 ? WR : P.wr;
    float* tile = WR > 0 ? tile_s : dyn_lds;
    BatchItem it;
    int px0, py0;
    if (!find_tile(P, xcd_tile(blockIdx.x, P.ntiles), PIX_TW, PIX_TH, it, px0, py0)) return;
    const LevelDesc R = P.lv[it.view * P.nlevels + P.level];
    stage_pix_tile(tile, P.gray + R.goff, it.w, it.h, px0, py0, wr);
    __syncthreads();
    const int x = px0 + (threadIdx.x & 63), y = py0 + (threadIdx.x >> 6);
    if (x >= it.w || y >= it.h) return;
    const ViewDesc vd = P.views[it.view];
    const PairRec* prs = P.pairs + (size_t)it.view * MAXSRC;
    const LevelPair* lps = P.lpairs + ((size_t)it.view * P.nlevels + P.level) * MAXSRC;
    const int pix = y * it.w + x;
    const long long base = it.off;
    float4 h = P.plane[base + pix];
    int count = 0;
    if (h.w > 0.f) {
        const auto ref = tile_ref<WR, TW>(tile, px0 - wr, py0 - wr, PIX_TW + 2 * wr);
        RefWinT<WR, WSTEP> rw;
        ref_stats_any<WR, WSTEP>(P, ref, x, y, wr, rw);
        f3 ray = pixel_ray(R, x, y);
        f3 X = mk3(ray.x * h.w, ray.y * h.w, h.w);
        float lx = sqrtf(dot3(X, X));
#pragma nounroll
        for (int j = 0; j < vd.nsrc; ++j) {
            const PairRec& pr = prs[j];
            const LevelDesc S = P.lv[pr.src * P.nlevels + P.level];
            f3 Sv = mk3(pr.c[0] - X.x, pr.c[1] - X.y, pr.c[2] - X.z);
            float ls = sqrtf(dot3(Sv, Sv));
            if (!(ls > 0.f)) continue;
            float cost = -dot3(Sv, X) / (ls * lx);
            if (cost > P.cos_filter_tri) continue;
            float cphi = dot3(Sv, xyz(h)) / ls;
            if (cphi <= 0.f) continue;
            float H[9];
            if (!homography(R, lps[j], R.ifx, R.ify, (float)x, (float)y, h.w, xyz(h), H)) continue;
            const GeoFetch gf = geo_fetch(P, R, S, pr, x, y, h.w);  // used after the window
            float m = ncc_cost_any<WR, WSTEP, EVAL_PIPE>(P, rw, ref, S, H, x, y);
            float e = P.ncc_norm * c3d_expf(-m * m * P.inv2ncc);
            if (e / (e + 0.5f) < P.q_min) continue;
            if (geo_finish(R, S, pr, x, y, gf) > P.filter_gmax) continue;
            count++;
        }
    }
    P.count[base + pix] = (uint8_t)(count < 255 ? count : 255);
}

// ================================================================ cost probe (no reference counterpart)
template <int WR, int WSTEP>
__global__ __launch_bounds__(256) void k_pair_costs(KParams P, int view, int slot, int n, const int* xy, const float4* planes,
                                                    float* out) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const LevelDesc R = P.lv[view * P.nlevels + P.level];
    const PairRec& pr = P.pairs[(size_t)view * MAXSRC + slot];
    const LevelPair& lp = P.lpairs[((size_t)view * P.nlevels + P.level) * MAXSRC + slot];
    const LevelDesc S = P.lv[pr.src * P.nlevels + P.level];
    int x = xy[2 * i], y = xy[2 * i + 1];
    RefGlobal g{P.gray + R.goff, R.w, R.h};
    const int wr = WR > 0 ? WR : P.wr;
    RefWinT<WR, WSTEP> rw;
    ref_stats_any<WR, WSTEP>(P, g, x, y, wr, rw);
    float4 h = planes[i];
    float H[9];
    float c = 2.f;
    if (homography(R, lp, R.ifx, R.ify, (float)x, (float)y, h.w, xyz(h), H)) c = ncc_cost_any<WR, WSTEP>(P, rw, g, S, H, x, y);
    out[i] = c;
}

// ================================================================ launchers

// dynamic LDS bytes of the any-radius (WR = 0) reference tiles
static size_t half_tile_bytes(int wr, int rows, int tpp) { return (size_t)half_pitch(tpp, wr) * (half_bh(tpp) * rows + 2 * wr) * sizeof(float); }
static size_t span_tile_bytes(int wr) { return (size_t)(HALF_SPAN + 2 * wr) * (PIX_TH + 2 * wr) * sizeof(float); }
static size_t pix_tile_bytes(int wr) { return (size_t)(PIX_TW + 2 * wr) * (PIX_TH + 2 * wr) * sizeof(float); }

template <int WR, int WSTEP, int ROWS, int TPP, bool FEW>
static void launch_half_rows(const KParams& P, size_t lds, hipStream_t s) {
    if (P.geometric) hipLaunchKernelGGL((k_half<WR, WSTEP, true, ROWS, TPP, FEW>), dim3(P.ntiles), dim3(ROWS * 64), lds, s, P);
    else hipLaunchKernelGGL((k_half<WR, WSTEP, false, ROWS, TPP, FEW>), dim3(P.ntiles), dim3(ROWS * 64), lds, s, P);
}

// P.ntiles must count the tiles of the shape (half_tiles(..., rows, tpp)); the compiled shapes are
// (rows, lanes per pixel) = (1, 1), (2, 1), (4, 1) and (4, 2), which a caller may ask for, and
// (1, 2), (1, 4) and (1, 8), which half_lanes picks for small batches
template <int WR, int WSTEP>
static hipError_t launch_half(const KParams& P0, int rows, int tpp, hipStream_t s) {
    if (!half_shape_ok(rows, tpp) && !(rows == 1 && (tpp == 2 || tpp == 4 || tpp == 8))) return hipErrorInvalidValue;
    KParams P = P0;
    P.wv_stride = rows * 64;
    size_t lds = (size_t)P.wv_stride * (P.max_nsrc > 0 ? P.max_nsrc : 1) * sizeof(float);
    if (WR == 0) lds += half_tile_bytes(P.wr, rows, tpp);
    constexpr bool HELD = WR > 0 && Win<(WR > 0 ? WR : 1), WSTEP>::HELD;  // else both builds are one
    const bool few = HELD && P.ntiles * rows <= few_waves(P.geometric);
    if (rows == 1 && tpp == 1 && few) launch_half_rows<WR, WSTEP, 1, 1, HELD>(P, lds, s);
    else if (rows == 1 && tpp == 1) launch_half_rows<WR, WSTEP, 1, 1, false>(P, lds, s);
    else if (rows == 1 && tpp == 2) launch_half_rows<WR, WSTEP, 1, 2, true>(P, lds, s);
    else if (rows == 1 && tpp == 4) launch_half_rows<WR, WSTEP, 1, 4, true>(P, lds, s);
    else if (rows == 1) launch_half_rows<WR, WSTEP, 1, 8, true>(P, lds, s);
    else if (rows == 2) launch_half_rows<WR, WSTEP, 2, 1, false>(P, lds, s);
    else if (tpp == 1) launch_half_rows<WR, WSTEP, 4, 1, false>(P, lds, s);
    else launch_half_rows<WR, WSTEP, 4, 2, true>(P, lds, s);
    return hipGetLastError();
}
template <int WR, int WSTEP>
static hipError_t launch_eval(const KParams& P, int mode, hipStream_t s) {
    hipLaunchKernelGGL((k_eval<WR, WSTEP, false>), dim3(P.ntiles), dim3(256), WR == 0 ? pix_tile_bytes(P.wr) : 0, s, P, mode);
    return hipGetLastError();
}
// P.ntiles must count 128 x 4 spans (span_tiles); P.color selects the pixels
template <int WR, int WSTEP>
static hipError_t launch_eval_color(const KParams& P, hipStream_t s) {
    hipLaunchKernelGGL((k_eval<WR, WSTEP, true>), dim3(P.ntiles), dim3(256), WR == 0 ? span_tile_bytes(P.wr) : 0, s, P, 0);
    return hipGetLastError();
}
template <int WR, int WSTEP>
static hipError_t launch_filter(const KParams& P, hipStream_t s) {
    hipLaunchKernelGGL((k_filter<WR, WSTEP>), dim3(P.ntiles), dim3(256), WR == 0 ? pix_tile_bytes(P.wr) : 0, s, P);
    return hipGetLastError();
}
template <int WR, int WSTEP>
static hipError_t launch_pair_costs(const KParams& P, int view, int slot, int n, const int* xy, const float4* planes, float* out,
                                    hipStream_t s) {
    hipLaunchKernelGGL((k_pair_costs<WR, WSTEP>), dim3((n + 255) / 256), dim3(256), 0, s, P, view, slot, n, xy, planes, out);
    return hipGetLastError();
}
template <int WR, int WSTEP>
static const void* half_symbol() {
    return reinterpret_cast<const void*>(&k_half<WR, WSTEP, false, 4, 1, false>);
}

template <int WR, int WSTEP>
static constexpr KernelSet make_set() {
    return KernelSet{WR, WSTEP, &launch_half<WR, WSTEP>, &launch_eval<WR, WSTEP>, &launch_eval_color<WR, WSTEP>,
                     &launch_filter<WR, WSTEP>, &launch_pair_costs<WR, WSTEP>, &half_symbol<WR, WSTEP>};
}

// Window variants compiled into the library (radius, step): the fast profile (5, 2) and the
// variants of the reference's window report (patchmatch_gpu.rs:164) whose window holds at most
// 49 samples, with the bilateral weights in registers; the quality profile's (5, 1), which forms them
// row by row (window_rows); every other radius up to 20 runs the any-radius kernels (wr = 0 below)
// of its step.
static const KernelSet kSets[] = {make_set<5, 2>(), make_set<4, 2>(), make_set<3, 2>(), make_set<2, 2>(), make_set<3, 1>(),
                                  make_set<2, 1>(), make_set<1, 1>(), make_set<5, 1>()};
static const KernelSet kAny[] = {make_set<0, 1>(), make_set<0, 2>()};

const KernelSet* kernel_set(int wr, int wstep, bool any_radius) {
    if (wr < 1 || wr > MAX_WR || wstep < 1 || wstep > 2) return nullptr;
    if (!any_radius)
        for (const KernelSet& k : kSets)
            if (k.wr == wr && k.wstep == wstep) return &k;
    return &kAny[wstep - 1];
}

}  // namespace C3D_QUAD_NS
}  // namespace c3d
