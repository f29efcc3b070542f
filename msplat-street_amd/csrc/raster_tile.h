// Per-tile front-to-back alpha compositing (forward) and its backward, as device
// functions shared by the one-view kernels (one workgroup per tile) and the persistent
// batched kernels (workgroups pull (view, tile) items from a queue).
//
// Both are bound by VALU issue (the forward fills it, the backward uses 79% of it: its one
// wave per tile leaves the rest to the slowest tiles), so what counts is instructions per
// pixel and record and the records that are visited at all: 18 instructions in the forward (28 before), 32 in the
// backward (45). On the 475k street scene at 1264x832 the forward kernel went 211 -> 155 us
// and the backward 449 -> 362 us, at 3M gaussians and 3840x2160 the forward 381 -> 250 us;
// the exact ellipse test in place of the bounding box gives about 15% and 8% of it.
//
// Forward: two waves per 16x16 tile, two pixels per lane. Gaussian records of the tile's
// list are staged through LDS in batches (the LDS batch depth is a kernel variant).
//
// Backward without global atomics: per gaussian of a batch, the wave's contributions
// are summed (DPP within rows of 16 lanes, permlane swaps across rows) only when some
// lane contributed (ballot), written to a per-wave LDS partial, and the partials are
// summed in wave order into the intersection's gradient slot. Slots are laid out in the pre-sort order of the intersections
// (record-major, tiles row-major), so the per-gaussian reduction reads each record's
// slots contiguously and in the reference's tile order.
#pragma once

#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace msplat {

// The pixels of one view: `image`, `final_T`, `final_idx` and `v_image` point at the
// view's first pixel.
struct TileView {
    uint32_t width, height;
    int tiles_x;
    float bg[3];
    float *image, *final_T;
    int32_t *final_idx;
    const float *v_image;
    // prior-guided (aux) frames: the per-pixel background, the expected-depth sum, and
    // the prior losses' gradients dL/dD, dL/dA (2 per pixel)
    const float *bg_img = nullptr;
    float *out_depth = nullptr;
    const float *v_aux = nullptr;
};

// Buffers shared by every view: ranges over global tile ids, the sorted record ids,
// per-record splats and tile rectangles (in the record's view), and gradient slots.
struct TileData {
    const int32_t *tile_start, *gid;
    const float4 *splat_a, *splat_b;
    const float *splat_blue;
    const uint2 *rect;
    const uint32_t *offsets;
    float4 *slot_a, *slot_b;
    float *slot_c;
    uint8_t *slot_f;  // 1: the slot's nine values were written; 0 (set before the launch): all zero
    unsigned long long *slots_written;  // null, or a running count of written slots
    bool cull;  // skip gaussians that splat_misses_tile proves invisible in the tile
    // aux frames: per record view depth, and the intersections' depth gradient slots
    const float *depths = nullptr;
    float *slot_d = nullptr;
};

// True when the splat composites no pixel of the tile whose top-left pixel is (x0, y0):
// the ellipse {0.5 d^T Q d <= L'} misses the tile's pixel centres' rectangle, with Q the
// conic and L' above the largest sigma that passes both sigma < SIGMA_MAX and
// opacity exp(-sigma) >= ALPHA_MIN. The form is convex with its minimum 0 at the splat's
// centre, so over the rectangle it is smallest at the centre when that lies inside, else on
// an edge that faces it: on the edge x = xe at dy = -b xe / c (clamped to the edge), on the
// edge y = ye at dx = -b ye / a. The pixel loops compute log2(e) sigma from the
// scaled conic to a relative error below 24 u kappa (u = 2^-24, kappa the conic's condition
// number) and alpha to a few ulp, and the minimum here is off by less than 16 u kappa of
// itself (its terms' absolute sum is at most 2 kappa times the form; an inexact minimiser
// only costs its error squared), so the test is made only for kappa < 1024 (40 u kappa <
// 2.5e-3) and L' is the exact level raised by 2^-8 relative plus 2^-8 absolute. Any pair it
// rejects would fail the validity test in every pixel, and an invalid pair changes nothing
// (it adds exact zeros), so skipping it leaves every output bit unchanged. The ellipse's
// bounding box, tested before, kept about a fifth more of the street scene's records.
__device__ inline bool splat_misses_tile(const float4 &A, const float4 &B, float x0, float y0) {
    const float a = A.z, b = A.w, c = B.x;
    const float det = a * c - b * b, tr = a + c;
    if (!(det > 0.f) || !(tr * tr < 1024.f * det)) return false;  // (a+c)^2/det = kappa + 2 + 1/kappa
    const float L = fminf(SIGMA_MAX, __logf(B.y * (1.f / ALPHA_MIN)));
    if (!(L > 1.f / 64.f)) return false;
    const float xa = x0 - A.x, xb = xa + (float)(TILE - 1), ya = y0 - A.y, yb = ya + (float)(TILE - 1);
    const float xe = fminf(fmaxf(0.f, xa), xb), ye = fminf(fmaxf(0.f, ya), yb);  // nearest to the centre
    const float yv = fminf(fmaxf(-b * xe * __builtin_amdgcn_rcpf(c), ya), yb);
    const float xh = fminf(fmaxf(-b * ye * __builtin_amdgcn_rcpf(a), xa), xb);
    const float v = (a * xe + 2.f * b * yv) * xe + c * yv * yv;  // on the edge x = xe
    const float h = (c * ye + 2.f * b * xh) * ye + a * xh * xh;  // on the edge y = ye
    const float m = xe != 0.f ? (ye != 0.f ? fminf(v, h) : v) : (ye != 0.f ? h : 0.f);
    return 0.5f * m > L * (1.f + 1.f / 256.f) + 1.f / 256.f;
}

// The pixel loops work with e = log2(e) sigma, the negated exponent of alpha's power of two
// (alpha = opacity 2^-e, one v_exp_f32), from a conic scaled when it is staged in LDS:
// a' = log2(e)/2 a, b' = log2(e) b, c' = log2(e)/2 c, so that
// e = (a' dx) dx + (c' dy + b' dx) dy: adx2 = (a' dx) dx and bdx = b' dx are per record,
// which the backward hoists out of its pixel rows, and a pixel adds two multiply-adds. One
// fixed evaluation order is shared by the forward and backward loops, so that both make
// the same validity decisions. A pair is valid when 0 <= sigma < SIGMA_MAX and
// alpha >= ALPHA_MIN; both upper bounds on e are one number per record,
// min(log2(e) SIGMA_MAX, log2(opacity / ALPHA_MIN)), staged as the bit pattern `limit`
// below which e's bits must lie. Non-negative floats order as their bits, and a negative e
// or a NaN has larger bits than any limit, so one unsigned compare makes the three tests.
constexpr float POW_HALF = 0.72134752044448170f;  // log2(e) / 2
constexpr float POW_ONE = 1.44269504088896341f;   // log2(e)
__device__ constexpr float E_MAX = SIGMA_MAX * POW_ONE;

// A staged record, three 16-byte LDS reads: (x, y, a', b'), (c', opacity, limit, list
// position), (r, g, b, view depth), colours stored as composited, max(raw + 0.5, 0).
// Pixels per record cost three wide reads instead of five narrower ones.
__device__ inline uint32_t splat_limit(float opacity) {
    opacity = fminf(opacity, 2.f);  // a NaN is 2: alpha is min(ALPHA_MAX, NaN) = ALPHA_MAX up to E_MAX
    if (!(opacity >= ALPHA_MIN)) return 0u;  // nothing is below: never valid
    // the logarithm's own rounding, half a unit of e, decided 18% more pairs wrongly (against
    // 64 bits) than opacity 2^-e >= ALPHA_MIN does: the last bits are taken by that test
    const uint32_t l = max(__float_as_uint(fmaxf(__builtin_amdgcn_logf(opacity * (1.f / ALPHA_MIN)), 0.f)), 2u) - 2u;
    uint32_t above = 1;
#pragma unroll
    for (uint32_t u = 1; u <= 4; u++) above += opacity * __builtin_amdgcn_exp2f(-__uint_as_float(l + u)) >= ALPHA_MIN;
    return min(l + above, __float_as_uint(E_MAX));  // below the first e that fails; e < E_MAX
}
__device__ inline void stage_splat(float4 *la, float4 *lb, float4 *lc, int pos, const float4 &A, const float4 &B,
                                   float blue, float z, int k) {
    la[pos] = make_float4(A.x, A.y, A.z * POW_HALF, A.w * POW_ONE);
    lb[pos] = make_float4(B.x * POW_HALF, B.y, __uint_as_float(splat_limit(B.y)), __int_as_float(k));
    lc[pos] = make_float4(fmaxf(B.z + 0.5f, 0.f), fmaxf(B.w + 0.5f, 0.f), fmaxf(blue + 0.5f, 0.f), z);
}
__device__ inline float splat_exponent(float adx2, float bdx, float c, float dy) {
    return __builtin_fmaf(__builtin_fmaf(c, dy, bdx), dy, adx2);
}
__device__ inline float splat_alpha(float opacity, float e) {
    return fminf(ALPHA_MAX, opacity * __builtin_amdgcn_exp2f(-e));
}
__device__ inline bool splat_valid(float e, float limit) { return __float_as_uint(e) < __float_as_uint(limit); }

// Position of the calling thread's item among the workgroup's kept items (in thread
// order) and, in `total`, their number. Every thread of the NW-wave workgroup calls it;
// `wcount` must not be written again before every wave has returned (callers alternate
// two buffers or pass a barrier in between).
template <int NW>
__device__ inline int kept_position(bool keep, int *wcount, int &total) {
    const uint64_t bal = __ballot(keep);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) wcount[w] = __popcll(bal);
    __syncthreads();
    int off = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) {
        const int cnt = wcount[i];
        off += i < w ? cnt : 0;
        total += cnt;
    }
    return off + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
}

// The forward workgroup: FPT pixels per lane, FNT / 64 waves per tile. Wave w owns rows
// [4 FPT w, 4 FPT (w + 1)) and lane l the pixels (l % 16, 4 FPT w + l / 16 + 4 k), k < FPT.
// Every lane of a wave reads every staged record (48 bytes, 24 cycles of the CU's LDS port a
// wave), which with one pixel per lane and four waves per tile takes longer than the
// arithmetic (227 us on the street scene); with two pixels per lane a tile reads each
// record twice, and dx and its products are shared by a lane's pixels (179 us). Four pixels
// per lane hold too many registers (230 us).
constexpr int FPT = 2, FNT = 256 / FPT;

// A lane's front-to-back composite
struct Composite {
    float T[FPT], r[FPT], g[FPT], b[FPT], depth[FPT];
    int last[FPT];    // list position of the last contributor
    int last_j[FPT];  // the same in the batch being composited (its LDS index), -1: none in it
    bool done[FPT];   // terminated, or outside the image
    __device__ inline bool all_done() const {
        bool d = true;
#pragma unroll
        for (int k = 0; k < FPT; k++) d = d && done[k];
        return d;
    }
};

// Composites the staged records [0, n8) (n8 a multiple of 8) into the lane's pixels (fx,
// fy[k]). Groups of G: the alphas first (independent of each other), then the
// transmittance through the group as if no pixel terminated in it, T - alpha T in one
// rounding. (By the rounded factor 1 - alpha, which the backward divides by again, it takes
// one instruction more, 1% of a train step, and is no closer to 64 bits: over six scenes
// each of four cases the median record's gradient error moves by -1 to +2%, images' by +1%.)
// Transmittance only falls, so when it ends above T_MIN in every pixel of the wave none
// did, and the colours follow without a test per record. Otherwise (a pixel terminates
// once) the group is composited step by step: skip (invalid), accept, or terminate
// (transmittance would drop to T_MIN: last = k - 1, as the CPU). A chunk's pixels that
// terminated in an earlier one (CHUNK) start at or below T_MIN with every alpha zero, and
// don't count.
template <bool AUX, bool CHUNK = false>
__device__ inline void composite_batch(const float4 *la, const float4 *lb, const float4 *lc, int n8, float fx,
                                       const float (&fy)[FPT], Composite &p) {
#pragma clang fp contract(fast)
    constexpr int G = 4;
    for (int j0 = 0; j0 < n8; j0 += G) {
        float alpha[G][FPT], T[FPT];
        bool ok[G][FPT], low = false;
#pragma unroll
        for (int k = 0; k < FPT; k++) T[k] = p.T[k];
#pragma unroll
        for (int u = 0; u < G; u++) {
            const float4 A = la[j0 + u], B = lb[j0 + u];
            const float dx = A.x - fx, adx2 = (A.z * dx) * dx, bdx = A.w * dx;
#pragma unroll
            for (int k = 0; k < FPT; k++) {
                const float e = splat_exponent(adx2, bdx, B.x, A.y - fy[k]);
                ok[u][k] = !p.done[k] && splat_valid(e, B.z);
                alpha[u][k] = ok[u][k] ? splat_alpha(B.y, e) : 0.f;
                T[k] -= alpha[u][k] * T[k];
            }
        }
#pragma unroll
        for (int k = 0; k < FPT; k++) low = low || (T[k] <= T_MIN && !(CHUNK && p.done[k]));
        if (__ballot(low) == 0) {
#pragma unroll
            for (int u = 0; u < G; u++) {
                const float4 C = lc[j0 + u];
#pragma unroll
                for (int k = 0; k < FPT; k++) {
                    const float vis = alpha[u][k] * p.T[k];
                    p.r[k] += C.x * vis;
                    p.g[k] += C.y * vis;
                    p.b[k] += C.z * vis;
                    if (AUX) p.depth[k] += C.w * vis;
                    p.T[k] -= alpha[u][k] * p.T[k];
                    p.last_j[k] = ok[u][k] ? j0 + u : p.last_j[k];
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < G; u++) {
                const float4 C = lc[j0 + u];
#pragma unroll
                for (int k = 0; k < FPT; k++) {
                    const bool valid = ok[u][k] && !p.done[k];
                    const float nT = p.T[k] - alpha[u][k] * p.T[k];
                    const bool term = valid && nT <= T_MIN, accept = valid && !term;
                    const float vis = accept ? alpha[u][k] * p.T[k] : 0.f;
                    p.r[k] += C.x * vis;
                    p.g[k] += C.y * vis;
                    p.b[k] += C.z * vis;
                    if (AUX) p.depth[k] += C.w * vis;
                    p.T[k] = accept ? nT : p.T[k];
                    if (term) p.last[k] = __float_as_int(lb[j0 + u].w) - 1;
                    p.last_j[k] = term ? -1 : accept ? j0 + u : p.last_j[k];
                    p.done[k] = p.done[k] || term;
                }
            }
            if (__ballot(!p.all_done()) == 0) break;
        }
    }
#pragma unroll
    for (int k = 0; k < FPT; k++) {
        if (p.last_j[k] >= 0) p.last[k] = __float_as_int(lb[p.last_j[k]].w);
        p.last_j[k] = -1;
    }
}

// Stages records [base, base + FB) of [.., e) that can reach the tile into LDS, in list
// order, padded to a multiple of 8 with records that are valid nowhere (limit 0); returns
// the padded count.
template <int FB, bool AUX = false>
__device__ inline int stage_forward_batch(const TileData &d, int base, int e, float x0, float y0, float4 *la,
                                          float4 *lb, float4 *lc, int (*wcount)[FNT / 64]) {
    int n = 0;
#pragma unroll
    for (int c = 0; c < FB; c += FNT) {
        const int i = c + threadIdx.x, k = base + i;
        bool keep = false;
        float4 A0, B0;
        float C0 = 0.f, Z0 = 0.f;
        if (i < FB && k < e) {
            const int g = d.gid[k];
            A0 = d.splat_a[g];
            B0 = d.splat_b[g];
            C0 = d.splat_blue[g];
            if (AUX) Z0 = d.depths[g];
            keep = !(d.cull && splat_misses_tile(A0, B0, x0, y0));
        }
        int total;
        const int pos = n + kept_position<FNT / 64>(keep, wcount[(c / FNT) & 1], total);
        if (keep) stage_splat(la, lb, lc, pos, A0, B0, C0, Z0, k);
        n += total;
    }
    const int n8 = (n + 7) & ~7;
    if ((int)threadIdx.x < n8 - n)
        la[n + threadIdx.x] = lb[n + threadIdx.x] = lc[n + threadIdx.x] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    return n8;
}

// nd_rasterize_forward (core/cpu/msplat_cpu.cpp:574-626) for global tile `gt`, which is
// tile `lt` of view `v`. Every thread of the FNT-thread workgroup calls it; FB gaussian
// records are staged in LDS per batch.
// With AUX (rasterize_forward_aux, cpu:574-626 with f.aux): also the expected-depth sum
// sum_i z_i alpha_i T_i into out_depth, over the per-pixel background bg_img.
template <int FB, bool AUX = false>
__device__ inline void forward_tile(const TileView &v, const TileData &d, int gt, int lt) {
#pragma clang fp contract(fast)
    __shared__ float4 la[FB], lb[FB], lc[FB];
    __shared__ int wcount[2][FNT / 64];
    const int tx = lt % v.tiles_x, ty = lt / v.tiles_x;
    const float x0 = (float)(tx * TILE), y0 = (float)(ty * TILE);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int px = tx * TILE + (lane & 15), py = ty * TILE + 4 * FPT * w + (lane >> 4);
    const int s = d.tile_start[gt], e = d.tile_start[gt + 1];
    Composite p;
    float fy[FPT];
#pragma unroll
    for (int k = 0; k < FPT; k++) {
        fy[k] = (float)(py + 4 * k);
        p.T[k] = 1.f;
        p.r[k] = p.g[k] = p.b[k] = p.depth[k] = 0.f;
        p.last[k] = s - 1;
        p.last_j[k] = -1;
        p.done[k] = !(px < (int)v.width && py + 4 * k < (int)v.height);
    }
    for (int base = s; base < e; base += FB) {
        if (__syncthreads_count(p.all_done()) == FNT) break;
        const int n8 = stage_forward_batch<FB, AUX>(d, base, e, x0, y0, la, lb, lc, wcount);
        if (__ballot(!p.all_done()) != 0) composite_batch<AUX>(la, lb, lc, n8, (float)px, fy, p);
    }
#pragma unroll
    for (int k = 0; k < FPT; k++) {
        if (!(px < (int)v.width && py + 4 * k < (int)v.height)) continue;
        const size_t pid = (size_t)(py + 4 * k) * v.width + px;
        const float T = p.T[k];
        v.final_T[pid] = T;
        v.final_idx[pid] = p.last[k];
        float bg0 = v.bg[0], bg1 = v.bg[1], bg2 = v.bg[2];
        if (AUX) {
            bg0 = v.bg_img[3 * pid];
            bg1 = v.bg_img[3 * pid + 1];
            bg2 = v.bg_img[3 * pid + 2];
            v.out_depth[pid] = p.depth[k];
        }
        v.image[3 * pid] = fminf(fmaxf(bg0 * T + p.r[k], 0.f), 1.f);
        v.image[3 * pid + 1] = fminf(fmaxf(bg1 * T + p.g[k], 0.f), 1.f);
        v.image[3 * pid + 2] = fminf(fmaxf(bg2 * T + p.b[k], 0.f), 1.f);
    }
}

// ── Depth-chunked compositing for views with few tiles ─────────────────────────
// A view with few tiles runs few workgroups, each over a long list. The chunked form
// splits every tile's list into K consecutive parts of equal length (chunk c of a list
// [s, e) is [s + c len / K, s + (c + 1) len / K)) and runs one workgroup per (tile,
// chunk), in four launches:
//  1. each chunk's per-pixel product of (1 - alpha) over its valid records, stopped once
//     it reaches T_MIN (every later chunk then starts at or below T_MIN);
//  2. per pixel, the exclusive prefix products in chunk order: the transmittance at each
//     chunk's start;
//  3. each chunk composites front to back from that transmittance with the reference's
//     absolute termination test T (1 - alpha) <= T_MIN; a pixel whose starting
//     transmittance is already at or below T_MIN has terminated in an earlier chunk and
//     composites nothing; a chunk records its colour sum, its end transmittance (negated
//     when the pixel terminated in it) and its last index;
//  4. a merge per pixel: the chunks' colours summed in order up to the terminating
//     chunk, the final transmittance and last contributor.
// The result is the sequential composite of rasterize_forward (cpu:574-626) up to float
// rounding of the transmittance products and colour sums. The backward first computes,
// per pixel and chunk, S at the chunk's end (the background term plus the colours of the
// later chunks up to the terminating one), then runs each chunk back to front from its
// end transmittance and that S.
struct ChunkView {
    int k, K;           // this chunk, chunks per tile
    size_t npix;        // pixels of the view (the stride between chunk planes)
    float *prod;        // [K][npix] the chunk's product of (1 - alpha); after the prefix pass the
                        // transmittance at the chunk's start; before a backward, S at its end
    float4 *state;      // [K][npix] (colour r, g, b, end transmittance; negated: terminated here)
    int32_t *last;      // [K][npix] last index the chunk composited (or k - 1 at termination), -1: none
};

__device__ inline void chunk_range(int s, int e, int k, int K, int &cs, int &ce) {
    const long len = e - s;
    cs = s + (int)(len * k / K);
    ce = s + (int)(len * (k + 1) / K);
}

// Launch 1 (PRODUCT) or 3 of the chunked forward for chunk ch.k of global tile gt. The
// product may run on below T_MIN within a batch: every later chunk then starts at or below
// it either way.
template <int FB, bool PRODUCT>
__device__ inline void forward_chunk(const TileView &v, const TileData &d, const ChunkView &ch, int gt, int lt) {
#pragma clang fp contract(fast)
    __shared__ float4 la[FB], lb[FB], lc[FB];
    __shared__ int wcount[2][FNT / 64];
    const int tx = lt % v.tiles_x, ty = lt / v.tiles_x;
    const float x0 = (float)(tx * TILE), y0 = (float)(ty * TILE);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int px = tx * TILE + (lane & 15), py = ty * TILE + 4 * FPT * w + (lane >> 4);
    int s, e;
    chunk_range(d.tile_start[gt], d.tile_start[gt + 1], ch.k, ch.K, s, e);
    const float fx = (float)px;
    Composite p;
    float fy[FPT];
    bool inside[FPT], entered[FPT];
    size_t o[FPT];
#pragma unroll
    for (int k = 0; k < FPT; k++) {
        fy[k] = (float)(py + 4 * k);
        inside[k] = px < (int)v.width && py + 4 * k < (int)v.height;
        o[k] = (size_t)ch.k * ch.npix + (inside[k] ? (size_t)(py + 4 * k) * v.width + px : 0);
        p.T[k] = !PRODUCT && inside[k] ? ch.prod[o[k]] : 1.f;  // at the chunk's start
        p.r[k] = p.g[k] = p.b[k] = p.depth[k] = 0.f;
        p.last[k] = p.last_j[k] = -1;
        entered[k] = PRODUCT || p.T[k] > T_MIN;  // else it terminated in an earlier chunk
        p.done[k] = !inside[k] || !entered[k];
    }
    for (int base = s; base < e; base += FB) {
        if (__syncthreads_count(p.all_done()) == FNT) break;
        const int n8 = stage_forward_batch<FB>(d, base, e, x0, y0, la, lb, lc, wcount);
        if (__ballot(!p.all_done()) == 0) continue;
        if (PRODUCT) {
            for (int j0 = 0; j0 < n8; j0 += 8) {
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const float4 A = la[j0 + u], B = lb[j0 + u];
                    const float dx = A.x - fx, adx2 = (A.z * dx) * dx, bdx = A.w * dx;
#pragma unroll
                    for (int k = 0; k < FPT; k++) {
                        const float x = splat_exponent(adx2, bdx, B.x, A.y - fy[k]);
                        const float alpha = splat_valid(x, B.z) ? splat_alpha(B.y, x) : 0.f;
                        p.T[k] -= alpha * p.T[k];
                    }
                }
#pragma unroll
                for (int k = 0; k < FPT; k++) p.done[k] = !inside[k] || !(p.T[k] > T_MIN);
                if (__ballot(!p.all_done()) == 0) break;
            }
        } else {
            composite_batch<false, true>(la, lb, lc, n8, fx, fy, p);
        }
    }
#pragma unroll
    for (int k = 0; k < FPT; k++) {
        if (!inside[k]) continue;
        if (PRODUCT) {
            ch.prod[o[k]] = p.T[k];
        } else {  // done inside the image: terminated in this chunk, unless it never entered it
            ch.state[o[k]] = make_float4(p.r[k], p.g[k], p.b[k], p.done[k] && entered[k] ? -p.T[k] : p.T[k]);
            ch.last[o[k]] = p.last[k];
        }
    }
}

// rasterize_backward (core/cpu/msplat_cpu.cpp:959-1031), slot values per intersection:
// a = (v_x, v_y, v_conic.x, v_conic.y), b = (v_conic.z, v_r, v_g, v_b), c = v_logit.
//
// PPT pixels per thread: 4/PPT waves per tile, wave w owning rows [4 PPT w, 4 PPT (w+1))
// and lane l the pixels (l % 16, 4 PPT w + l / 16 + 4 k), k < PPT.
//
// Per pixel the back-to-front recursion keeps T and one running scalar
//   S = <buffer + T_final bg, v_out>,  so  v_alpha = T <rgb, v_out> - S / (1 - alpha),
// and the per-gaussian gradients are assembled after the reduction from sufficient
// statistics of v_sigma = -alpha v_alpha:
//   v_conic = 1/2 (sum vs dx^2, sum vs dx dy, sum vs dy^2),
//   v_xy = (a sum vs dx + b sum vs dy, b sum vs dx + c sum vs dy),
//   v_logit = -(1 - o) sum vs, v_rgb = sum fac v_out (channels with raw + 0.5 >= 0).
// A lane first adds its PPT pixels; the sums are then made over the wave (wave_moments)
// and written to LDS, to be added over the waves in fixed order when the batch's slots are
// written. One partial per wave keeps the LDS footprint small enough for several waves per
// SIMD.
// Every slot flag is zero when the kernel starts (slot_prepare_kernel). A slot whose nine values are all
// zero (a record culled from the tile, behind every pixel's last contributor, or valid
// in no pixel) is not touched: its floats stay as they are, and the slot sums skip it.
// Skipping a zero term changes no sum: the sums start at +0, and adding +0 or -0 to +0
// or to a nonzero value returns it unchanged.
// With CHUNK the workgroup runs chunk ch.k of the tile's list (a depth-chunked forward
// made the frame): each pixel starts from the chunk's end transmittance and from S over
// the final transmittance's background plus the later chunks' colours.
// With AUX (rasterize_backward with f.aux, cpu:963-1025): each pixel also carries the
// prior losses' gradients v_d = dL/dD and v_a = dL/dA, which add
// (z T - Sd / (1 - alpha)) v_d + (T - Sa / (1 - alpha)) v_a to v_alpha, Sd and Sa being
// the sums of z fac and fac over the records behind. These terms have the colour term's
// form T c - S / (1 - alpha) with c = z v_d + v_a, so one running sum S of fac (c_rgb +
// z v_d + v_a) carries all three; the per-pixel background is bg_img, and each record's
// sum of fac v_d goes to its depth slot.
//
// The wave sums: lane l holds column l % 16 and the row group l / 16, so the nine sums are
// made of six (q0 = sum vs, q2 = sum vs dy, q5 = sum vs dy^2, and the three colours): adding
// over the row groups first, the dx-weighted ones follow per column. A permlane swap of two
// values leaves the halves (rows) of one in one register and of the other in the other, so
// one swap and one add sum both, each into its own rows: six values end in two registers
//   R0 rows (q0, q5, q2, q6), R1 rows (q7, q7, q8, q8),
// and three registers are summed along their rows of 16 lanes:
//   R0, M = (dx q0, q7, dx q2, q8), N = dx^2 R0 (row 0; row 2 carries the depth sum q9).
// 28 instructions against 38 for a butterfly over the nine values.
// a * b, and 0 whenever a factor is 0 (also against an infinity or a NaN): a pixel whose
// upstream gradient is not finite leaves the positions, conics and opacities of the records
// it does not see as they are. Their colour and depth sums, 0 times that gradient, become NaN
// where the pixel's wave adds them up for another pixel.
__device__ inline float mul_or_zero(float a, float b) {
    float r;
    asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

constexpr int NPART = 12;  // a record's wave sums: R0, M, N, four rows each
struct alignas(16) PartSums {  // in LDS; R0 and M are read back as float4
    float v[NPART];
};
static_assert(alignof(PartSums) == 16 && sizeof(PartSums) == 4 * NPART, "whole float4s, side by side");
struct WaveSums {
    float r0, m, n;
};
__device__ inline float sum_halves(float lo, float hi) {  // lanes 0-31: the wave's lo halves' sum, 32-63: hi's
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}
__device__ inline float sum_row_pairs(float even, float odd) {  // even rows: even's row pairs' sums, odd rows: odd's
    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(even), __float_as_uint(odd), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}
template <bool AUX>
__device__ inline WaveSums wave_moments(float q0, float q2, float q5, float q6, float q7, float q8, float q9, float dx,
                                        int row) {
    const float r0 = sum_row_pairs(sum_halves(q0, q2), sum_halves(q5, q6));
    const float c = sum_halves(q7, q8);
    const float r1 = AUX ? sum_row_pairs(sum_halves(q9, q9), c) : sum_row_pairs(c, c);  // (q9 | q7, q7, q9 | q8, q8)
    const float rx = r0 * dx;
    WaveSums s;
    s.r0 = row_sum16(r0);
    s.m = row_sum16(row & 1 ? r1 : rx);
    s.n = row_sum16(AUX && row == 2 ? r1 : rx * dx);
    return s;
}

template <int PPT, int BATCH, bool CHUNK = false, bool AUX = false>
__device__ inline void backward_tile(const TileView &v, const TileData &d, int gt, int lt,
                                     const ChunkView *ch = nullptr) {
#pragma clang fp contract(fast)
    constexpr int NT = 256 / PPT, NW = NT / 64;
    __shared__ float4 la[BATCH], lb[BATCH], lc[BATCH];  // stage_splat
    __shared__ float4 lconic[BATCH];  // the record's conic as projected (la and lb hold it scaled)
    __shared__ uint32_t lslot[BATCH];
    __shared__ uint8_t lmask[BATCH];  // bit c: raw colour c + 0.5 >= 0 (its gradient passes)
    __shared__ uint32_t ltouch[NW][(BATCH + 31) / 32];  // per wave, bit j: it had a valid pair with record j
    __shared__ PartSums part[NW][BATCH];
    __shared__ int smax[NW];
    __shared__ int wcount[2][NW];
    __shared__ int lclamp;  // some staged record's opacity reaches ALPHA_MAX: alphas may be clamped
    const int tx = lt % v.tiles_x, ty = lt / v.tiles_x;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int s = d.tile_start[gt], e = d.tile_start[gt + 1];
    if (CHUNK) chunk_range(s, e, ch->k, ch->K, s, e);
    if (s == e) return;
    const int px = tx * TILE + (lane & 15);
    const float x0 = (float)(tx * TILE), y0 = (float)(ty * TILE);
    float fy[PPT], T[PPT], S[PPT], vr[PPT], vg[PPT], vb[PPT];
    float vd[AUX ? PPT : 1], va[AUX ? PPT : 1];
    int last[PPT];
    int m = s - 1;
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int py = ty * TILE + 4 * PPT * w + (lane >> 4) + 4 * k;
        fy[k] = (float)py;
        T[k] = 0.f; S[k] = 0.f; vr[k] = 0.f; vg[k] = 0.f; vb[k] = 0.f;
        if (AUX) { vd[k] = 0.f; va[k] = 0.f; }
        last[k] = s - 1;
        if (px < (int)v.width && py < (int)v.height) {
            const size_t pid = (size_t)py * v.width + px;
            T[k] = v.final_T[pid];
            last[k] = min(v.final_idx[pid], e - 1);
            vr[k] = v.v_image[3 * pid];
            vg[k] = v.v_image[3 * pid + 1];
            vb[k] = v.v_image[3 * pid + 2];
            if (AUX) {
                vd[k] = v.v_aux[2 * pid];
                va[k] = v.v_aux[2 * pid + 1];
                S[k] = T[k] * (v.bg_img[3 * pid] * vr[k] + v.bg_img[3 * pid + 1] * vg[k] + v.bg_img[3 * pid + 2] * vb[k]);
            } else {
                S[k] = T[k] * (v.bg[0] * vr[k] + v.bg[1] * vg[k] + v.bg[2] * vb[k]);
            }
            if (CHUNK) {  // the chunk's end transmittance and S over everything behind it
                const size_t o = (size_t)ch->k * ch->npix + pid;
                T[k] = fabsf(ch->state[o].w);
                S[k] = ch->prod[o];
            }
        }
        m = max(m, last[k]);
    }
    // the block's furthest contributing intersection: nothing behind it is visited
    for (int dd = 32; dd >= 1; dd >>= 1) m = max(m, __shfl_xor(m, dd));
    if (lane == 0) smax[w] = m;
    __syncthreads();
    int kmax = smax[0];
#pragma unroll
    for (int i = 1; i < NW; i++) kmax = max(kmax, smax[i]);
    const float fx = (float)px;

    uint32_t nwritten = 0;  // slots this thread writes (counted when slots_written is given)
    for (int end = kmax + 1; end > s; end -= BATCH) {
        const int start = max(s, end - BATCH);
        const int n = end - start;
        __syncthreads();
        if (threadIdx.x == 0) lclamp = 0;
        // stage the batch's records that can reach the tile, in list order
        int kept = 0;
        for (int c = 0; c < n; c += NT) {
            const int i = c + threadIdx.x;
            bool keep = false;
            float4 A0, B0;
            float C0 = 0.f;
            uint32_t p = 0;
            float Z0 = 0.f;
            if (i < n) {
                const int g = d.gid[start + i];
                A0 = d.splat_a[g];
                B0 = d.splat_b[g];
                C0 = d.splat_blue[g];
                if (AUX) Z0 = d.depths[g];
                keep = !(d.cull && splat_misses_tile(A0, B0, x0, y0));
                if (keep) {
                    const uint2 r = d.rect[g];
                    const int rx0 = r.x & 0xFFFF, rx1 = r.x >> 16, ry0 = r.y & 0xFFFF;
                    p = d.offsets[g] + (uint32_t)((ty - ry0) * (rx1 - rx0) + (tx - rx0));
                }
            }
            int total;
            const int pos = kept + kept_position<NW>(keep, wcount[(c / NT) & 1], total);
            if (keep) {
                stage_splat(la, lb, lc, pos, A0, B0, C0, Z0, start + i);
                lconic[pos] = make_float4(A0.z, A0.w, B0.x, 0.f);
                lmask[pos] = (uint8_t)((B0.z + 0.5f >= 0.f ? 1 : 0) | (B0.w + 0.5f >= 0.f ? 2 : 0) |
                                       (C0 + 0.5f >= 0.f ? 4 : 0));
                lslot[pos] = p;
                if (!(B0.y < ALPHA_MAX)) lclamp = 1;  // kept_position's barrier is behind the reset
            }
            kept += total;
        }
        if (NW > 1)  // one wave writes its sums only to the records it reads them back from
            for (int i = threadIdx.x; i < NW * BATCH * NPART; i += NT) ((float *)part)[i] = 0.f;
        __syncthreads();
        // Per pixel, an invalid pair has alpha 0, which leaves T (times 1 / (1 - 0)) and S as
        // they are and adds zeros (vs by the product that is 0 whenever a factor is). Most
        // batches hold no opacity that reaches ALPHA_MAX, and their alphas need neither the
        // clamp nor the test that drops a clamped alpha's gradient.
        uint32_t touched[(BATCH + 31) / 32] = {};  // uniform
        auto records = [&](auto clamp) {
            constexpr bool CLAMP = decltype(clamp)::value;
            for (int j = kept - 1; j >= 0; j--) {
                const float4 A = la[j], B = lb[j], C = lc[j];
                const int kk = __float_as_int(B.w);
                // the lane's pixels share a column: dx and its products are per gaussian
                const float dx = A.x - fx;
                const float adx2 = (A.z * dx) * dx, bdx = A.w * dx;
                float q0 = 0.f, q2 = 0.f, q5 = 0.f, q6 = 0.f, q7 = 0.f, q8 = 0.f, q9 = 0.f;
                bool contrib = false;
#pragma unroll
                for (int k = 0; k < PPT; k++) {
                    const float dy = A.y - fy[k];
                    const float x = splat_exponent(adx2, bdx, B.x, dy);
                    const bool valid = kk <= last[k] && splat_valid(x, B.z);
                    contrib = contrib || valid;
                    const float raw = CLAMP ? splat_alpha(B.y, x) : B.y * __builtin_amdgcn_exp2f(-x);
                    const float alpha = valid ? raw : 0.f;
                    const float ra = __builtin_amdgcn_rcpf(1.f - alpha);
                    const float Tn = T[k] * ra, fac = alpha * Tn;
                    float cv = C.x * vr[k] + C.y * vg[k] + C.z * vb[k];
                    if (AUX) {
                        cv += C.w * vd[k] + va[k];
                        q9 += fac * vd[k];
                    }
                    const float v_alpha = S[k] * ra - Tn * cv;  // negated
                    T[k] = Tn;
                    S[k] += fac * cv;
                    q6 += fac * vr[k];
                    q7 += fac * vg[k];
                    q8 += fac * vb[k];
                    const float vs = mul_or_zero(CLAMP && !(alpha < ALPHA_MAX) ? 0.f : alpha, v_alpha);
                    const float vsy = vs * dy;
                    q0 += vs;
                    q2 += vsy;
                    q5 += vsy * dy;
                }
                if (__ballot(contrib) != 0) {
                    const WaveSums t = wave_moments<AUX>(q0, q2, q5, q6, q7, q8, q9, dx, lane >> 4);
                    const int c = lane & 15;
                    float sum = c == 0 ? t.r0 : c == 1 ? t.m : t.n;
                    asm volatile("" : "+v"(sum));  // the last row step before the branch, not in it
                    if (c < 3) part[w][j].v[4 * c + (lane >> 4)] = sum;
#pragma unroll
                    for (int i = 0; i < (BATCH + 31) / 32; i++) touched[i] |= (j >> 5) == i ? 1u << (j & 31) : 0u;
                }
            }
        };
        if (lclamp) records(std::true_type{});
        else records(std::false_type{});
        if (lane == 0)
#pragma unroll
            for (int i = 0; i < (BATCH + 31) / 32; i++) ltouch[w][i] = touched[i];
        __syncthreads();
        for (int j = threadIdx.x; j < kept; j += NT) {
            const uint32_t p = lslot[j];
            uint32_t any = 0;
#pragma unroll
            for (int r = 0; r < NW; r++) any |= ltouch[r][j >> 5];
            if (!((any >> (j & 31)) & 1u)) continue;  // every wave's partials are zero
            nwritten++;
            float4 R0 = *(const float4 *)&part[0][j].v[0], M = *(const float4 *)&part[0][j].v[4];
            float n0 = part[0][j].v[8], n2 = part[0][j].v[10];
#pragma unroll
            for (int r = 1; r < NW; r++) {
                const float4 R = *(const float4 *)&part[r][j].v[0], m = *(const float4 *)&part[r][j].v[4];
                R0.x += R.x; R0.y += R.y; R0.z += R.z; R0.w += R.w;
                M.x += m.x; M.y += m.y; M.z += m.z; M.w += m.w;
                n0 += part[r][j].v[8];
                n2 += part[r][j].v[10];
            }
            // sums of vs: R0.x; dx vs: M.x; dy vs: R0.z; dx^2: n0; dx dy: M.z; dy^2: R0.y; colours R0.w, M.y, M.w
            const float4 Q = lconic[j];  // the unscaled conic (a, b, c)
            const float ox = Q.x * M.x + Q.y * R0.z, oy = Q.y * M.x + Q.z * R0.z;
            const uint32_t cm = lmask[j];
            const bool mr = cm & 1u, mg = cm & 2u, mb = cm & 4u;
            d.slot_a[p] = make_float4(ox, oy, 0.5f * n0, 0.5f * M.z);
            d.slot_b[p] = make_float4(0.5f * R0.y, mr ? R0.w : 0.f, mg ? M.y : 0.f, mb ? M.w : 0.f);
            d.slot_c[p] = -(1.f - lb[j].y) * R0.x;
            d.slot_f[p] = 1;
            if (AUX) d.slot_d[p] = n2;
        }
    }
    if (d.slots_written) {  // one atomic per wave
        for (int dd = 32; dd >= 1; dd >>= 1) nwritten += __shfl_xor(nwritten, dd);
        if (lane == 0 && nwritten) atomicAdd(d.slots_written, (unsigned long long)nwritten);
    }
}

}  // namespace msplat
