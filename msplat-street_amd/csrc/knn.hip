// Exact 3-nearest-neighbour mean distance and Gaussian initialisation
// (msplat_knn3_mean_dist / msplat_init_gaussians, core/cpu/msplat_cpu.cpp:1499-1605).
//
// Points are ordered along a 30-bit Morton curve (LSD radix sort) and grouped into leaves of
// 64 consecutive points, with two further levels of 64 children per node, each node with its
// AABB. One wave searches for the 64 queries of a leaf, which lie close together: it seeds
// every query's three best squared distances from the leaf itself, then walks the tree,
// testing 64 children at a time (one per lane) against the leaf's own box and the largest of
// the queries' third-best distances. Of a leaf that may hold a closer point, each query
// tests the box itself, and the few that still need it are taken one by one, the 64 lanes
// computing the distances to the leaf's 64 points. Culling uses a conservative margin, so
// the three smallest squared distances (computed as dx*dx + dy*dy + dz*dz in float, unfused)
// are exactly those of a brute-force search.
//
// What bounds it: the scalar steps of a wave (a leaf visited, a query taken) and the latency
// of its dependent loads. A leaf of 64 is what one wave holds as queries and as candidates.
// It replaced one thread per query walking boxes of 128 points, whose 64 lanes disagreed on
// almost every box: the 475k points of a street, 2300 -> 280 us (a whole initialisation, 2450
// -> 390 us); 20k points, 1318 -> 243 us with the ordering; 200k points in one cell of the
// curve, beside an outlier at a thousand times their extent, 26.7 -> 3.6 ms.
#include "common.h"
#include "kernels.h"

namespace msplat {

constexpr int KNN_FAN = 64;  // points per leaf, children per node

__device__ inline uint32_t spread10(uint32_t v) {
    v &= 0x3FF;
    v = (v | (v << 16)) & 0x030000FF;
    v = (v | (v << 8)) & 0x0300F00F;
    v = (v | (v << 4)) & 0x030C30C3;
    v = (v | (v << 2)) & 0x09249249;
    return v;
}

// per-block min/max of the points; one float[6] per block
__global__ __launch_bounds__(256) void bounds_kernel(const float *pts, uint32_t n, float *out) {
    __shared__ float s[6][256];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        for (int a = 0; a < 3; a++) {
            lo[a] = fminf(lo[a], pts[3 * i + a]);
            hi[a] = fmaxf(hi[a], pts[3 * i + a]);
        }
    for (int a = 0; a < 3; a++) {
        s[a][threadIdx.x] = lo[a];
        s[3 + a][threadIdx.x] = hi[a];
    }
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st)
            for (int a = 0; a < 3; a++) {
                s[a][threadIdx.x] = fminf(s[a][threadIdx.x], s[a][threadIdx.x + st]);
                s[3 + a][threadIdx.x] = fmaxf(s[3 + a][threadIdx.x], s[3 + a][threadIdx.x + st]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) out[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// reduces the per-block bounds to one (written to out[0..6))
__global__ __launch_bounds__(256) void bounds_final_kernel(const float *blk, int nblk, float *out) {
    __shared__ float s[6][256];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int b = threadIdx.x; b < nblk; b += 256)
        for (int a = 0; a < 3; a++) {
            lo[a] = fminf(lo[a], blk[6 * b + a]);
            hi[a] = fmaxf(hi[a], blk[6 * b + 3 + a]);
        }
    for (int a = 0; a < 3; a++) {
        s[a][threadIdx.x] = lo[a];
        s[3 + a][threadIdx.x] = hi[a];
    }
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st)
            for (int a = 0; a < 3; a++) {
                s[a][threadIdx.x] = fminf(s[a][threadIdx.x], s[a][threadIdx.x + st]);
                s[3 + a][threadIdx.x] = fmaxf(s[3 + a][threadIdx.x], s[3 + a][threadIdx.x + st]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) out[threadIdx.x] = s[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void morton_kernel(const float *pts, uint32_t n, const float *bb, uint32_t *codes,
                                                    int32_t *idx) {
    const float lo[3] = {bb[0], bb[1], bb[2]}, hi[3] = {bb[3], bb[4], bb[5]};
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t q[3];
    for (int a = 0; a < 3; a++) {
        const float ext = hi[a] - lo[a];
        float t = ext > 0.f ? (pts[3 * i + a] - lo[a]) / ext : 0.f;
        q[a] = (uint32_t)fminf(fmaxf(t * 1023.f, 0.f), 1023.f);
    }
    codes[i] = spread10(q[0]) | (spread10(q[1]) << 1) | (spread10(q[2]) << 2);
    idx[i] = (int32_t)i;
}

__global__ __launch_bounds__(256) void gather_points_kernel(const float *pts, const int32_t *order, uint32_t n,
                                                           float4 *sorted) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int32_t j = order[i];
    sorted[i] = make_float4(pts[3 * j], pts[3 * j + 1], pts[3 * j + 2], 0.f);
}

// An AABB as two float4: lo at [2 i], hi at [2 i + 1]
struct KnnBox {
    float lo[3], hi[3];
};
__device__ inline KnnBox load_box(const float4 *boxes, uint32_t i) {
    const float4 l = boxes[2 * (size_t)i], h = boxes[2 * (size_t)i + 1];
    return KnnBox{{l.x, l.y, l.z}, {h.x, h.y, h.z}};
}

// Boxes of groups of KNN_FAN consecutive points (LEAF) or boxes, one wave each
template <bool LEAF>
__global__ __launch_bounds__(256) void group_bounds_kernel(const float4 *in, uint32_t n, float4 *out) {
    const uint32_t g = blockIdx.x * 4 + (threadIdx.x >> 6), i = g * KNN_FAN + (threadIdx.x & 63);
    if (g * KNN_FAN >= n) return;  // the whole wave
    KnnBox b{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
    if (i < n) {
        if (LEAF) {
            const float4 p = in[i];
            b = KnnBox{{p.x, p.y, p.z}, {p.x, p.y, p.z}};
        } else {
            b = load_box(in, i);
        }
    }
    for (int d = 32; d >= 1; d >>= 1)
        for (int a = 0; a < 3; a++) {
            b.lo[a] = fminf(b.lo[a], __shfl_xor(b.lo[a], d));
            b.hi[a] = fmaxf(b.hi[a], __shfl_xor(b.hi[a], d));
        }
    if ((threadIdx.x & 63) == 0) {
        out[2 * (size_t)g] = make_float4(b.lo[0], b.lo[1], b.lo[2], 0.f);
        out[2 * (size_t)g + 1] = make_float4(b.hi[0], b.hi[1], b.hi[2], 0.f);
    }
}

__device__ inline float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline KnnBox lane_box(const KnnBox &b, int l) {
    KnnBox r;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        r.lo[a] = lane_value(b.lo[a], l);
        r.hi[a] = lane_value(b.hi[a], l);
    }
    return r;
}

// Whether two boxes may hold points at a float-rounded squared distance below `best`:
// every rounding here and in a point distance is below 1e-6 of its value, and the bound is
// shrunk by 1e-5 (an underflow makes it smaller still).
__device__ inline bool boxes_within(const KnnBox &p, const KnnBox &q, float best) {
    float d2 = 0.f;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float d = fmaxf(0.f, fmaxf(p.lo[a] - q.hi[a], q.lo[a] - p.hi[a]));
        d2 += d * d;
    }
    return d2 * (1.f - 1e-5f) < best;
}

// d into the sorted three smallest b0 <= b1 <= b2
__device__ inline void insert3(float d, float &b0, float &b1, float &b2) {
    b2 = __builtin_amdgcn_fmed3f(b1, b2, d);
    b1 = __builtin_amdgcn_fmed3f(b0, b1, d);
    b0 = fminf(b0, d);
}

__device__ inline float wave_max(float v) {
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    return v;
}

__global__ __launch_bounds__(256) void knn3_kernel(const float4 *sp, const int32_t *order, uint32_t n,
                                                  const float4 *leaf, uint32_t nleaf, const float4 *mid, uint32_t nmid,
                                                  const float4 *top, uint32_t ntop, float *mean_dist) {
    const int lane = threadIdx.x & 63;
    const uint32_t g = blockIdx.x * 4 + (threadIdx.x >> 6);  // the wave's leaf
    if (g >= nleaf) return;
    const uint32_t i = g * KNN_FAN + lane;
    float4 q = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
    if (i < n) q = sp[i];
    const bool live = isfinite(q.x) && isfinite(q.y) && isfinite(q.z);  // else no point is at a finite distance
    float b0 = INFINITY, b1 = INFINITY, b2 = live ? INFINITY : -INFINITY;
    // the leaf's own points
    for (int k = 0; k < KNN_FAN && g * KNN_FAN + k < n; k++) {
        const float dx = lane_value(q.x, k) - q.x, dy = lane_value(q.y, k) - q.y, dz = lane_value(q.z, k) - q.z;
        const float d = dx * dx + dy * dy + dz * dz;
        if (live && lane != k && d < b2) insert3(d, b0, b1, b2);
    }
    const KnnBox own = load_box(leaf, g);
    float best = wave_max(b2);  // of the live queries
    const KnnBox me{{q.x, q.y, q.z}, {q.x, q.y, q.z}};
    // leaf c with box b (both the same in every lane)
    auto visit = [&](uint32_t c, const KnnBox &b) {
        uint64_t need = __ballot(live && boxes_within(b, me, b2));
        if (need == 0) return;
        const uint32_t j = c * KNN_FAN + lane;
        float4 p = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
        if (j < n) p = sp[j];
        while (need) {
            const int t = __builtin_ctzll(need);
            need &= need - 1;
            const float dx = p.x - lane_value(q.x, t), dy = p.y - lane_value(q.y, t), dz = p.z - lane_value(q.z, t);
            const float d = dx * dx + dy * dy + dz * dz;
            uint64_t closer = __ballot(d < lane_value(b2, t));
            while (closer) {
                const int s = __builtin_ctzll(closer);
                closer &= closer - 1;
                const float ds = lane_value(d, s);
                if (lane == t) insert3(ds, b0, b1, b2);
            }
        }
    };
    // neighbours along the curve first, then the own middle node: they shrink the bound
    if (g > 0) visit(g - 1, load_box(leaf, g - 1));
    if (g + 1 < nleaf) visit(g + 1, load_box(leaf, g + 1));
    best = wave_max(b2);
    const uint32_t home = g / KNN_FAN;
    // (a leaf visited twice would insert its points twice: the neighbours are left out)
    auto skip = [&](uint32_t c) { return c == g || c + 1 == g || c == g + 1; };
    // Middle node m with box mb. A leaf whose points straddle a jump of the curve has a box
    // that overlaps most of the tree (alone, it took 0.8 ms at 475k points), so the queries
    // that need the node are found first, and its leaves are tested against those alone.
    auto walk_mid = [&](uint32_t m, const KnnBox &mb) {
        const bool need = live && boxes_within(mb, me, b2);
        if (__ballot(need) == 0) return;
        KnnBox near;
        float far2 = need ? b2 : -INFINITY;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            near.lo[a] = need ? me.lo[a] : INFINITY;
            near.hi[a] = need ? me.hi[a] : -INFINITY;
        }
        for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
            for (int a = 0; a < 3; a++) {
                near.lo[a] = fminf(near.lo[a], __shfl_xor(near.lo[a], d));
                near.hi[a] = fmaxf(near.hi[a], __shfl_xor(near.hi[a], d));
            }
            far2 = fmaxf(far2, __shfl_xor(far2, d));
        }
        const uint32_t c = m * KNN_FAN + lane;
        KnnBox b{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
        if (c < nleaf) b = load_box(leaf, c);
        uint64_t todo = __ballot(c < nleaf && !skip(c) && boxes_within(b, near, far2));
        while (todo) {
            const int t = __builtin_ctzll(todo);
            todo &= todo - 1;
            visit(m * KNN_FAN + t, lane_box(b, t));
        }
        best = wave_max(b2);
    };
    walk_mid(home, load_box(mid, home));
    for (uint32_t t0 = 0; t0 < ntop; t0 += KNN_FAN) {
        const uint32_t t = t0 + lane;
        uint64_t tops = __ballot(t < ntop && boxes_within(load_box(top, t < ntop ? t : 0), own, best));
        while (tops) {
            const uint32_t u = t0 + __builtin_ctzll(tops);
            tops &= tops - 1;
            const uint32_t m = u * KNN_FAN + lane;
            const KnnBox b = load_box(mid, m < nmid ? m : 0);
            uint64_t mids = __ballot(m < nmid && m != home && boxes_within(b, own, best));
            while (mids) {
                const int k = __builtin_ctzll(mids);
                mids &= mids - 1;
                walk_mid(u * KNN_FAN + k, lane_box(b, k));
            }
        }
    }
    if (i >= n) return;
    float sum = 0.f, cnt = 0.f;
    if (isfinite(b0)) { sum += sqrtf(b0); cnt += 1.f; }
    if (isfinite(b1)) { sum += sqrtf(b1); cnt += 1.f; }
    if (isfinite(b2)) { sum += sqrtf(b2); cnt += 1.f; }
    mean_dist[order[i]] = cnt > 0.f ? sum / cnt : 1.f;
}

// log-scales, Shoemake rotations from the PCG stream, DC colour, constant opacity
__global__ __launch_bounds__(256) void init_gaussians_kernel(const float *md, const uint8_t *rgb, uint32_t n,
                                                            uint32_t seed, float logit, float *scales, float *quats,
                                                            float *dc, float *opac) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float ls = log_cr(fmaxf(md[i], 1e-7f));
    scales[3 * i] = ls;
    scales[3 * i + 1] = ls;
    scales[3 * i + 2] = ls;
    const float u = rand_uniform(seed, 3u * i), v = rand_uniform(seed, 3u * i + 1u), w = rand_uniform(seed, 3u * i + 2u);
    const float tau = 6.28318530717958647692f;
    quats[4 * i + 0] = sqrtf(1.f - u) * sin_cr(tau * v);
    quats[4 * i + 1] = sqrtf(1.f - u) * cos_cr(tau * v);
    quats[4 * i + 2] = sqrtf(u) * sin_cr(tau * w);
    quats[4 * i + 3] = sqrtf(u) * cos_cr(tau * w);
    for (int k = 0; k < 3; k++) dc[3 * i + k] = ((float)rgb[3 * i + k] * (1.f / 255.f) - 0.5f) / SH_C0;
    opac[i] = logit;
}

int knn3_launch(const float *pts, uint32_t n, float *mean_dist, KnnScratch &w, hipStream_t s) {
    if (n == 0) return 0;
    const int nb = (int)((n + 255) / 256);
    const int nbb = nb < 1024 ? nb : 1024;
    bounds_kernel<<<nbb, 256, 0, s>>>(pts, n, w.bounds);
    bounds_final_kernel<<<1, 256, 0, s>>>(w.bounds, nbb, w.bounds + 6 * 1024);
    morton_kernel<<<nb, 256, 0, s>>>(pts, n, w.bounds + 6 * 1024, w.codes, w.order);
    fill_u32<<<1, 1, 0, s>>>(w.n_dev, n);
    for (int shift = 0; shift < 30; shift += 8)
        launch_radix_pass(w.codes, w.order, w.codes_tmp, w.order_tmp, w.n_dev, n, shift, w.hist, w.digit_total, s),
            std::swap(w.codes, w.codes_tmp), std::swap(w.order, w.order_tmp);
    const uint32_t nleaf = (n + KNN_FAN - 1) / KNN_FAN, nmid = (nleaf + KNN_FAN - 1) / KNN_FAN,
                   ntop = (nmid + KNN_FAN - 1) / KNN_FAN;
    gather_points_kernel<<<nb, 256, 0, s>>>(pts, w.order, n, w.sorted);
    group_bounds_kernel<true><<<(nleaf + 3) / 4, 256, 0, s>>>(w.sorted, n, w.leaf);
    group_bounds_kernel<false><<<(nmid + 3) / 4, 256, 0, s>>>(w.leaf, nleaf, w.mid);
    group_bounds_kernel<false><<<(ntop + 3) / 4, 256, 0, s>>>(w.mid, nmid, w.top);
    knn3_kernel<<<(nleaf + 3) / 4, 256, 0, s>>>(w.sorted, w.order, n, w.leaf, nleaf, w.mid, nmid, w.top, ntop, mean_dist);
    return 0;
}

static size_t knn_boxes(uint32_t n) {  // of all three levels
    const size_t nleaf = ((size_t)n + KNN_FAN - 1) / KNN_FAN, nmid = (nleaf + KNN_FAN - 1) / KNN_FAN;
    return nleaf + nmid + (nmid + KNN_FAN - 1) / KNN_FAN;
}

size_t knn_scratch_bytes(uint32_t n) {
    return 16 * (size_t)n + 32 * knn_boxes(n) + 4 * 4 * (size_t)n + 6 * 1025 * 4 + 4 * radix_hist_words(n) + 4 * 256 + 64;
}

void knn_scratch_carve(void *base, uint32_t n, KnnScratch &w) {
    const size_t nleaf = ((size_t)n + KNN_FAN - 1) / KNN_FAN, nmid = (nleaf + KNN_FAN - 1) / KNN_FAN;
    w.sorted = (float4 *)base;
    w.leaf = w.sorted + n;
    w.mid = w.leaf + 2 * nleaf;
    w.top = w.mid + 2 * nmid;
    w.codes = (uint32_t *)(w.leaf + 2 * knn_boxes(n));
    w.codes_tmp = w.codes + n;
    w.order = (int32_t *)(w.codes_tmp + n);
    w.order_tmp = w.order + n;
    w.bounds = (float *)(w.order_tmp + n);
    w.hist = (uint32_t *)(w.bounds + 6 * 1025);
    w.digit_total = w.hist + radix_hist_words(n);
    w.n_dev = w.digit_total + 256;
}

void launch_init_gaussians(const float *md, const uint8_t *rgb, uint32_t n, uint32_t seed, float logit, float *scales,
                           float *quats, float *dc, float *opac, hipStream_t s) {
    if (n == 0) return;
    init_gaussians_kernel<<<(n + 255) / 256, 256, 0, s>>>(md, rgb, n, seed, logit, scales, quats, dc, opac);
}

}  // namespace msplat
