// Projection + SH colour, the visible records' depth order, and the stable LSD radix
// sort.
//
// Layout in HBM (per record, SoA, written once per view; a record is a gaussian in one
// view, record v * n + g in a batch of views):
//   splat_a = (x, y, conic.x, conic.y)   float4
//   splat_b = (conic.z, sigmoid(opacity), r, g)   float4
//   splat_blue = b, depths, aabb (float2), rect (x0 | x1 << 16, y0 | y1 << 16), count
//
// Binning keeps the reference's per-tile order, ascending (depth bits, gaussian id)
// (core/cpu/msplat_cpu.cpp:505-537): the visible records are compacted in id order and
// stably sorted by their 32-bit depth bits (4 passes over the visible records, not over
// the intersections), and the tiles' lists are expanded from that order (tile_lists.hip).
// Records own contiguous slot ranges (offsets[r], count[r]) in record order, tiles
// row-major within a record, which the backward's per-record reductions read.
#include <algorithm>

#include "kernels.h"
#include "proj_math.h"

namespace msplat {

// Block-wide exclusive scan of one u32 per thread (256 threads, 4 waves).
__device__ inline uint32_t block_scan_u32(uint32_t v, uint32_t &total, uint32_t *lds4) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds4[w] = x;
    __syncthreads();
    uint32_t pre = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i < w) pre += lds4[i];
        total += lds4[i];
    }
    __syncthreads();
    return pre + x - v;
}

// ── projection + SH colour (project_and_sh, msplat_cpu.cpp:452-500) ────────────
// Also writes the workgroup's intersection count and visible-record count.
// SP: the camera comes from the device StepParams block (a captured step), chosen at
// compile time so that the launch-by-launch step reads it from the kernel arguments.
// The SH coefficients of a wave's visible gaussians are staged in LDS by stage_sh
// (dynamic LDS: project_sh_lds bytes for the degree in use).
template <bool SP>
__global__ __launch_bounds__(256) void project_kernel(ProjectArgs a) {
    extern __shared__ float shl[];
    __shared__ uint32_t lds4[4];
    __shared__ uint8_t widx[4][64];
    const msplat_hip_camera &cam = SP ? a.sp->cam : a.cam;
    const int g = blockIdx.x * 256 + threadIdx.x;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t count = 0;
    bool need = false;
    float p[3] = {0.f, 0.f, 0.f}, pv[3] = {0.f, 0.f, 0.f}, conic[3] = {0.f, 0.f, 0.f}, radius = 0.f;
    float px = 0.f, py = 0.f, ax = 0.f, ay = 0.f;
    int x0 = 0, y0 = 0, x1 = 0, y1 = 0;
    if (g < a.n) {
        a.radii[g] = 0;
        a.count[g] = 0;
        p[0] = a.means[3 * g]; p[1] = a.means[3 * g + 1]; p[2] = a.means[3 * g + 2];
        cam_space(cam.viewmat, p, pv);
        if (pv[2] > cam.clip_thresh) {
            const float s[3] = {exp_cr(a.scales[3 * g]), exp_cr(a.scales[3 * g + 1]), exp_cr(a.scales[3 * g + 2])};
            const float q[4] = {a.quats[4 * g], a.quats[4 * g + 1], a.quats[4 * g + 2], a.quats[4 * g + 3]};
            float cov[6], c2[3];
            covariance3d(s, cam.glob_scale, q, cov);
            const float tfx = 0.5f * (float)cam.width / cam.fx, tfy = 0.5f * (float)cam.height / cam.fy;
            ewa_cov2d(cov, cam.viewmat, cam.fx, cam.fy, tfx, tfy, pv, c2);
            if (conic_radius(c2, conic, radius)) {
                to_pixel(cam.projmat, p, cam.width, cam.height, cam.cx, cam.cy, px, py);
                ax = ceilf(3.f * sqrtf(c2[0]));
                ay = ceilf(3.f * sqrtf(c2[2]));
                tile_rect(px, py, ax, ay, cam.tiles_x, cam.tiles_y, x0, y0, x1, y1);
                need = (x1 - x0) * (y1 - y0) > 0;
            }
        }
    }
    // staged when higher bands are in use, up to SH degree 3 (project_sh_lds); the DC
    // alone (three floats a lane) and degree 4 are read in place
    const size_t stride = 3 * (size_t)(sh_bases(cam.degree) - 1);
    const bool staged = cam.degree <= 3 && cam.degrees_to_use >= 1;
    const int u = 3 * (int)sh_bases(cam.degrees_to_use), us = u | 1;
    float *wl = shl + (size_t)w * 64 * us;
    if (staged) stage_sh(need, g - lane, a.dc, a.rest, stride, u, us, wl, widx[w]);
    if (need) {
        float d[3], col[3];
        view_direction(p, cam.cam_pos, d);
        const float *mine = wl + lane * us;
        if (staged) sh_color(cam.degrees_to_use, d, mine, mine + 3, col);
        else sh_color(cam.degrees_to_use, d, a.dc + 3 * (size_t)g, a.rest + stride * g, col);
        const float opac = 1.f / (1.f + exp_cr(-a.opac[g]));
        a.splat_a[g] = make_float4(px, py, conic[0], conic[1]);
        a.splat_b[g] = make_float4(conic[2], opac, col[0], col[1]);
        a.splat_blue[g] = col[2];
        a.depths[g] = pv[2];
        a.aabb[g] = make_float2(ax, ay);
        a.rect[g] = make_uint2((uint32_t)x0 | ((uint32_t)x1 << 16), (uint32_t)y0 | ((uint32_t)y1 << 16));
        a.radii[g] = (int)radius;
        count = (uint32_t)((x1 - x0) * (y1 - y0));
        a.count[g] = count;
    }
    uint32_t total, vis;
    block_scan_u32(count, total, lds4);
    block_scan_u32(count > 0 ? 1u : 0u, vis, lds4);
    if (threadIdx.x == 0) {
        a.block_sums[blockIdx.x] = total;
        a.block_vis[blockIdx.x] = vis;
    }
}

// Tile rectangles and counts re-derived from a frame's projection outputs (pixel
// centre in splat_a, aabb, radii), for binning outputs a caller injected.
__global__ __launch_bounds__(256) void rect_count_kernel(int n, const float4 *splat_a, const float2 *aabb,
                                                        const int32_t *radii, int tx, int ty, uint2 *rect,
                                                        uint32_t *count, uint32_t *block_sums, uint32_t *block_vis) {
    __shared__ uint32_t lds4[4];
    const int g = blockIdx.x * 256 + threadIdx.x;
    uint32_t c = 0;
    if (g < n) {
        if (radii[g] > 0) {
            const float4 A = splat_a[g];
            const float2 e = aabb[g];
            int x0, y0, x1, y1;
            tile_rect(A.x, A.y, e.x, e.y, tx, ty, x0, y0, x1, y1);
            if ((x1 - x0) * (y1 - y0) > 0) c = (uint32_t)((x1 - x0) * (y1 - y0));
            rect[g] = make_uint2((uint32_t)x0 | ((uint32_t)x1 << 16), (uint32_t)y0 | ((uint32_t)y1 << 16));
        }
        count[g] = c;
    }
    uint32_t total, vis;
    block_scan_u32(c, total, lds4);
    block_scan_u32(c > 0 ? 1u : 0u, vis, lds4);
    if (threadIdx.x == 0) {
        block_sums[blockIdx.x] = total;
        block_vis[blockIdx.x] = vis;
    }
}

// Exclusive scan of the per-block counts of a small array (one block, sequential
// chunks); writes the bases and the total (u64, so that > 2^31 is detected).
__global__ __launch_bounds__(256) void scan_blocks_kernel(uint32_t *sums, int nblocks, uint64_t *total,
                                                          uint32_t *total32, uint32_t *zero_also) {
    __shared__ uint32_t lds4[4];
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) {
        carry = 0;
        if (zero_also) *zero_also = 0;
    }
    __syncthreads();
    for (int base = 0; base < nblocks; base += 256) {
        const int i = base + threadIdx.x;
        uint32_t v = i < nblocks ? sums[i] : 0, t;
        uint32_t ex = block_scan_u32(v, t, lds4);
        uint64_t c = carry;
        if (i < nblocks) sums[i] = (uint32_t)(c + ex);
        __syncthreads();
        if (threadIdx.x == 0) carry = c + t;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *total = carry;
        *total32 = carry > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)carry;
    }
}

// ── multi-level exclusive scan of a u32 array (4096 entries per workgroup) ─────
constexpr int SCAN_CHUNK = 4096;

__global__ __launch_bounds__(256) void scan_partial_kernel(const uint32_t *a, uint32_t L, uint32_t *partial) {
    __shared__ uint32_t lds4[4];
    const uint32_t base = blockIdx.x * SCAN_CHUNK + threadIdx.x * 16;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (base + i < L) s += a[base + i];
    uint32_t t;
    block_scan_u32(s, t, lds4);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// Scans the chunk totals; the grand total goes to total/total32. Over `cap`, total32 is
// 0 and *overflow is set (when overflow is given; with `applied`, a set overflow also
// counts as over capacity).
__global__ __launch_bounds__(256) void scan_top_kernel(uint32_t *partial, int nchunks, ScanOut o) {
    __shared__ uint32_t lds4[4];
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nchunks; base += 256) {
        const int i = base + threadIdx.x;
        uint32_t v = i < nchunks ? partial[i] : 0, t;
        const uint32_t ex = block_scan_u32(v, t, lds4);
        const uint64_t c = carry;
        if (i < nchunks) partial[i] = (uint32_t)(c + ex);
        __syncthreads();
        if (threadIdx.x == 0) carry = c + t;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const uint64_t tot = carry;
        const bool over = tot > (uint64_t)o.cap || (o.applied && *o.overflow);
        if (o.total) *o.total = tot;
        if (o.total32) *o.total32 = over ? (o.overflow ? 0u : 0xFFFFFFFFu) : (uint32_t)tot;
        if (o.overflow) *o.overflow = over ? 1u : 0u;
        if (o.zero_also) *o.zero_also = 0u;
        if (o.applied && !over) *o.applied += 1u;
        if (o.running) *o.running += tot;
    }
}

// The whole scan in one workgroup of 1024 threads, 16384 entries at a time: one launch and
// one round for up to 4M gaussians' block sums or a 2560x1440 view's tiles.
constexpr int SCAN_SMALL_THREADS = 1024, SCAN_SMALL_CHUNK = 16 * SCAN_SMALL_THREADS;
__device__ inline void scan_small(uint32_t *a, uint32_t L, const ScanOut &o) {
    __shared__ uint32_t wsum[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint64_t carry = 0;  // the same in every thread
    const bool wide = ((uintptr_t)a & 15) == 0;  // a thread's 16 entries as four 16-byte loads and stores
    for (uint32_t chunk = 0; chunk < L; chunk += SCAN_SMALL_CHUNK) {
        const uint32_t base = chunk + threadIdx.x * 16;
        const bool whole = wide && base + 16 <= L;
        uint32_t v[16], sum = 0;
        if (whole) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint4 q = ((const uint4 *)(a + base))[i];
                v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = base + i < L ? a[base + i] : 0u;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) sum += v[i];
        uint32_t x = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d);
            if (lane >= d) x += y;
        }
        if (lane == 63) wsum[w] = x;
        __syncthreads();
        uint32_t pre = 0, total = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t t = wsum[i];
            pre += i < w ? t : 0u;
            total += t;
        }
        __syncthreads();  // wsum is written again
        uint32_t run = (uint32_t)carry + pre + x - sum;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t t = v[i];
            v[i] = run;
            run += t;
        }
        if (whole) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                ((uint4 *)(a + base))[i] = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (base + i < L) a[base + i] = v[i];
        }
        carry += total;
    }
    if (threadIdx.x == 0) {
        const uint64_t tot = carry;
        const bool over = tot > (uint64_t)o.cap || (o.applied && *o.overflow);
        if (o.total) *o.total = tot;
        if (o.total32) *o.total32 = over ? (o.overflow ? 0u : 0xFFFFFFFFu) : (uint32_t)tot;
        if (o.overflow) *o.overflow = over ? 1u : 0u;
        if (o.zero_also) *o.zero_also = 0u;
        if (o.applied && !over) *o.applied += 1u;
        if (o.running) *o.running += tot;
    }
}

__global__ __launch_bounds__(SCAN_SMALL_THREADS) void scan_small_kernel(uint32_t *a, uint32_t L, ScanOut o) {
    scan_small(a, L, o);
}

// Two small scans of the same length in one launch, one workgroup each
__global__ __launch_bounds__(SCAN_SMALL_THREADS) void scan_small_pair_kernel(uint32_t *a0, ScanOut o0, uint32_t *a1,
                                                                            ScanOut o1, uint32_t L) {
    if (blockIdx.x == 0) scan_small(a0, L, o0);
    else scan_small(a1, L, o1);
}

__global__ __launch_bounds__(256) void scan_apply_kernel(uint32_t *a, uint32_t L, const uint32_t *partial) {
    __shared__ uint32_t lds4[4];
    const uint32_t base = blockIdx.x * SCAN_CHUNK + threadIdx.x * 16;
    uint32_t v[16], s = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        v[i] = base + i < L ? a[base + i] : 0u;
        s += v[i];
    }
    uint32_t t;
    uint32_t ex = block_scan_u32(s, t, lds4) + partial[blockIdx.x];
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (base + i < L) {
            a[base + i] = ex;
            ex += v[i];
        }
}

// ── visible records in id order, keyed by depth bits ──────────────────────────
// Also each record's intersection offset (the slots of the raster backward lie in record
// order).
__global__ __launch_bounds__(256) void compact_kernel(CompactArgs a) {
    __shared__ uint32_t lds4[4];
    const int v = blockIdx.y;
    const int g = blockIdx.x * 256 + threadIdx.x;
    const size_t r = (size_t)v * a.n + g;
    const uint32_t c = g < a.n ? a.count[r] : 0u;
    const bool vis = c > 0;
    uint32_t t;
    const uint32_t ex = block_scan_u32(vis ? 1u : 0u, t, lds4);
    if (t == 0) return;  // uniform: nothing visible in this workgroup
    const uint32_t off = block_scan_u32(c, t, lds4);
    if (vis) {
        const size_t blk = (size_t)v * a.nbx + blockIdx.x;
        const uint32_t pos = a.block_vis[blk] + ex;
        a.dkeys[pos] = __float_as_uint(a.depths[r]);
        a.dvals[pos] = (int32_t)r;
        a.offsets[r] = a.block_sums[blk] + off;
    }
}

// Clears the slots' zero flags and lists the records with more than BIG_SLOTS
// intersections (in no particular order): each workgroup counts those of its part of the
// records, takes its place in the list with one atomic, and writes them. One atomic per
// 256 records, as the list was first built, serialised on its counter (about 12 ns each:
// 21 us at 475k records, 360 us for a batch of 8 views of 1M). Few workgroups pay less for
// the atomics, many clear the flags faster. By itself, with 17 slots a record and one record
// in eight listed, 256 workgroups / 1024: 10.7 / 18.0 us at 475k records, 17.1 / 21.0 at
// 1.5M, 23.8 / 22.8 at 2M (the line), 31.2 / 25.8 at 3M, 86 / 46 at 8M.
constexpr size_t SLOT_PREPARE_GRID = 1024;
constexpr uint32_t SLOT_PREPARE_MANY = 2u << 20;
__global__ __launch_bounds__(256) void slot_prepare_kernel(SlotPrepareArgs a) {
    __shared__ uint32_t lds4[4];
    __shared__ uint32_t s_base;
    const size_t tid = (size_t)blockIdx.x * 256 + threadIdx.x, quads = a.nwords / 4;
    for (size_t i = tid; i < quads; i += (size_t)gridDim.x * 256)
        reinterpret_cast<uint4 *>(a.flag_words)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (tid < a.nwords - 4 * quads) a.flag_words[4 * quads + tid] = 0u;
    if (a.overflow && *a.overflow) return;
    const uint32_t per = (a.nrec + gridDim.x - 1) / gridDim.x;
    const uint32_t b = min(blockIdx.x * per, a.nrec), e = min(b + per, a.nrec);
    uint32_t n = 0;
    for (uint32_t r = b + threadIdx.x; r < e; r += 256) n += a.count[r] > BIG_SLOTS ? 1u : 0u;
    uint32_t total;
    uint32_t p = block_scan_u32(n, total, lds4);
    if (total == 0) return;
    if (threadIdx.x == 0) s_base = atomicAdd(a.big_count, total);
    __syncthreads();
    p += s_base;
    for (uint32_t r = b + threadIdx.x; r < e; r += 256)
        if (a.count[r] > BIG_SLOTS) a.big_list[p++] = r;
}

// ── stable LSD radix sort, 8-bit digits, 32- or 64-bit keys, int32 payload ─────
// Each workgroup owns an element block of ITEMS consecutive elements (4096 for large
// sorts, 1024 for small ones, so that they still spread over the device): an upsweep
// histogram, a per-digit scan over blocks, and a scatter that ranks the elements stably
// within the block (wave multi-split over ballots of the digit bits), stages them in
// LDS in digit order, and writes each digit's run to consecutive addresses.

// The workgroups of a pass loop over the element blocks that the device-side count
// needs, so a grid sized for a capacity does no empty work; histogram column b of
// digit d lives at hist[d * stride + b].
template <int ITEMS>
__device__ inline uint32_t rs_blocks(const uint32_t *n_ptr) { return (*n_ptr + ITEMS - 1) / ITEMS; }

template <typename K, int ITEMS>
__global__ __launch_bounds__(256) void rs_hist_kernel(const K *keys, const uint32_t *n_ptr, int shift, uint32_t mask,
                                                     uint32_t *hist, int stride) {
    __shared__ uint32_t h[256];
    const uint32_t n = *n_ptr, nb = rs_blocks<ITEMS>(n_ptr);
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
        h[threadIdx.x] = 0;
        __syncthreads();
        const uint32_t start = b * ITEMS;
        for (int r = 0; r < ITEMS / 256; r++) {
            uint32_t e = start + r * 256 + threadIdx.x;
            if (e < n) atomicAdd(&h[(uint32_t)(keys[e] >> shift) & mask], 1u);
        }
        __syncthreads();
        hist[(size_t)threadIdx.x * stride + b] = h[threadIdx.x];
        __syncthreads();
    }
}

// one block per digit: exclusive scan of that digit's counts over blocks, digit total;
// each thread takes SCAN_RUN consecutive counts, so 2048 blocks take one round
constexpr int SCAN_RUN = 8;
template <int ITEMS>
__global__ __launch_bounds__(256) void rs_scan_kernel(uint32_t *hist, int stride, const uint32_t *n_ptr,
                                                     uint32_t *digit_total) {
    __shared__ uint32_t lds4[4];
    __shared__ uint32_t carry;
    const int nblocks = (int)rs_blocks<ITEMS>(n_ptr);
    uint32_t *row = hist + (size_t)blockIdx.x * stride;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nblocks; base += 256 * SCAN_RUN) {
        const int i0 = base + threadIdx.x * SCAN_RUN;
        uint32_t v[SCAN_RUN], sum = 0, t;
#pragma unroll
        for (int j = 0; j < SCAN_RUN; j++) {
            v[j] = i0 + j < nblocks ? row[i0 + j] : 0u;
            sum += v[j];
        }
        const uint32_t ex = block_scan_u32(sum, t, lds4);
        const uint32_t c = carry;
        uint32_t run = c + ex;
#pragma unroll
        for (int j = 0; j < SCAN_RUN; j++)
            if (i0 + j < nblocks) {
                row[i0 + j] = run;
                run += v[j];
            }
        __syncthreads();
        if (threadIdx.x == 0) carry = c + t;
        __syncthreads();
    }
    if (threadIdx.x == 0) digit_total[blockIdx.x] = carry;
}

// Wave w ranks its own contiguous quarter of the workgroup's elements, 64 at a time,
// with private per-digit counters (no workgroup barrier inside the loop); the waves'
// counts are then combined in wave order, which keeps the sort stable.
// One element block of a pass; `my_base` is this thread's digit's global start for the block.
template <typename K, int ITEMS>
__device__ inline void rs_scatter_block(const K *kin, const int32_t *vin, K *kout, int32_t *vout, uint32_t n,
                                        int shift, uint32_t mask, uint32_t start, uint32_t my_base,
                                        const ListEntries &entries) {
    constexpr int R = ITEMS / 256;  // rounds of 64 elements per wave
    __shared__ K sk[ITEMS];
    __shared__ int32_t sv[ITEMS];
    __shared__ uint32_t gbase[256], lstart[256];
    __shared__ uint32_t wcnt[4][256];
    __shared__ uint32_t lds4[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    gbase[tid] = my_base;
#pragma unroll
    for (int i = 0; i < 4; i++) wcnt[w][lane + 64 * i] = 0;
    const uint32_t wstart = start + (uint32_t)w * (64 * R);
    K key[R];
    int32_t val[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t e = wstart + r * 64 + lane;
        key[r] = e < n ? kin[e] : K(0);
        val[r] = e < n ? vin[e] : 0;
    }
    wave_sync();
    // per element: digit (bits 24..31) and rank among the wave's elements of that digit
    uint32_t dr[R];
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const bool valid = wstart + r * 64 + lane < n;
        const uint32_t digit = valid ? (uint32_t)(key[r] >> shift) & mask : 0;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (digit >> b) & 1;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t before = valid ? wcnt[w][digit] : 0u;
        wave_sync();
        if (valid && (peers & lt) == 0) wcnt[w][digit] = before + (uint32_t)__popcll(peers);
        wave_sync();
        dr[r] = (digit << 24) | (before + (uint32_t)__popcll(peers & lt));
    }
    __syncthreads();
    {   // per digit: wave offsets (in wave order) and the block's local start
        const uint32_t c0 = wcnt[0][tid], c1 = wcnt[1][tid], c2 = wcnt[2][tid], c3 = wcnt[3][tid];
        uint32_t t;
        const uint32_t ls = block_scan_u32(c0 + c1 + c2 + c3, t, lds4);
        lstart[tid] = ls;
        wcnt[0][tid] = ls;
        wcnt[1][tid] = ls + c0;
        wcnt[2][tid] = ls + c0 + c1;
        wcnt[3][tid] = ls + c0 + c1 + c2;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (wstart + r * 64 + lane < n) {
            const uint32_t p = wcnt[w][dr[r] >> 24] + (dr[r] & 0xFFFFFF);
            sk[p] = key[r];
            sv[p] = val[r];
        }
    }
    __syncthreads();
    const uint32_t cnt = min((uint32_t)ITEMS, n - start);
    for (uint32_t p = tid; p < cnt; p += 256) {
        const K k = sk[p];
        const uint32_t d = (uint32_t)(k >> shift) & mask;
        const uint32_t o = gbase[d] + (p - lstart[d]);
        const int32_t v = sv[p];
        vout[o] = v;
        if (entries.lrect) {
            const uint2 q = entries.rect[v];
            entries.lrect[o] = entries.direct ? make_uint2((uint32_t)v, pack_local(q, 0, 0)) : q;
        } else {
            kout[o] = k;
        }
    }
}

template <typename K, int ITEMS>
__global__ __launch_bounds__(256) void rs_scatter_kernel(const K *kin, const int32_t *vin, K *kout, int32_t *vout,
                                                        const uint32_t *n_ptr, int shift, uint32_t mask,
                                                        const uint32_t *hist, int stride, const uint32_t *digit_total,
                                                        ListEntries entries) {
    __shared__ uint32_t dex[256];
    __shared__ uint32_t lds4[4];
    {   // exclusive prefix of the digit totals
        uint32_t t;
        dex[threadIdx.x] = block_scan_u32(digit_total[threadIdx.x], t, lds4);
    }
    const uint32_t nb = rs_blocks<ITEMS>(n_ptr);
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
        __syncthreads();
        rs_scatter_block<K, ITEMS>(kin, vin, kout, vout, *n_ptr, shift, mask, b * ITEMS,
                                   dex[threadIdx.x] + hist[(size_t)threadIdx.x * stride + b], entries);
    }
}

// View id of each depth-sorted record, the key of one more stable pass that makes the
// record order view-major (each view's records in depth order)
__global__ __launch_bounds__(256) void view_keys_kernel(const int32_t *recs, const uint32_t *n_ptr, int n,
                                                       uint32_t *keys) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < *n_ptr) keys[i] = (uint32_t)(recs[i] / n);
}

// ── batched views ────────────────────────────────────────────────────────────

// Projection of gaussian g into every view of the batch: the parameters are read once
// and record v * n + g is written per view, with the same arithmetic as project_kernel
// (the records are bit-identical to one-view projections). Per view, the workgroup's
// intersection and visible-record counts go to block_sums / block_vis[v * nbx + b].
// The SH coefficients of the bands in use by any view (a.sh_u floats per gaussian) are
// staged in LDS once for all views (dynamic LDS: project_sh_lds bytes).
__global__ __launch_bounds__(256) void project_batch_kernel(BatchProjectArgs a) {
    extern __shared__ float shl[];
    __shared__ uint32_t lds4[4];
    __shared__ uint8_t widx[4][64];
    const int g = blockIdx.x * 256 + threadIdx.x;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool live = g < a.n;
    float p[3] = {0.f, 0.f, 0.f}, s[3] = {0.f, 0.f, 0.f}, q[4] = {1.f, 0.f, 0.f, 0.f}, logit = 0.f;
    if (live) {
        p[0] = a.means[3 * g]; p[1] = a.means[3 * g + 1]; p[2] = a.means[3 * g + 2];
        s[0] = exp_cr(a.scales[3 * g]); s[1] = exp_cr(a.scales[3 * g + 1]); s[2] = exp_cr(a.scales[3 * g + 2]);
        q[0] = a.quats[4 * g]; q[1] = a.quats[4 * g + 1]; q[2] = a.quats[4 * g + 2]; q[3] = a.quats[4 * g + 3];
        logit = a.opac[g];
    }
    const float opac = 1.f / (1.f + exp_cr(-logit));
    // staged up to SH degree 3 (sh_u > 0); degree 4 reads its coefficients in place
    const int us = a.sh_u | 1;
    float *wl = shl + (size_t)w * 64 * us;
    if (a.sh_u) stage_sh(live, g - lane, a.dc, a.rest, a.sh_stride, a.sh_u, us, wl, widx[w]);
    const float *mine = wl + lane * us;
    for (int v = 0; v < a.num_views; v++) {
        const msplat_hip_camera &cam = a.tab->views[v].cam;
        const size_t r = (size_t)v * a.n + g;
        uint32_t count = 0;
        if (live) {
            a.radii[r] = 0;
            a.count[r] = 0;
            float pv[3];
            cam_space(cam.viewmat, p, pv);
            if (pv[2] > cam.clip_thresh) {
                float cov[6], c2[3], conic[3], radius;
                covariance3d(s, cam.glob_scale, q, cov);
                const float tfx = 0.5f * (float)cam.width / cam.fx, tfy = 0.5f * (float)cam.height / cam.fy;
                ewa_cov2d(cov, cam.viewmat, cam.fx, cam.fy, tfx, tfy, pv, c2);
                if (conic_radius(c2, conic, radius)) {
                    float px, py;
                    to_pixel(cam.projmat, p, cam.width, cam.height, cam.cx, cam.cy, px, py);
                    const float ax = ceilf(3.f * sqrtf(c2[0])), ay = ceilf(3.f * sqrtf(c2[2]));
                    int x0, y0, x1, y1;
                    tile_rect(px, py, ax, ay, cam.tiles_x, cam.tiles_y, x0, y0, x1, y1);
                    if ((x1 - x0) * (y1 - y0) > 0) {
                        float d[3], col[3];
                        view_direction(p, cam.cam_pos, d);
                        if (a.sh_u) sh_color(cam.degrees_to_use, d, mine, mine + 3, col);
                        else sh_color(cam.degrees_to_use, d, a.dc + 3 * (size_t)g, a.rest + a.sh_stride * g, col);
                        a.splat_a[r] = make_float4(px, py, conic[0], conic[1]);
                        a.splat_b[r] = make_float4(conic[2], opac, col[0], col[1]);
                        a.splat_blue[r] = col[2];
                        a.depths[r] = pv[2];
                        a.rect[r] = make_uint2((uint32_t)x0 | ((uint32_t)x1 << 16),
                                               (uint32_t)y0 | ((uint32_t)y1 << 16));
                        a.radii[r] = (int)radius;
                        count = (uint32_t)((x1 - x0) * (y1 - y0));
                        a.count[r] = count;
                    }
                }
            }
        }
        uint32_t total, vis;
        block_scan_u32(count, total, lds4);
        block_scan_u32(count > 0 ? 1u : 0u, vis, lds4);
        if (threadIdx.x == 0) {
            a.block_sums[(size_t)v * a.nbx + blockIdx.x] = total;
            a.block_vis[(size_t)v * a.nbx + blockIdx.x] = vis;
        }
    }
}

// ── host launchers ───────────────────────────────────────────────────────────

size_t scan_partial_words(uint32_t L) { return (size_t)(L + SCAN_CHUNK - 1) / SCAN_CHUNK + 1; }

void launch_scan_u32(uint32_t *a, uint32_t L, uint32_t *partial, const ScanOut &o, hipStream_t s) {
    if (L <= 3 * SCAN_SMALL_CHUNK) {  // one launch
        scan_small_kernel<<<1, SCAN_SMALL_THREADS, 0, s>>>(a, L, o);
        return;
    }
    const int nchunks = (int)((L + SCAN_CHUNK - 1) / SCAN_CHUNK);
    if (nchunks > 0) scan_partial_kernel<<<nchunks, 256, 0, s>>>(a, L, partial);
    scan_top_kernel<<<1, 256, 0, s>>>(partial, nchunks, o);
    if (nchunks > 0) scan_apply_kernel<<<nchunks, 256, 0, s>>>(a, L, partial);
}

void launch_scan_u32_pair(uint32_t *a0, const ScanOut &o0, uint32_t *a1, const ScanOut &o1, uint32_t L,
                          uint32_t *partial0, uint32_t *partial1, hipStream_t s) {
    if (L <= 3 * SCAN_SMALL_CHUNK) {
        scan_small_pair_kernel<<<2, SCAN_SMALL_THREADS, 0, s>>>(a0, o0, a1, o1, L);
        return;
    }
    launch_scan_u32(a0, L, partial0, o0, s);
    launch_scan_u32(a1, L, partial1, o1, s);
}

// LDS of project_kernel's SH staging (four waves of 64 lanes, an odd count of floats per
// lane) for the bands up to `degree`; none when the stored degree is 4 or only the DC is
// in use (read in place)
size_t project_sh_lds(uint32_t degree, uint32_t stored) {
    return stored > 3 || degree == 0 ? 0 : 4 * 64 * (size_t)((3 * sh_bases(degree)) | 1) * sizeof(float);
}

void launch_project(const ProjectArgs &a, hipStream_t s) {
    const int nb = (a.n + 255) / 256;
    if (nb > 0) {
        // a captured step takes the degree in use from device memory: room for every band stored
        if (a.sp) project_kernel<true><<<nb, 256, project_sh_lds(a.cam.degree, a.cam.degree), s>>>(a);
        else project_kernel<false><<<nb, 256, project_sh_lds(a.cam.degrees_to_use, a.cam.degree), s>>>(a);
    }
}

void launch_rect_count(int n, const float4 *splat_a, const float2 *aabb, const int32_t *radii, int tx, int ty,
                       uint2 *rect, uint32_t *count, uint32_t *block_sums, uint32_t *block_vis, hipStream_t s) {
    const int nb = (n + 255) / 256;
    if (nb > 0)
        rect_count_kernel<<<nb, 256, 0, s>>>(n, splat_a, aabb, radii, tx, ty, rect, count, block_sums, block_vis);
}

void launch_scan_blocks(uint32_t *sums, int nblocks, uint64_t *total, uint32_t *total32, hipStream_t s,
                        uint32_t *zero_also) {
    scan_blocks_kernel<<<1, 256, 0, s>>>(sums, nblocks, total, total32, zero_also);
}

void launch_slot_prepare(const SlotPrepareArgs &a, hipStream_t s) {
    const size_t blocks = std::max((a.nwords + 1023) / 1024, ((size_t)a.nrec + 255) / 256);
    const size_t most = a.nrec < SLOT_PREPARE_MANY ? SLOT_PREPARE_GRID / 4 : SLOT_PREPARE_GRID;
    if (blocks) slot_prepare_kernel<<<(unsigned)std::min(blocks, most), 256, 0, s>>>(a);
}

void launch_compact(const CompactArgs &a, hipStream_t s) {
    if (a.nbx > 0 && a.num_views > 0) compact_kernel<<<dim3(a.nbx, a.num_views), 256, 0, s>>>(a);
}

// Element blocks of a pass: RS_ITEMS elements from RS_LARGE elements up, RS_ITEMS_SMALL
// below (the histogram words hold the smaller blocks' count either way).
constexpr int RS_ITEMS_SMALL = 1024;
constexpr uint32_t RS_LARGE = 2u << 20;

size_t radix_hist_words(uint32_t n_max) {
    return (size_t)256 * ((n_max + RS_ITEMS_SMALL - 1) / RS_ITEMS_SMALL + 1);
}

// Grid caps of the capacity-sized launches: the workgroups loop over what the device
// count needs.
constexpr uint32_t HIST_GRID = 2048, SCATTER_GRID = 1024;

template <typename K, int ITEMS>
static void radix_pass_items(const K *kin, const int32_t *vin, K *kout, int32_t *vout, const uint32_t *n_dev,
                             uint32_t n_max, int shift, uint32_t mask, uint32_t *hist, uint32_t *digit_total,
                             hipStream_t s, const ListEntries &entries) {
    const uint32_t nblocks = (n_max + ITEMS - 1) / ITEMS;
    if (nblocks == 0) return;
    rs_hist_kernel<K, ITEMS><<<std::min(nblocks, HIST_GRID), 256, 0, s>>>(kin, n_dev, shift, mask, hist, (int)nblocks);
    rs_scan_kernel<ITEMS><<<256, 256, 0, s>>>(hist, (int)nblocks, n_dev, digit_total);
    rs_scatter_kernel<K, ITEMS><<<std::min(nblocks, SCATTER_GRID), 256, 0, s>>>(kin, vin, kout, vout, n_dev, shift,
                                                                                mask, hist, (int)nblocks, digit_total,
                                                                                entries);
}

template <typename K>
static void radix_pass(const K *kin, const int32_t *vin, K *kout, int32_t *vout, const uint32_t *n_dev,
                       uint32_t n_max, int shift, uint32_t mask, uint32_t *hist, uint32_t *digit_total, hipStream_t s,
                       const ListEntries &entries = ListEntries{nullptr, nullptr, false}) {
    if (n_max >= RS_LARGE)
        radix_pass_items<K, RS_ITEMS>(kin, vin, kout, vout, n_dev, n_max, shift, mask, hist, digit_total, s, entries);
    else
        radix_pass_items<K, RS_ITEMS_SMALL>(kin, vin, kout, vout, n_dev, n_max, shift, mask, hist, digit_total, s,
                                            entries);
}

void launch_radix_pass(const uint64_t *kin, const int32_t *vin, uint64_t *kout, int32_t *vout, const uint32_t *n_dev,
                       uint32_t n_max, int shift, uint32_t *hist, uint32_t *digit_total, hipStream_t s, uint32_t mask) {
    radix_pass<uint64_t>(kin, vin, kout, vout, n_dev, n_max, shift, mask, hist, digit_total, s);
}

void launch_radix_pass(const uint32_t *kin, const int32_t *vin, uint32_t *kout, int32_t *vout, const uint32_t *n_dev,
                       uint32_t n_max, int shift, uint32_t *hist, uint32_t *digit_total, hipStream_t s, uint32_t mask,
                       const ListEntries &entries) {
    radix_pass<uint32_t>(kin, vin, kout, vout, n_dev, n_max, shift, mask, hist, digit_total, s, entries);
}

void launch_view_keys(const int32_t *recs, const uint32_t *n_dev, uint32_t n_max, int n, uint32_t *keys,
                      hipStream_t s) {
    if (n_max) view_keys_kernel<<<(n_max + 255) / 256, 256, 0, s>>>(recs, n_dev, n, keys);
}

void launch_batch_project(const BatchProjectArgs &a, hipStream_t s) {
    if (a.nbx > 0) project_batch_kernel<<<a.nbx, 256, 4 * 64 * (size_t)(a.sh_u | 1) * sizeof(float), s>>>(a);
}

}  // namespace msplat
