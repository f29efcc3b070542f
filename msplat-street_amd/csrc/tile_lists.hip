// Per-tile lists of the visible records in depth order, by two expansions of the
// depth-ordered list: into supertiles of 8x8 tiles, then each supertile's list into its
// 64 tiles. The reference sorts one key per (tile, record) intersection
// (core/cpu/msplat_cpu.cpp:505-567); here an intersection is written once, in place.
//
// Both levels run the same step. A node (a region of 8x8 child cells with a list of
// records) is cut into units of consecutive list entries, one workgroup each, whose waves
// take consecutive parts, 64 entries at a time, one per lane. Lane r forms the 64-bit mask
// of the cells its record covers (8 bits per row of cells), and a 64x64 bit transpose over
// the wave leaves lane c with the set of entries that cover cell c. Their number is a
// popcount, and their places in the cell's list follow in entry order, so the lists are
// stable by construction: no sort keys, no ranking. Per level, three launches: the counts
// per cell of every unit and of the waves within it, an exclusive prefix of the units'
// counts over each node, and the expansion, whose lane c writes the entries of cell c.
//   level 1: node = 8x8 supertiles (1024x1024 pixels), its list the whole view's
//            depth-ordered records, of which those that miss the node are dropped first;
//            cell = supertile
//   level 2: node = supertile; cell = tile
// A view of at most 8x8 tiles is one supertile and starts at level 2.
//
// Measured (sum of the launches between the depth sort and the rasterizer, one view unless
// said), before: an emission of every intersection's key, two radix passes (histogram,
// digit scan, ranking scatter) and a range search, which moved each key five times; after:
//   3M gaussians, 3840x2160 (94 M intersections)    3350 -> 660 us
//   2M gaussians, 1920x1080 (31 M)                   800 -> 225 us
//   475k, 1264x832 (8 M)                             183 ->  60 us
//   batch of 8 views, 1M gaussians, train step      4640 -> 560 us
//   20k, 128x128 (35k)                                33 ->  18 us
// What bounds it: level 2's expansion by its stores (31 M words in 100 us at 1920x1080,
// runs of about ten words), level 1's by the latency of its few waves; a small frame by
// its launches (3-6 us each). The depth sort's last pass writes the first entries, in place of
// a gather after it (per frame 4.7 us of launches for 3 of work at 475k, 7 less at 3M).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace msplat {

// Each level's entries are dealt to at most this many waves (8 on each of the 1024 SIMDs),
// plus one partly filled unit per node. Level 1 has few nodes with long lists: large
// units keep the prefix over a node's units short (one workgroup walks it). Level 2 has
// many shorter lists, which would leave most of a large unit idle.
constexpr uint32_t LIST_WAVES = 8192;
constexpr uint32_t WAVES1 = 16, WAVES2 = 4;  // waves per unit
constexpr uint32_t UNITS1 = LIST_WAVES / WAVES1, UNITS2 = LIST_WAVES / WAVES2;

// ── 64x64 bit transpose over a wave ──────────────────────────────────────────
// Lane r holds row r (bit c = column c); afterwards lane c holds column c. Six exchange
// steps with partner lane ^ d, d = 32..1: a lane keeps the half of its bits whose index
// agrees with its own in bit d and takes the partner's, moved by d.
struct BitTranspose {
    uint32_t sel16, sel8, keep4, keep2, keep1, rot4, rot2, rot1;
    __device__ explicit BitTranspose(int lane) {
        // v_perm_b32 selectors over (second, first): bytes 0-3 of the first, 4-7 of the second
        sel16 = lane & 16 ? 0x07060302u : 0x05040100u;  // halves of (odd row, even row)
        sel8 = lane & 8 ? 0x03070105u : 0x06020400u;    // bytes of (partner, own)
        keep4 = lane & 4 ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
        keep2 = lane & 2 ? 0xCCCCCCCCu : 0x33333333u;
        keep1 = lane & 1 ? 0xAAAAAAAAu : 0x55555555u;
        rot4 = lane & 4 ? 4u : 28u;  // rotate right: >> d for the upper partner, << d for the lower
        rot2 = lane & 2 ? 2u : 30u;
        rot1 = lane & 1 ? 1u : 31u;
    }
    template <int CTRL>
    static __device__ inline uint32_t dpp(uint32_t v) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
    }
    __device__ inline uint32_t within32(uint32_t x) const {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);  // even row's value, odd row's value
        x = __builtin_amdgcn_perm(r[1], r[0], sel16);
        x = __builtin_amdgcn_perm(dpp<0x128>(x), x, sel8);  // row_ror:8
        uint32_t p = dpp<0x1b>(dpp<0x141>(x));              // row_half_mirror, quad reversed: lane ^ 4
        x = (x & keep4) | (__builtin_amdgcn_alignbit(p, p, rot4) & ~keep4);
        p = dpp<0x4e>(x);  // quad_perm [2,3,0,1]
        x = (x & keep2) | (__builtin_amdgcn_alignbit(p, p, rot2) & ~keep2);
        p = dpp<0xb1>(x);  // quad_perm [1,0,3,2]
        return (x & keep1) | (__builtin_amdgcn_alignbit(p, p, rot1) & ~keep1);
    }
    __device__ inline void operator()(uint32_t &lo, uint32_t &hi) const {
        const auto r = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
        lo = within32(r[0]);
        hi = within32(r[1]);
    }
};

// Mask of the cells [x0, x1) x [y0, y1) of an 8x8 node (bit 8 y + x); empty when either
// range is.
__device__ inline void cell_mask(int x0, int x1, int y0, int y1, uint32_t &lo, uint32_t &hi) {
    lo = hi = 0u;
    if (x0 < x1 && y0 < y1) {
        const uint32_t row = (1u << x1) - (1u << x0);
        const uint32_t rows = row * 0x01010101u;
        const uint64_t ys = (~0ull << (8 * y0)) & (~0ull >> (64 - 8 * y1));
        lo = rows & (uint32_t)ys;
        hi = rows & (uint32_t)(ys >> 32);
    }
}

// The last i in [0, n) with starts[i] <= u (starts rises from starts[0] = 0), found by the
// whole wave: each round tests 64 probes of the range.
__device__ inline uint32_t find_start(const uint32_t *starts, uint32_t n, uint32_t u, int lane) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t st = (hi - lo + 63) / 64;
        const uint32_t i = lo + (uint32_t)lane * st;
        const uint32_t c = (uint32_t)__popcll(__ballot(i < hi && starts[i] <= u));
        lo += (c - 1) * st;
        hi = min(lo + st, hi);
    }
    return lo;
}

// groups of 64 entries per wave of a level with `total` list entries over its nodes
__device__ inline uint32_t wave_groups(uint64_t total) {
    uint32_t g = 1;
    while ((uint64_t)g * 64u * LIST_WAVES < total) g <<= 1;
    return g;
}

template <uint32_t WAVES>
__device__ inline uint32_t unit_count(uint32_t len, uint32_t groups) {
    return (len + 64 * WAVES * groups - 1) / (64 * WAVES * groups);
}

__device__ inline uint32_t visible(const TileListArgs &a) {
    return a.overflow && *a.overflow ? 0u : *a.nvis;  // a frame over capacity has empty lists
}

// View v's part of the depth-ordered list of a batch: the visible records before it, from
// the scanned visible counts per (view, block)
__device__ inline uint32_t view_first(const TileListArgs &a, int v, uint32_t nvis) {
    return v < a.tab->num_views ? min(a.block_vis[(size_t)v * a.nbx], nvis) : nvis;
}

// ── level 1 nodes ────────────────────────────────────────────────────────────
// Node i of view v covers supertiles [8 hx, 8 hx + 8) x [8 hy, 8 hy + 8).
struct Node1 {
    uint32_t s, e, groups, first_unit;
    int hx, hy;
};

template <bool BATCH>
__device__ inline uint32_t level1_nodes(const TileListArgs &a) {
    return BATCH ? a.tab->node_base[a.tab->num_views] : (uint32_t)a.nodes;
}

__device__ inline uint32_t one_view_groups(const TileListArgs &a, uint32_t nvis) {
    return wave_groups((uint64_t)nvis * (uint64_t)a.nodes);
}

template <bool BATCH>
__device__ inline uint32_t level1_units(const TileListArgs &a) {
    if (BATCH) return a.unit1[level1_nodes<true>(a)];
    const uint32_t nvis = visible(a);
    return (uint32_t)a.nodes * unit_count<WAVES1>(nvis, one_view_groups(a, nvis));
}

template <bool BATCH>
__device__ inline Node1 level1_node(const TileListArgs &a, uint32_t i) {
    Node1 k;
    if (BATCH) {
        int v = 0;
        while (v + 1 < a.tab->num_views && a.tab->node_base[v + 1] <= i) v++;
        const uint32_t nvis = visible(a), local = i - a.tab->node_base[v];
        const uint32_t nx = ((uint32_t)a.tab->views[v].cam.tiles_x + 63) / 64;
        k.s = view_first(a, v, nvis);
        k.e = view_first(a, v + 1, nvis);
        k.groups = a.plan[0];
        k.first_unit = a.unit1[i];
        k.hx = (int)(local % nx);
        k.hy = (int)(local / nx);
    } else {
        const uint32_t nvis = visible(a), nx = ((uint32_t)a.tiles_x + 63) / 64;
        k.s = 0;
        k.e = nvis;
        k.groups = one_view_groups(a, nvis);
        k.first_unit = i * unit_count<WAVES1>(nvis, k.groups);
        k.hx = (int)(i % nx);
        k.hy = (int)(i / nx);
    }
    return k;
}

// Exclusive scan of one value per thread over a 1024-thread workgroup.
__device__ inline uint32_t block_scan_1024(uint32_t v, uint32_t &total, uint32_t *lds16) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds16[w] = x;
    __syncthreads();
    uint32_t pre = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint32_t t = lds16[i];
        pre += i < w ? t : 0u;
        total += t;
    }
    __syncthreads();
    return pre + x - v;
}

// Batch: the level-1 units of every node (one workgroup)
__global__ __launch_bounds__(1024) void list_plan1_kernel(TileListArgs a) {
    __shared__ uint32_t lds16[16];
    const uint32_t nodes = level1_nodes<true>(a), nvis = visible(a);
    uint64_t entries = 0;  // uniform: at most MAX_VIEWS terms
    for (int v = 0; v < a.tab->num_views; v++)
        entries += (uint64_t)(view_first(a, v + 1, nvis) - view_first(a, v, nvis)) *
                   (a.tab->node_base[v + 1] - a.tab->node_base[v]);
    const uint32_t g = wave_groups(entries);
    if (threadIdx.x == 0) a.plan[0] = g;
    uint32_t carry = 0;
    for (uint32_t b = 0; b < nodes; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        uint32_t units = 0, total;
        if (i < nodes) {
            int v = 0;
            while (v + 1 < a.tab->num_views && a.tab->node_base[v + 1] <= i) v++;
            const uint32_t len = view_first(a, v + 1, nvis) - view_first(a, v, nvis);
            units = unit_count<WAVES1>(len, g);
        }
        const uint32_t ex = block_scan_1024(units, total, lds16);
        if (i < nodes) a.unit1[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) a.unit1[nodes] = carry;
}

// The supertiles' list starts and level-2 units from their totals (one workgroup).
// plan[1] = the level-2 groups per unit.
template <bool BATCH>
__device__ inline void plan2(const TileListArgs &a, uint32_t *lds16) {
    const uint32_t n = 64 * level1_nodes<BATCH>(a);
    uint32_t carry = 0;
    for (uint32_t b = 0; b < n; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        uint32_t total;
        const uint32_t ex = block_scan_1024(i < n ? a.super_total[i] : 0u, total, lds16);
        if (i < n) a.super_start[i] = carry + ex;
        carry += total;
    }
    const uint32_t g = wave_groups(carry);
    if (threadIdx.x == 0) {
        a.super_start[n] = carry;
        a.plan[1] = g;
    }
    uint32_t units = 0;
    for (uint32_t b = 0; b < n; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        uint32_t total;
        const uint32_t ex = block_scan_1024(i < n ? unit_count<WAVES2>(a.super_total[i], g) : 0u, total, lds16);
        if (i < n) a.unit2[i] = units + ex;
        units += total;
    }
    if (threadIdx.x == 0) a.unit2[n] = units;
}

// ── level 2 nodes ────────────────────────────────────────────────────────────
struct Node2 {
    uint32_t s, e, groups, first_unit;
};

// A view of one supertile has no plan: its list is the whole view's
__device__ inline Node2 level2_node(const TileListArgs &a, uint32_t i) {
    if (a.direct) {
        const uint32_t nvis = visible(a);
        return Node2{0u, nvis, wave_groups(nvis), 0u};
    }
    return Node2{a.super_start[i], a.super_start[i + 1], a.plan[1], a.unit2[i]};
}

template <bool BATCH>
__device__ inline uint32_t level2_nodes(const TileListArgs &a) {
    return a.direct ? 1u : 64 * level1_nodes<BATCH>(a);
}

template <bool BATCH>
__device__ inline uint32_t level2_units(const TileListArgs &a) {
    if (a.direct) {
        const uint32_t nvis = visible(a);
        return unit_count<WAVES2>(nvis, wave_groups(nvis));
    }
    return a.unit2[level2_nodes<BATCH>(a)];
}

// Global id of the tile of supertile i that lane c owns, -1 outside the view's grid
template <bool BATCH>
__device__ inline int tile_of(const TileListArgs &a, uint32_t i, int c) {
    const uint32_t node = i >> 6;
    uint32_t local = node, base = 0;
    int tx = a.tiles_x, ty = a.tiles_y;
    if (BATCH) {
        int v = 0;
        while (v + 1 < a.tab->num_views && a.tab->node_base[v + 1] <= node) v++;
        local = node - a.tab->node_base[v];
        base = a.tab->tile_base[v];
        tx = a.tab->views[v].cam.tiles_x;
        ty = a.tab->views[v].cam.tiles_y;
    }
    const uint32_t nx = ((uint32_t)tx + 63) / 64;
    const int x = (int)(64 * (local % nx) + 8 * (i & 7) + (c & 7));
    const int y = (int)(64 * (local / nx) + 8 * ((i >> 3) & 7) + (c >> 3));
    return x < tx && y < ty ? (int)base + y * tx + x : -1;
}

// ── list entries ─────────────────────────────────────────────────────────────
// A level-1 entry is a record and its tile rectangle; a level-2 entry is a record and the
// rectangle within its supertile (pack_local). The last pass of the depth sort writes the
// first entries (level 1 reads them once per node) beside the records.
__device__ inline void local_mask(uint32_t p, uint32_t &lo, uint32_t &hi) {
    cell_mask((int)(p & 15), (int)((p >> 4) & 15), (int)((p >> 8) & 15), (int)((p >> 12) & 15), lo, hi);
}

// supertiles of node (hx, hy) that the tile rectangle touches
__device__ inline void super_mask(uint2 r, int hx, int hy, uint32_t &lo, uint32_t &hi) {
    const int x0 = (int)((r.x & 0xFFFF) >> 3) - 8 * hx, x1 = (int)(((r.x >> 16) + 7) >> 3) - 8 * hx;
    const int y0 = (int)((r.y & 0xFFFF) >> 3) - 8 * hy, y1 = (int)(((r.y >> 16) + 7) >> 3) - 8 * hy;
    cell_mask(max(x0, 0), min(x1, 8), max(y0, 0), min(y1, 8), lo, hi);
}

// ── level 1: the records of a wave's part that touch the node ────────────────
// Reads entries [s, e) of the list and calls step(n) for every 64 records that touch the
// node (n < 64 the last time), which lie in order in rect[0, n) / rec[0, n): the wave's
// part of LDS, 128 entries. Dropping the others first keeps the masks full where a view
// has many nodes (12 at 3840x2160).
template <bool IDS, typename F>
__device__ inline void touching_records(const TileListArgs &a, const Node1 &k, uint32_t s, uint32_t e, int lane,
                                        uint2 *rect, int32_t *rec, F step) {
    const uint32_t x0 = 64 * (uint32_t)k.hx, y0 = 64 * (uint32_t)k.hy;
    constexpr int AHEAD = 4;  // groups whose loads are in flight together
    uint32_t n = 0;
    for (uint32_t b0 = s; b0 < e; b0 += 64 * AHEAD) {
        uint2 r[AHEAD];
        int32_t g[AHEAD];
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
            const uint32_t j = b0 + 64 * q + (uint32_t)lane;
            r[q] = make_uint2(0u, 0u);  // an empty rectangle: no hit
            g[q] = 0;
            if (j < e) {
                r[q] = a.lrect[j];
                if (IDS) g[q] = a.list[j];
            }
        }
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
            const bool hit = (r[q].x & 0xFFFF) < x0 + 64 && (r[q].x >> 16) > x0 && (r[q].y & 0xFFFF) < y0 + 64 &&
                             (r[q].y >> 16) > y0;
            const uint64_t m = __ballot(hit);
            if (m == 0) continue;
            if (hit) {
                const uint32_t p = n + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                rect[p] = r[q];
                if (IDS) rec[p] = g[q];
            }
            n += (uint32_t)__popcll(m);
            wave_sync();
            if (n < 64) continue;
            step(64u);
            n -= 64;
            wave_sync();
            uint2 tr = make_uint2(0u, 0u);
            int32_t tg = 0;
            if ((uint32_t)lane < n) {
                tr = rect[64 + lane];
                if (IDS) tg = rec[64 + lane];
            }
            wave_sync();
            if ((uint32_t)lane < n) {
                rect[lane] = tr;
                if (IDS) rec[lane] = tg;
            }
            wave_sync();
        }
    }
    if (n) step(n);
    wave_sync();
}

// ── counts ───────────────────────────────────────────────────────────────────
// A unit's counts: each wave's exclusive prefix over the unit's waves goes to
// wave_cnt[(u WAVES + w) 64 + c], the unit's totals to cnt[64 u + c]. sums is LDS scratch.
template <uint32_t WAVES>
__device__ inline void unit_prefix(uint32_t u, uint32_t n, uint32_t *cnt, uint32_t *wave_cnt, uint32_t (*sums)[64]) {
    const int lane = threadIdx.x & 63;
    const uint32_t w = threadIdx.x >> 6;
    sums[w][lane] = n;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t k = 0; k < WAVES; k++) {
        const uint32_t t = sums[k][lane];
        before += k < w ? t : 0u;
        total += t;
    }
    wave_cnt[((size_t)u * WAVES + w) * 64 + lane] = before;
    if (w == 0) cnt[(size_t)u * 64 + lane] = total;
    __syncthreads();  // sums is written again for the next unit
}

template <bool BATCH>
__global__ __launch_bounds__(64 * WAVES1) void list_count1_kernel(TileListArgs a) {
    __shared__ uint2 s_rect[WAVES1][128];
    __shared__ uint32_t sums[WAVES1][64];
    const int lane = threadIdx.x & 63;
    const uint32_t w = threadIdx.x >> 6;
    const BitTranspose tr(lane);
    const uint32_t units = level1_units<BATCH>(a), nodes = level1_nodes<BATCH>(a);
    for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
        const uint32_t i = BATCH ? find_start(a.unit1, nodes, u, lane) : u / (units / nodes);
        const Node1 k = level1_node<BATCH>(a, i);
        const uint32_t s = min(k.s + ((u - k.first_unit) * WAVES1 + w) * 64 * k.groups, k.e);
        const uint32_t e = min(s + 64 * k.groups, k.e);
        uint32_t n = 0;
        uint2 *rect = s_rect[w];
        touching_records<false>(a, k, s, e, lane, rect, nullptr, [&](uint32_t m) {
            uint32_t lo = 0, hi = 0;
            if ((uint32_t)lane < m) super_mask(rect[lane], k.hx, k.hy, lo, hi);
            tr(lo, hi);
            n += (uint32_t)(__popc(lo) + __popc(hi));
        });
        unit_prefix<WAVES1>(u, n, a.cnt1, a.wave1, sums);
    }
}

template <bool BATCH>
__global__ __launch_bounds__(64 * WAVES2) void list_count2_kernel(TileListArgs a) {
    __shared__ uint32_t sums[WAVES2][64];
    const int lane = threadIdx.x & 63;
    const uint32_t w = threadIdx.x >> 6;
    const BitTranspose tr(lane);
    const uint32_t units = level2_units<BATCH>(a), nodes = level2_nodes<BATCH>(a);
    const uint2 *entries = a.direct ? a.lrect : a.coarse;
    for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
        const uint32_t i = a.direct ? 0u : find_start(a.unit2, nodes, u, lane);
        const Node2 k = level2_node(a, i);
        const uint32_t s = min(k.s + ((u - k.first_unit) * WAVES2 + w) * 64 * k.groups, k.e);
        const uint32_t e = min(s + 64 * k.groups, k.e);
        uint32_t n = 0, next = s + lane < e ? entries[s + lane].y : 0u;
        for (uint32_t b = s; b < e; b += 64) {
            const uint32_t c = next;  // an empty rectangle past the end
            next = b + 64 + lane < e ? entries[b + 64 + lane].y : 0u;
            uint32_t lo, hi;
            local_mask(c, lo, hi);
            tr(lo, hi);
            n += (uint32_t)(__popc(lo) + __popc(hi));
        }
        unit_prefix<WAVES2>(u, n, a.cnt2, a.wave2, sums);
    }
}

// ── prefix over a node's units ───────────────────────────────────────────────
// One workgroup per node: each wave sums its part of the node's rows of 64 counts, the
// waves' sums are prefixed in LDS, and each wave replaces its rows by the exclusive
// prefix. Eight rows' loads are in flight at a time. Returns lane c's total (wave 0).
template <int NW>
__device__ inline uint32_t prefix_rows(uint32_t *cnt, uint32_t r0, uint32_t r1, uint32_t (*sums)[64]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t per = (r1 - r0 + NW - 1) / NW;
    const uint32_t b = min(r0 + (uint32_t)w * per, r1), e = min(b + per, r1);
    uint32_t s = 0;
    for (uint32_t r = b; r < e; r += 8) {
        uint32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = r + k < e ? cnt[(size_t)(r + k) * 64 + lane] : 0u;
#pragma unroll
        for (int k = 0; k < 8; k++) s += v[k];
    }
    sums[w][lane] = s;
    __syncthreads();
    uint32_t run = 0, total = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const uint32_t t = sums[k][lane];
        run += k < w ? t : 0u;
        total += t;
    }
    __syncthreads();  // sums is written again for the next node
    for (uint32_t r = b; r < e; r += 8) {
        uint32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = r + k < e ? cnt[(size_t)(r + k) * 64 + lane] : 0u;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (r + k < e) cnt[(size_t)(r + k) * 64 + lane] = run;
            run += v[k];
        }
    }
    return total;
}

constexpr int PREFIX_WAVES = 16;

template <bool BATCH>
__global__ __launch_bounds__(64 * PREFIX_WAVES) void list_prefix1_kernel(TileListArgs a) {
    __shared__ uint32_t sums[PREFIX_WAVES][64];
    const uint32_t nodes = level1_nodes<BATCH>(a);
    for (uint32_t i = blockIdx.x; i < nodes; i += gridDim.x) {
        const Node1 k = level1_node<BATCH>(a, i);
        const uint32_t units = unit_count<WAVES1>(k.e - k.s, k.groups);
        const uint32_t t = prefix_rows<PREFIX_WAVES>(a.cnt1, k.first_unit, k.first_unit + units, sums);
        if (threadIdx.x < 64) a.super_total[64 * i + threadIdx.x] = t;
    }
}

template <bool BATCH>
__global__ __launch_bounds__(1024) void list_plan2_kernel(TileListArgs a) {
    __shared__ uint32_t lds16[16];
    plan2<BATCH>(a, lds16);
}

// Both for a view of few nodes, in one workgroup: 7.7 us for 9.5 at one and two nodes, but
// 11.6 for 9.4 at four.
constexpr uint32_t FEW_NODES = 2;
static_assert(64 * PREFIX_WAVES == 1024, "one workgroup shape");
__global__ __launch_bounds__(1024) void list_prefix1_plan2_kernel(TileListArgs a) {
    __shared__ uint32_t sums[PREFIX_WAVES][64];
    __shared__ uint32_t lds16[16];
    for (uint32_t i = 0; i < (uint32_t)a.nodes; i++) {
        const Node1 k = level1_node<false>(a, i);
        const uint32_t units = unit_count<WAVES1>(k.e - k.s, k.groups);
        const uint32_t t = prefix_rows<PREFIX_WAVES>(a.cnt1, k.first_unit, k.first_unit + units, sums);
        if (threadIdx.x < 64) a.super_total[64 * i + threadIdx.x] = t;
    }
    __syncthreads();  // the totals, which other threads of the workgroup read
    plan2<false>(a, lds16);
}

// Level 2: a tile's total goes to tile_start[tile], to be scanned in tile order
template <bool BATCH>
__global__ __launch_bounds__(64 * PREFIX_WAVES) void list_prefix2_kernel(TileListArgs a) {
    __shared__ uint32_t sums[PREFIX_WAVES][64];
    const uint32_t nodes = level2_nodes<BATCH>(a);
    for (uint32_t i = blockIdx.x; i < nodes; i += gridDim.x) {
        const Node2 k = level2_node(a, i);
        const uint32_t units = unit_count<WAVES2>(k.e - k.s, k.groups);
        const uint32_t t = prefix_rows<PREFIX_WAVES>(a.cnt2, k.first_unit, k.first_unit + units, sums);
        if (threadIdx.x < 64) {
            const int tile = tile_of<BATCH>(a, i, (int)threadIdx.x);
            if (tile >= 0) a.tile_start[tile] = (int32_t)t;
        }
    }
}

// ── expansion ────────────────────────────────────────────────────────────────
// Level 1 writes few entries (about two supertiles per record): each lane stores those of
// its supertile as it finds them, two per round so that their LDS reads overlap.
template <bool BATCH>
__global__ __launch_bounds__(64 * WAVES1) void list_expand1_kernel(TileListArgs a) {
    __shared__ uint2 s_rect[WAVES1][128];
    __shared__ int32_t s_rec[WAVES1][128];
    const int lane = threadIdx.x & 63;
    const uint32_t w = threadIdx.x >> 6;
    const BitTranspose tr(lane);
    const uint32_t units = level1_units<BATCH>(a), nodes = level1_nodes<BATCH>(a);
    for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
        const uint32_t i = BATCH ? find_start(a.unit1, nodes, u, lane) : u / (units / nodes);
        const Node1 k = level1_node<BATCH>(a, i);
        const uint32_t s = min(k.s + ((u - k.first_unit) * WAVES1 + w) * 64 * k.groups, k.e);
        const uint32_t e = min(s + 64 * k.groups, k.e);
        if (s >= e) continue;  // no workgroup barrier below
        uint32_t pos = a.super_start[64 * i + lane] + a.cnt1[(size_t)u * 64 + lane] +
                       a.wave1[((size_t)u * WAVES1 + w) * 64 + lane];
        const int ox = 64 * k.hx + 8 * (lane & 7), oy = 64 * k.hy + 8 * (lane >> 3);  // the lane's supertile, in tiles
        uint2 *rect = s_rect[w];
        int32_t *rec = s_rec[w];
        auto emit = [&](uint32_t m, uint32_t base) {
            while (__any(m != 0)) {
                const bool h0 = m != 0;
                const uint32_t j0 = base + (h0 ? (uint32_t)__builtin_ctz(m) : 0u);
                m &= m - 1u;
                const bool h1 = m != 0;
                const uint32_t j1 = base + (h1 ? (uint32_t)__builtin_ctz(m) : 0u);
                m &= m - 1u;
                const uint2 r0 = rect[j0], r1 = rect[j1];
                const int32_t g0 = rec[j0], g1 = rec[j1];
                if (h0) a.coarse[pos] = make_uint2((uint32_t)g0, pack_local(r0, ox, oy));
                if (h1) a.coarse[pos + 1] = make_uint2((uint32_t)g1, pack_local(r1, ox, oy));
                pos += (h0 ? 1u : 0u) + (h1 ? 1u : 0u);
            }
        };
        touching_records<true>(a, k, s, e, lane, rect, rec, [&](uint32_t m) {
            uint32_t lo = 0, hi = 0;
            if ((uint32_t)lane < m) super_mask(rect[lane], k.hx, k.hy, lo, hi);
            tr(lo, hi);
            emit(lo, 0);
            emit(hi, 32);
        });
    }
}

// Level 2 writes every intersection. Stored by the lane that owns the tile, each would be
// a request of its own to L2 (64 lists, a word each, per store instruction). So here lane r
// keeps its record and the wave goes through the 64 tiles: a ballot of the mask bit gives
// the records of a tile, whose lanes store them side by side.
template <bool BATCH>
__global__ __launch_bounds__(64 * WAVES2) void list_expand2_kernel(TileListArgs a) {
    const int lane = threadIdx.x & 63;
    const uint32_t w = threadIdx.x >> 6;
    const BitTranspose tr(lane);
    const uint32_t units = level2_units<BATCH>(a), nodes = level2_nodes<BATCH>(a);
    const uint2 *entries = a.direct ? a.lrect : a.coarse;
    for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
        const uint32_t i = a.direct ? 0u : find_start(a.unit2, nodes, u, lane);
        const Node2 k = level2_node(a, i);
        const uint32_t s = min(k.s + ((u - k.first_unit) * WAVES2 + w) * 64 * k.groups, k.e);
        const uint32_t e = min(s + 64 * k.groups, k.e);
        if (s >= e) continue;  // no workgroup barrier below
        const int tile = tile_of<BATCH>(a, i, lane);
        // lane t: the next place in tile t's list
        uint32_t pos = (tile >= 0 ? (uint32_t)a.tile_start[tile] : 0u) + a.cnt2[(size_t)u * 64 + lane] +
                       a.wave2[((size_t)u * WAVES2 + w) * 64 + lane];
        uint2 next = s + lane < e ? entries[s + lane] : make_uint2(0u, 0u);
        for (uint32_t b = s; b < e; b += 64) {
            const uint2 c = next;  // an empty rectangle past the end
            if (b + 64 + lane < e) next = entries[b + 64 + lane];
            else next = make_uint2(0u, 0u);
            uint32_t half[2];
            local_mask(c.y, half[0], half[1]);
            uint32_t lo = half[0], hi = half[1];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint32_t bits = half[h];
                for (int t0 = 0; t0 < 32; t0 += 8, bits >>= 8) {  // a row of tiles at a time
                    if (__ballot((bits & 0xFFu) != 0) == 0) continue;
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        const bool in = (bits & (1u << q)) != 0;
                        const uint64_t m = __builtin_amdgcn_ballot_w64(in);
                        if (m == 0) continue;
                        const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)pos, 32 * h + t0 + q);
                        if (in)
                            a.gids[p + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = (int32_t)c.x;
                    }
                }
            }
            tr(lo, hi);
            pos += (uint32_t)(__popc(lo) + __popc(hi));
        }
    }
}

// The 64-bit (tile << 32 | depth bits) view of the m listed intersections, one workgroup per tile
__global__ __launch_bounds__(256) void list_keys64_kernel(const int32_t *tile_start, int m, const int32_t *gid,
                                                         const float *depths, uint64_t *out) {
    const uint32_t t = blockIdx.x;
    const int e = min(tile_start[t + 1], m);
    for (int k = tile_start[t] + (int)threadIdx.x; k < e; k += 256)
        out[k] = ((uint64_t)t << 32) | (uint64_t)__float_as_uint(depths[gid[k]]);
}

// ── host ─────────────────────────────────────────────────────────────────────

uint32_t tile_list_nodes(int tiles_x, int tiles_y) {
    return (uint32_t)((tiles_x + 63) / 64) * (uint32_t)((tiles_y + 63) / 64);
}

bool tile_list_direct(int tiles_x, int tiles_y) { return tiles_x <= 8 && tiles_y <= 8; }

size_t tile_list_scratch_words(uint32_t nodes) {
    const size_t n1 = nodes, n2 = 64 * (size_t)nodes;
    return 64 * (WAVES1 + 1) * (UNITS1 + n1) + 64 * (WAVES2 + 1) * (UNITS2 + n2) + (n1 + 1) + n2 + (n2 + 1) + (n2 + 1) + 2;
}

void tile_list_carve(uint32_t *p, uint32_t nodes, TileListArgs &a) {
    const size_t n1 = nodes, n2 = 64 * (size_t)nodes;
    a.cnt1 = p;
    a.wave1 = a.cnt1 + 64 * (UNITS1 + n1);
    a.cnt2 = a.wave1 + 64 * WAVES1 * (UNITS1 + n1);
    a.wave2 = a.cnt2 + 64 * (UNITS2 + n2);
    a.unit1 = a.wave2 + 64 * WAVES2 * (UNITS2 + n2);
    a.super_total = a.unit1 + (n1 + 1);
    a.super_start = a.super_total + n2;
    a.unit2 = a.super_start + (n2 + 1);
    a.plan = a.unit2 + (n2 + 1);
}

// Launch bounds (the kernels loop over their units): a wave takes at least 64 entries, so
// there are at most entries / (64 WAVES) units besides a partly filled one per node, and
// never more than LIST_WAVES / WAVES besides those.
template <uint32_t WAVES>
static uint32_t unit_blocks(uint64_t entries, uint32_t nodes) {
    const uint64_t units = entries / (64 * WAVES) + nodes;
    return (uint32_t)std::min<uint64_t>(units, LIST_WAVES / WAVES);
}

template <bool BATCH>
static void lists_begin(const TileListArgs &a, uint32_t nodes, uint32_t nvis_max, hipStream_t s) {
    if (a.direct) return;
    if (BATCH) list_plan1_kernel<<<1, 1024, 0, s>>>(a);
    list_count1_kernel<BATCH><<<unit_blocks<WAVES1>((uint64_t)nodes * nvis_max, nodes), 64 * WAVES1, 0, s>>>(a);
    if (!BATCH && nodes <= FEW_NODES) {
        list_prefix1_plan2_kernel<<<1, 1024, 0, s>>>(a);
        return;
    }
    list_prefix1_kernel<BATCH><<<nodes < 1024 ? nodes : 1024, 64 * PREFIX_WAVES, 0, s>>>(a);
    list_plan2_kernel<BATCH><<<1, 1024, 0, s>>>(a);
}

template <bool BATCH>
static void lists_end(const TileListArgs &a, uint32_t nodes, uint32_t nvis_max, uint32_t m_max, uint32_t ntiles,
                      uint32_t *partial, hipStream_t s) {
    const uint32_t n2 = a.direct ? 1 : 64 * nodes;
    const uint32_t g2 = unit_blocks<WAVES2>(a.direct ? nvis_max : m_max, n2);
    if (!a.direct)
        list_expand1_kernel<BATCH><<<unit_blocks<WAVES1>((uint64_t)nodes * nvis_max, nodes), 64 * WAVES1, 0, s>>>(a);
    list_count2_kernel<BATCH><<<g2, 64 * WAVES2, 0, s>>>(a);
    list_prefix2_kernel<BATCH><<<n2 < 2048 ? n2 : 2048, 64 * PREFIX_WAVES, 0, s>>>(a);
    launch_scan_u32((uint32_t *)a.tile_start, ntiles + 1, partial,
                    ScanOut{nullptr, nullptr, 0xFFFFFFFFu, nullptr, nullptr, nullptr, nullptr}, s);
    list_expand2_kernel<BATCH><<<g2, 64 * WAVES2, 0, s>>>(a);
}

void launch_tile_lists_begin(const TileListArgs &a, bool batch, uint32_t nodes, uint32_t nvis_max, hipStream_t s) {
    if (batch) lists_begin<true>(a, nodes, nvis_max, s);
    else lists_begin<false>(a, nodes, nvis_max, s);
}

void launch_tile_lists_end(const TileListArgs &a, bool batch, uint32_t nodes, uint32_t nvis_max, uint32_t m_max,
                           uint32_t ntiles, uint32_t *partial, hipStream_t s) {
    if (batch) lists_end<true>(a, nodes, nvis_max, m_max, ntiles, partial, s);
    else lists_end<false>(a, nodes, nvis_max, m_max, ntiles, partial, s);
}

void launch_list_keys64(const int32_t *tile_start, int ntiles, int m, const int32_t *gid, const float *depths, uint64_t *out,
                        hipStream_t s) {
    if (ntiles > 0) list_keys64_kernel<<<ntiles, 256, 0, s>>>(tile_start, m, gid, depths, out);
}

}  // namespace msplat
