// npa_draw.hip - isotropic Gaussian footprints into 16x16 pixel tiles on the matrix cores (gfx950):
// splat_particles_2d (crates/burn_automata_kernels/src/splat.rs:30-93) and splat_projected
// (crates/burn_automata/src/render_loss/image.rs:18-79) after their particles' preparation.
//
// A weight exp(-(dx^2 + dy^2) / 2 sigma^2) is the product of its column's and its row's, so a tile's
// channel is a matrix product over its items: image_c[y][x] = sum_p (c_p scale_p e_p(y)) e_p(x). A wave
// takes four items at a time: lane l serves item l / 16, evaluates e(x) of column l % 16 and e(y) of row
// l % 16 (zero outside the item's footprint), and v_mfma_f32_16x16x4_f32 adds the four items to all 256
// pixels, one instruction per channel: two exponentials per item and lane in place of one per pixel, and
// no vector instruction per pixel at all.
//
// No sort either: a block covers a group of G x G tiles; its waves test the packed tile rectangles of
// their shares of the window's items and keep the indices of those that touch the group, in ascending
// order; then they draw the group's tiles from the kept items (several waves per tile for small groups,
// their sums added in a fixed order). The items of crowded groups are divided among further blocks, by a sample
// of the items alone. So items are added in a fixed order and the image is deterministic; it differs from the
// reference's running sums only by rounding.
//
// Bound: the matrix instructions, 32 cycles per channel and four items (160 cycles for five channels), and
// the tests, about twelve instructions per 64 items and group. Against the former passes (items sorted by
// tile, a wave evaluating every pixel's exponential): four 64x64 views of 16,384 particles 161 -> 45 us with
// their preparation, a 512x512 splat of 65,536 89 -> 28 us, a 160x160 view of 4,000 102 -> 35 us, 300,000
// at 2048x2048 1,094 -> 405 us, 500,000 at 4096x4096 8.5 -> 1.7 ms, and on a part of the image 300,000 at 2048x2048
// 1,519 -> 433 us, four 512x512 views of 100,000 790 -> 608 us. At most a sixth slower where all items lie on a few
// pixels of a large image (20,000 on a fiftieth of four 512x512 views 255 -> 288 us); the sorted passes are gone.
#include "npa_draw.hpp"

#include <algorithm>

namespace npa {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr uint32_t kDrawPer = 8;      // rectangles a lane tests per step, the next ones' loads in flight
constexpr uint32_t kDrawSeg = 768;    // kept items a wave holds before the block draws
constexpr uint32_t kDrawQueue = 72;   // a wave's queue: 64 new entries after up to 7

// An item's tiles against a group's: every byte of the item's word (see draw_rect) at most the group's.
__device__ __forceinline__ uint32_t rect_limit(uint32_t gx0, uint32_t gx1, uint32_t gy0, uint32_t gy1) {
    return draw_rect(gx1, gx0, gy1, gy0) | 0x80808080u;
}
__device__ __forceinline__ bool rect_touches(uint32_t r, uint32_t limit) {
    return (~(limit - r) & 0x80808080u) == 0u;  // no byte borrows from its guard bit
}

// The pixels this lane accumulates: column l % 16, rows 4 (l / 16) + r.
template <int NCH>
struct DrawTile {
    v4f acc[NCH];
    int x, y;        // this lane's column, and the row it evaluates weights for
    int yp;          // this lane's first accumulated row
    float xf, yf;

    __device__ __forceinline__ void init(uint32_t tx, uint32_t ty, uint32_t lane) {
        x = (int)(tx * 16 + lane % 16);
        y = (int)(ty * 16 + lane % 16);
        yp = (int)(ty * 16 + 4 * (lane / 16));
        xf = (float)x;
        yf = (float)y;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) acc[ch] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // Adds four items, one per 16 lanes; ALL: every lane's item is live, else the others add nothing.
    template <bool ALL>
    __device__ __forceinline__ void add(const float4& a, const float4& b, const uint4& w, bool live) {
        const float dx = xf - a.x, dy = yf - a.y;
        float ex = __builtin_amdgcn_exp2f(-(dx * dx) * a.z);
        float ey = __builtin_amdgcn_exp2f(-(dy * dy) * a.z) * a.w;
        ex = (uint32_t)x - w.x <= w.z && (ALL || live) ? ex : 0.0f;
        ey = (uint32_t)y - w.y <= w.z && (ALL || live) ? ey : 0.0f;
        float c[5] = {b.x, b.y, b.z, 1.0f, b.w};
        const uint64_t odd = __ballot((ALL || live) && w.w != 0u);
        if (odd) {  // rare
            add_special(a, b, w, odd);
            if (w.w != 0u) ex = ey = 0.0f;
        }
        if (odd || !ALL) {  // nothing but zeros from a special item, or from what an idle lane has loaded
#pragma unroll
            for (int ch = 0; ch < 5; ++ch) c[ch] = w.w == 0u && (ALL || live) ? c[ch] : 0.0f;
        }
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch)
            acc[ch] = __builtin_amdgcn_mfma_f32_16x16x4f32(ch == 3 ? ey : ey * c[ch], ex, acc[ch], 0, 0, 0);
    }
    // Items with a value that is not finite touch only the pixels of their footprint.
    __device__ __forceinline__ void add_special(const float4& a, const float4& b, const uint4& w, uint64_t odd) {
        for (uint32_t k = 0; k < 4; ++k) {
            if (!((odd >> (16 * k)) & 1ull)) continue;
            auto of = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16 * k)); };
            auto ofu = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 16 * k); };
            const float px = of(a.x), py = of(a.y), k2 = of(a.z), scale = of(a.w);
            const float c[5] = {of(b.x), of(b.y), of(b.z), 1.0f, of(b.w)};
            const int x0 = (int)ofu(w.x), y0 = (int)ofu(w.y);
            const uint32_t span = ofu(w.z);
            for (int r = 0; r < 4; ++r) {
                if ((uint32_t)(x - x0) > span || (uint32_t)(yp + r - y0) > span) continue;
                const float dx = xf - px, dy = (float)(yp + r) - py;
                const float v = __builtin_amdgcn_exp2f(-(dx * dx + dy * dy) * k2) * scale;
#pragma unroll
                for (int ch = 0; ch < NCH; ++ch) acc[ch][r] += ch == 3 ? v : c[ch] * v;
            }
        }
    }
};

// Which items a block draws: range `range` of `ranges` of the items of group `blk`'s window; the second range's
// partial tiles are at `slot` and so on.
struct DrawShare {
    uint32_t blk, range, ranges, slot;
};

// Grid: single tiles (G = 1): x = window * groups_x^2 + group, y = split of the window's items. Groups: the first
// P.groups blocks take one each, the others the further ranges of crowded groups (draw_crowd's jobs), and the
// block that finishes such a group last adds up its ranges, in order.
// NW waves per block: sixteen for groups of tiles, whose waves share the tests of every item of the window;
// four for single tiles, whose blocks are short and hide each other's latencies (four of them per CU).
template <int NCH, int G, int NW>
__global__ __launch_bounds__(NW * 64, 4) void k_draw_tiles(DrawPlan P, const float4* __restrict__ items,
                                                        const uint32_t* __restrict__ rects,
                                                        float* partials, uint32_t* crowd, float* image) {
    constexpr uint32_t TILES = G * G, WPT = NW / TILES;  // tiles per block, waves per tile
    constexpr uint32_t NR = NCH * 4;                             // accumulated values per lane
    // the waves' kept items (rectangle, index), then their queues; the sums of the waves at the end
    constexpr uint32_t LIST = NW * kDrawSeg * 2, QUEUE = NW * kDrawQueue, SUMS = NW * NR * 64;
    __shared__ uint32_t lds[LIST + QUEUE > SUMS ? LIST + QUEUE : SUMS];
    __shared__ uint32_t counts[NW], unfinished, last_ticket;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t per_win = P.groups_x * P.groups_x;
    DrawShare share;
    uint32_t crowded = 0;
    if constexpr (G == 1) {
        // the ranges of one crowded tile go to different CUs: each range's blocks start at another tile (a CU
        // gets about every 256th block)
        share.blk = (uint32_t)((blockIdx.x + (uint64_t)blockIdx.y * (gridDim.x * 5 / 8 | 1u) + blockIdx.y / 4) % gridDim.x);
        share.range = blockIdx.y;
        share.ranges = P.splits;
        share.slot = 0;
    } else {
        share = {blockIdx.x, 0u, 1u, 0u};
        if (P.extra) {
            if (blockIdx.x >= P.groups) {
                const uint32_t job = blockIdx.x - P.groups;
                if (job >= crowd[kCrowdJobs]) return;  // whole block
                const uint32_t j = crowd[kCrowdJobs + 1 + job];
                share.blk = j & 0xffffu;
                share.range = j >> 16;
            }
            crowded = crowd[kCrowdGroups + share.blk];
        }
    }
    const uint32_t blk = share.blk;
    const uint32_t win = blk / per_win, grp = blk - win * per_win;
    const uint32_t gx0 = grp % P.groups_x * G, gy0 = grp / P.groups_x * G;
    const uint32_t tg = wave % TILES, part = wave / TILES;
    const uint32_t tx = gx0 + tg % G, ty = gy0 + tg / G;
    const uint32_t sh = P.rect_shift;
    const uint32_t glim = rect_limit(gx0 >> sh, (gx0 + G - 1) >> sh, gy0 >> sh, (gy0 + G - 1) >> sh);
    const uint32_t tlim = rect_limit(tx >> sh, tx >> sh, ty >> sh, ty >> sh);
    DrawTile<NCH> tile;
    tile.init(tx, ty, lane);
    uint2* list = reinterpret_cast<uint2*>(lds);
    uint32_t* queue = lds + LIST + wave * kDrawQueue;
    // this block's items, and this wave's share of the tests
    const uint64_t win_beg = (uint64_t)win * P.per_window;
    const uint64_t win_end = win_beg + P.per_window < P.count ? win_beg + P.per_window : P.count;
    const uint32_t n = win_end > win_beg ? (uint32_t)(win_end - win_beg) : 0u;
    uint32_t pos, end;
    auto take_share = [&] {
        const uint32_t part_n = (n + share.ranges - 1) / share.ranges;
        const uint32_t first = min(n, share.range * part_n), last = min(n, first + part_n);
        const uint32_t mine = (last - first + NW - 1) / NW;
        pos = min(last, first + wave * mine);
        end = min(last, pos + mine);
    };
    take_share();
    const uint32_t* rw = rects + win_beg;
    uint32_t r[kDrawPer];
    auto fetch = [&](uint32_t at) {
#pragma unroll
        for (uint32_t i = 0; i < kDrawPer; ++i) {
            const uint32_t k = at + i * 64 + lane;
            r[i] = k < end ? rw[k] : kDrawNone;
        }
    };
    fetch(pos);
    if (crowded & 0xffu) {  // known by now: few groups are, and start again with their range
        share.ranges = (crowded & 0xffu) + 1;
        share.slot = crowded >> 8;
        take_share();
        fetch(pos);
    }
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // Eight entries of the queue at a time; their loads are issued before the eight entries before them
    // are drawn.
    struct Eight {
        float4 a[2], b[2];
        uint4 w[2];
    } E0, E1;
    uint32_t waiting = 0;  // entries in this wave's queue
    bool ahead = false;    // E0 holds eight entries not drawn yet
    float warm = 0.0f;
    auto load = [&](uint32_t at, uint32_t count, Eight& e) {
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t k = 4 * h + lane / 16;
            const float4* it = items + (uint64_t)queue[at + (k < count ? k : 0u)] * 3;
            e.a[h] = it[0];
            e.b[h] = it[1];
            e.w[h] = reinterpret_cast<const uint4*>(it)[2];
        }
    };
    auto draw = [&](const Eight& e) {
        tile.template add<true>(e.a[0], e.b[0], e.w[0], true);
        tile.template add<true>(e.a[1], e.b[1], e.w[1], true);
    };

    for (;;) {
        // each wave tests its items in turn and keeps those that touch the group
        uint32_t kept = 0;
        if (threadIdx.x == 0) unfinished = 0;
        while (pos < end && kept + kDrawPer * 64 <= kDrawSeg) {
            uint32_t c[kDrawPer];
#pragma unroll
            for (uint32_t i = 0; i < kDrawPer; ++i) c[i] = r[i];
            fetch(pos + kDrawPer * 64);
#pragma unroll
            for (uint32_t i = 0; i < kDrawPer; ++i) {
                const bool hit = rect_touches(c[i], glim);
                const uint64_t m = __ballot(hit);
                if (!m) continue;  // wave-uniform
                if (hit)
                    list[wave * kDrawSeg + kept + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] =
                        make_uint2(c[i], pos + i * 64 + lane);
                kept += (uint32_t)__popcll(m);
            }
            pos += kDrawPer * 64;
        }
        __syncthreads();  // `unfinished` is cleared
        if (lane == 0) {
            counts[wave] = kept;
            if (pos < end) unfinished = 1;
        }
        __syncthreads();
        const bool more = unfinished != 0;
        // the kept items as one list, ascending: entry e is the (e - before[s])-th of wave s
        const uint32_t cw = lane < NW ? counts[lane] : 0u;
        const uint32_t incl = row_incl_add(cw);
        uint32_t before[NW + 1];
        before[0] = 0;
#pragma unroll
        for (uint32_t s = 0; s < NW; ++s) before[s + 1] = (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)s);
        const uint32_t total = before[NW];
        // a tile's waves take equal consecutive ranges of it
        const uint32_t range = (total + WPT - 1) / WPT;
        const uint32_t k_end = min(total, (part + 1) * range);
        for (uint32_t k0 = part * range; k0 < k_end; k0 += 64) {
            const uint32_t e = k0 + lane;
            uint32_t at = e;
#pragma unroll
            for (uint32_t s = 1; s < NW; ++s) at = e >= before[s] ? s * kDrawSeg + e - before[s] : at;
            const uint2 it = e < k_end ? list[at] : make_uint2(kDrawNone, 0u);
            const bool hit = G == 1 && sh == 0 ? e < k_end : rect_touches(it.x, tlim);
            const uint64_t m = __ballot(hit);
            // One word of every item kept, in flight while the entries before it are drawn: the items come from
            // the last cache level, at about a microsecond for every eight that a wave draws, and then from L2.
            // (Single tiles' ranges are short.)
            if constexpr (G > 1) asm volatile("" ::"v"(warm));
            if (hit) {
                const uint32_t at_item = (uint32_t)win_beg + it.y;
                queue[waiting + (uint32_t)__popcll(m & lanemask_lt())] = at_item;
                if constexpr (G > 1) warm = items[(uint64_t)at_item * 3].x;
            }
            waiting += (uint32_t)__popcll(m);
            wave_fence();
            uint32_t q = 0;
            if (!ahead && waiting >= 8) {
                load(0, 8, E0);
                q = 8;
                ahead = true;
            }
            for (; waiting - q >= 16; q += 16) {
                load(q, 8, E1);
                draw(E0);
                load(q + 8, 8, E0);
                draw(E1);
            }
            if (waiting - q >= 8) {
                load(q, 8, E1);
                draw(E0);
                E0 = E1;
                q += 8;
            }
            const uint32_t rest = waiting - q;  // up to seven wait for the next entries
            const uint32_t keep = lane < rest ? queue[q + lane] : 0u;
            wave_fence();
            if (lane < rest) queue[lane] = keep;
            waiting = rest;
            wave_fence();
        }
        if (!more) break;
        __syncthreads();  // the list and the counts are read before they are filled again
        fetch(pos);
    }
    if (ahead) draw(E0);
    if (waiting) {
        load(0, waiting, E0);
        tile.template add<false>(E0.a[0], E0.b[0], E0.w[0], lane / 16 < waiting);
        tile.template add<false>(E0.a[1], E0.b[1], E0.w[1], 4 + lane / 16 < waiting);
    }
    __syncthreads();
    float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch)
#pragma unroll
        for (int q = 0; q < 4; ++q) sums[(wave * NR + ch * 4 + q) * 64 + lane] = tile.acc[ch][q];
    __syncthreads();
    auto out = [&](uint32_t x, uint32_t y) {
        if constexpr (NCH == 4)
            return image + (((uint64_t)(win / P.win_cols) * P.size + y) * P.stride + (uint64_t)(win % P.win_cols) * P.size + x) * 4;
        else
            return image + (((uint64_t)win * P.size + y) * P.size + x) * NCH;
    };
    auto put = [&](float* o, const float (&v)[NCH]) {
        if constexpr (NCH == 4) {
            *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) o[ch] = v[ch];
        }
    };
    for (uint32_t t = threadIdx.x; t < TILES * 256; t += NW * 64) {
        const uint32_t tl = t / 256, row = t % 256 / 16, col = t % 16;
        const uint32_t x = (gx0 + tl % G) * 16 + col, y = (gy0 + tl / G) * 16 + row;
        if (x >= (uint32_t)P.size || y >= (uint32_t)P.size) continue;
        float v[NCH];
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            v[ch] = 0.0f;
            for (uint32_t p = 0; p < WPT; ++p)
                v[ch] += sums[((p * TILES + tl) * NR + ch * 4 + row % 4) * 64 + row / 4 * 16 + col];
        }
        if (G == 1 && P.splits > 1) {
            const uint64_t pixel = ((uint64_t)win * P.size + y) * P.size + x, all = (uint64_t)P.windows * P.size * P.size;
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) partials[((uint64_t)blockIdx.y * NCH + ch) * all + pixel] = v[ch];
        } else if (G > 1 && share.range > 0) {
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) partials[((uint64_t)(blockIdx.x - P.groups) * NCH + ch) * (TILES * 256) + t] = v[ch];
        } else {
            put(out(x, y), v);
        }
    }
    if constexpr (G > 1) {
        if (share.ranges == 1) return;
        // the last of the group's blocks adds the ranges up: the first in the image, the others from their slots
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        if (threadIdx.x == 0) last_ticket = __hip_atomic_fetch_add(&crowd[blk], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (last_ticket != share.ranges - 1) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (threadIdx.x == 0) crowd[blk] = 0;  // for the next drawing
        for (uint32_t t = threadIdx.x; t < TILES * 256; t += NW * 64) {
            const uint32_t tl = t / 256, row = t % 256 / 16, col = t % 16;
            const uint32_t x = (gx0 + tl % G) * 16 + col, y = (gy0 + tl / G) * 16 + row;
            if (x >= (uint32_t)P.size || y >= (uint32_t)P.size) continue;
            float* o = out(x, y);
            const float* slot = partials + (uint64_t)share.slot * NCH * (TILES * 256) + t;
            float v[NCH];
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) v[ch] = o[ch];
            for (uint32_t s = 1; s < share.ranges; s += 8) {  // eight ranges' loads at a time
                float w[8][NCH];
#pragma unroll
                for (uint32_t u = 0; u < 8; ++u, slot += NCH * (TILES * 256))
#pragma unroll
                    for (int ch = 0; ch < NCH; ++ch) w[u][ch] = s + u < share.ranges ? slot[ch * (TILES * 256)] : 0.0f;
#pragma unroll
                for (uint32_t u = 0; u < 8; ++u)
#pragma unroll
                    for (int ch = 0; ch < NCH; ++ch) v[ch] += w[u][ch];
            }
            put(o, v);
        }
    }
}

// Adds the splits' partial images (channel-planar) in order.
template <int NCH>
__global__ __launch_bounds__(256) void k_draw_reduce(DrawPlan P, const float* __restrict__ partials, float* __restrict__ image) {
    const uint64_t all = (uint64_t)P.windows * P.size * P.size;
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= all) return;
    float v[NCH];
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) v[ch] = 0.0f;
    for (uint32_t s = 0; s < P.splits; ++s)
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) v[ch] += partials[((uint64_t)s * NCH + ch) * all + p];
    if constexpr (NCH == 4) {
        const uint64_t area = (uint64_t)P.size * P.size;
        const uint64_t win = p / area, y = (p - win * area) / P.size, x = p % P.size;
        const uint64_t at = ((win / P.win_cols) * P.size + y) * P.stride + (win % P.win_cols) * P.size + x;
        reinterpret_cast<float4*>(image)[at] = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) image[p * NCH + ch] = v[ch];
    }
}

bool make_draw_plan(int size, int radius, uint32_t windows, uint32_t per_window, uint32_t count, uint32_t channels,
                    uint32_t win_cols, DrawPlan* plan) {
    DrawPlan p{};
    p.size = size;
    p.tiles_x = (size + 15) / 16;
    p.windows = windows;
    p.per_window = per_window;
    p.count = count;
    p.channels = channels;
    p.win_cols = win_cols;
    p.stride = (int)(win_cols * (uint32_t)size);
    p.rect_shift = p.tiles_x > 127 ? 1 : 0;
    const uint64_t cus = (uint64_t)device_cu_count();
    auto blocks = [&](uint32_t g) {
        const uint64_t gx = ((uint64_t)p.tiles_x + g - 1) / g;
        return gx * gx * windows;
    };
    // the largest groups that still give every CU a block
    p.group = blocks(4) >= cus ? 4 : blocks(2) >= cus ? 2 : 1;
    p.groups_x = ((uint32_t)p.tiles_x + p.group - 1) / p.group;
    p.groups = (uint32_t)std::min<uint64_t>(blocks(p.group), UINT32_MAX);
    // Groups: an object on a part of the window leaves most CUs without items, so the further ranges of crowded
    // groups' items go to blocks of their own, at most one per CU (draw_crowd). Measured, one block per group
    // against ranges: 100,000 particles on a tenth of a 512x512 view 2,232 -> 178 us, four such views 4,626 ->
    // 608 us, on a fiftieth of a 1024x1024 view 5,793 -> 311 us, a splat of 300,000 on a tenth of 2048x2048 2,722 ->
    // 433 us; even drawings keep their times (65,536 at 512x512 27 us).
    p.extra = p.group > 1 && p.groups <= kDrawGroups && count >= 1024 ? std::min(count / 256, kCrowdMost) : 0;
    // Single tiles: ranges of at least 512 of a window's items go to blocks of their own, for four blocks per
    // CU and for about 128 items per block where the items spread over the window (four times that where
    // an object fills its middle), so that crowded tiles leave no CU waiting. Measured, one range against
    // the rule's: four 64x64 views of 16,384 particles 60 -> 45 us, 200x200 of 32,768 202 -> 88 us, 100x100
    // of 32,768 154 -> 85 us. Small footprints have few items per tile and stay with the first rule (a
    // 256x256 splat of 20,000 particles: 17 us with four ranges, 29 us with sixteen).
    p.splits = 1;
    if (p.group == 1) {
        const uint64_t n = std::min(per_window, count);
        const double side = std::min(1.0, (2.0 * radius + 17.0) / size);
        const uint64_t crowd = (uint64_t)((double)n * side * side / 128.0);
        p.splits = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({std::max(4 * cus / blocks(1), crowd), n / 512, 16}));
    }
    p.partial_floats = p.splits > 1 ? (uint64_t)p.splits * channels * windows * size * size
                                    : (uint64_t)p.extra * channels * p.group * p.group * 256;
    if (blocks(p.group) >= (1ull << 31)) return false;
    *plan = p;
    return true;
}

__global__ __launch_bounds__(256) void k_draw_clear(uint32_t* tickets) {
    tickets[blockIdx.x * 256 + threadIdx.x] = 0;
}

hipError_t reserve_draw(const DrawPlan& p, SplatWorkspace& ws, hipStream_t stream) {
    hipError_t e = ws.partials.reserve(p.partial_floats * 4);
    if (e != hipSuccess || !p.extra || ws.crowd.ptr) return e;
    if ((e = ws.crowd.reserve(kCrowdWords * 4)) != hipSuccess) return e;
    // the tickets are zero between drawings: the block that takes a group's last one clears it
    hipLaunchKernelGGL(k_draw_clear, dim3(kDrawGroups / 256), dim3(256), 0, stream, ws.crowd.as<uint32_t>());
    if ((e = hipGetLastError()) != hipSuccess) ws.crowd.release();  // cleared by the next drawing, then
    return e;
}

template <int NCH>
static hipError_t launch_draw_n(const DrawPlan& p, const DrawItem* items, const uint32_t* rects, SplatWorkspace& ws,
                                float* image, hipStream_t stream) {
    auto k = p.group == 4 ? k_draw_tiles<NCH, 4, 16> : p.group == 2 ? k_draw_tiles<NCH, 2, 16> : k_draw_tiles<NCH, 1, 4>;
    hipLaunchKernelGGL(k, dim3(p.groups + p.extra, p.splits), dim3(p.group == 1 ? 256 : 1024), 0, stream, p,
                       reinterpret_cast<const float4*>(items), rects, ws.partials.as<float>(), ws.crowd.as<uint32_t>(),
                       image);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.splits == 1) return e;
    const uint64_t pixels = (uint64_t)p.windows * p.size * p.size;
    hipLaunchKernelGGL(k_draw_reduce<NCH>, dim3((uint32_t)((pixels + 255) / 256)), dim3(256), 0, stream, p,
                       ws.partials.as<float>(), image);
    return hipGetLastError();
}

hipError_t launch_draw(const DrawPlan& p, const DrawItem* items, const uint32_t* rects, SplatWorkspace& ws, float* image,
                       hipStream_t stream) {
    return p.channels == 4 ? launch_draw_n<4>(p, items, rects, ws, image, stream)
                           : launch_draw_n<5>(p, items, rects, ws, image, stream);
}

}  // namespace npa
