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
// No sort either: a block covers a group of G x G tiles, tests every item of its window's 32-bit tile
// rectangle (8,192 at a time, the next ones' loads in flight) and keeps the indices of those that touch the
// group, in ascending order; the block's waves then draw the group's tiles from that list (several waves per
// tile for small groups, their sums added in a fixed order). So items are added in a fixed order and the
// image is deterministic; it differs from the reference's running sums only by rounding.
//
// Bound: the matrix instructions, 32 cycles per channel and four items (160 cycles for five channels), plus
// the tests, 8 instructions per 64 items and group.
#include "npa_draw.hpp"

#include <algorithm>

namespace npa {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr uint32_t kDrawWaves = 16;
constexpr uint32_t kDrawPer = 8;                                // items a thread tests per batch
constexpr uint32_t kDrawBatch = kDrawWaves * 64 * kDrawPer;     // 8,192
constexpr uint32_t kDrawQueue = 72;                             // a wave's queue: 64 new entries after up to 7

__device__ __forceinline__ bool rect_touches(uint32_t r, uint32_t gx0, uint32_t gx1, uint32_t gy0, uint32_t gy1) {
    return (r & 255u) <= gx1 && ((r >> 8) & 255u) >= gx0 && ((r >> 16) & 255u) <= gy1 && (r >> 24) >= gy0;
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
    // Adds four items, one per 16 lanes; `live` false: this lane's item adds nothing.
    __device__ __forceinline__ void add(const float4& a, const float4& b, const uint4& w, bool live) {
        const int x0 = (int)w.x, y0 = (int)w.y;
        const uint64_t odd = __ballot(live && w.w != 0u);
        const bool use = live && w.w == 0u;
        const float dx = xf - a.x, dy = yf - a.y;
        float ex = __builtin_amdgcn_exp2f(-(dx * dx) * a.z);
        float ey = __builtin_amdgcn_exp2f(-(dy * dy) * a.z) * a.w;
        ex = use && (uint32_t)(x - x0) <= w.z ? ex : 0.0f;
        ey = use && (uint32_t)(y - y0) <= w.z ? ey : 0.0f;
        const float c[5] = {use ? b.x : 0.0f, use ? b.y : 0.0f, use ? b.z : 0.0f, 1.0f, use ? b.w : 0.0f};
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch)
            acc[ch] = __builtin_amdgcn_mfma_f32_16x16x4f32(ch == 3 ? ey : ey * c[ch], ex, acc[ch], 0, 0, 0);
        if (odd) add_special(a, b, w, odd);
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

// Grid: x = window * groups_x^2 + group, y = split of the window's items.
template <int NCH, int G>
__global__ __launch_bounds__(kDrawWaves * 64) void k_draw_tiles(DrawPlan P, const float4* __restrict__ items,
                                                                const uint32_t* __restrict__ rects,
                                                                float* __restrict__ partials, float* __restrict__ image) {
    constexpr uint32_t TILES = G * G, WPT = kDrawWaves / TILES;  // tiles per block, waves per tile
    constexpr uint32_t NR = NCH * 4;                             // accumulated values per lane
    // the batch's kept items (rectangle, index), then the waves' queues; the sums of the waves at the end
    constexpr uint32_t LIST = kDrawBatch * 2, QUEUE = kDrawWaves * kDrawQueue, SUMS = kDrawWaves * NR * 64;
    __shared__ uint32_t lds[LIST + QUEUE > SUMS ? LIST + QUEUE : SUMS];
    __shared__ uint32_t counts[kDrawPer * kDrawWaves];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t per_win = P.groups_x * P.groups_x;
    const uint32_t win = blockIdx.x / per_win, grp = blockIdx.x - win * per_win;
    const uint32_t gx0 = grp % P.groups_x * G, gy0 = grp / P.groups_x * G;
    const uint32_t tg = wave % TILES, part = wave / TILES;
    const uint32_t tx = gx0 + tg % G, ty = gy0 + tg / G;
    DrawTile<NCH> tile;
    tile.init(tx, ty, lane);
    uint2* list = reinterpret_cast<uint2*>(lds);
    uint32_t* queue = lds + LIST + wave * kDrawQueue;
    // this block's items
    const uint64_t win_beg = (uint64_t)win * P.per_window;
    const uint64_t win_end = win_beg + P.per_window < P.count ? win_beg + P.per_window : P.count;
    const uint32_t n = win_end > win_beg ? (uint32_t)(win_end - win_beg) : 0u;
    const uint32_t share = (n + P.splits - 1) / P.splits;
    const uint32_t first = min(n, blockIdx.y * share), last = min(n, first + share);
    const uint32_t* rw = rects + win_beg;

    uint32_t waiting = 0;  // entries in this wave's queue
    // draws eight entries of the queue, the first `count` of them live; their loads are issued together
    auto draw = [&](uint32_t at, uint32_t count) {
        float4 a[2], b[2];
        uint4 w[2];
        bool live[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t k = 4 * h + lane / 16;
            live[h] = k < count;
            const uint64_t idx = queue[at + (live[h] ? k : 0u)];
            const float4* it = items + idx * 3;
            a[h] = it[0];
            b[h] = it[1];
            w[h] = reinterpret_cast<const uint4*>(it)[2];
        }
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h)
            if (4 * h < count) tile.add(a[h], b[h], w[h], live[h]);
    };
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    uint32_t r[kDrawPer];
    auto fetch = [&](uint32_t base) {
#pragma unroll
        for (uint32_t i = 0; i < kDrawPer; ++i) {
            const uint32_t k = base + i * (kDrawWaves * 64) + threadIdx.x;
            r[i] = k < last ? rw[k] : kDrawNone;
        }
    };
    fetch(first);
    for (uint32_t base = first; base < last; base += kDrawBatch) {
        uint64_t hit[kDrawPer];
        uint32_t kept[kDrawPer];
#pragma unroll
        for (uint32_t i = 0; i < kDrawPer; ++i) {
            kept[i] = r[i];
            hit[i] = __ballot(rect_touches(r[i], gx0, gx0 + G - 1, gy0, gy0 + G - 1));
            if (lane == 0) counts[i * kDrawWaves + wave] = (uint32_t)__popcll(hit[i]);
        }
        fetch(base + kDrawBatch);
        __syncthreads();
        // ascending positions: instruction i, then wave, then lane (two of the 128 counts per lane)
        const uint32_t c0 = counts[2 * lane], c1 = counts[2 * lane + 1];
        const uint32_t incl = wave_incl_add(c0 + c1);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
#pragma unroll
        for (uint32_t i = 0; i < kDrawPer; ++i) {
            const uint32_t slot = i * kDrawWaves + wave;  // wave-uniform
            const uint32_t upto = (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)(slot / 2));
            const uint32_t s1 = (uint32_t)__builtin_amdgcn_readlane((int)c1, (int)(slot / 2));
            const uint32_t s0 = (uint32_t)__builtin_amdgcn_readlane((int)c0, (int)(slot / 2));
            const uint32_t at = upto - s1 - (slot % 2 ? 0u : s0);
            if ((hit[i] >> lane) & 1ull)
                list[at + (uint32_t)__popcll(hit[i] & lanemask_lt())] =
                    make_uint2(kept[i], base + i * (kDrawWaves * 64) + threadIdx.x);
        }
        __syncthreads();
        for (uint32_t k0 = part * 64; k0 < total; k0 += WPT * 64) {
            const uint2 e = k0 + lane < total ? list[k0 + lane] : make_uint2(kDrawNone, 0u);
            const bool mine = rect_touches(e.x, tx, tx, ty, ty);
            const uint64_t m = __ballot(mine);
            if (mine) queue[waiting + (uint32_t)__popcll(m & lanemask_lt())] = (uint32_t)win_beg + e.y;
            waiting += (uint32_t)__popcll(m);
            wave_fence();
            uint32_t at = 0;
            for (; waiting - at >= 8; at += 8) draw(at, 8);
            const uint32_t rest = waiting - at;  // up to seven wait for the next entries
            const uint32_t keep = lane < rest ? queue[at + lane] : 0u;
            wave_fence();
            if (lane < rest) queue[lane] = keep;
            waiting = rest;
            wave_fence();
        }
        __syncthreads();  // the list and the counts are read before the next batch fills them
    }
    if (waiting) draw(0, waiting);
    __syncthreads();
    float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch)
#pragma unroll
        for (int q = 0; q < 4; ++q) sums[(wave * NR + ch * 4 + q) * 64 + lane] = tile.acc[ch][q];
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < TILES * 256; t += kDrawWaves * 64) {
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
        if (P.splits > 1) {
            const uint64_t pixel = ((uint64_t)win * P.size + y) * P.size + x, all = (uint64_t)P.windows * P.size * P.size;
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) partials[((uint64_t)blockIdx.y * NCH + ch) * all + pixel] = v[ch];
        } else if constexpr (NCH == 4) {
            const uint64_t at = ((uint64_t)(win / P.win_cols) * P.size + y) * P.stride + (uint64_t)(win % P.win_cols) * P.size + x;
            reinterpret_cast<float4*>(image)[at] = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            float* o = image + (((uint64_t)win * P.size + y) * P.size + x) * NCH;
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) o[ch] = v[ch];
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

bool make_draw_plan(int size, uint32_t windows, uint32_t per_window, uint32_t count, uint32_t channels, uint32_t win_cols,
                    DrawPlan* plan) {
    DrawPlan p{};
    p.size = size;
    p.tiles_x = (size + 15) / 16;
    p.windows = windows;
    p.per_window = per_window;
    p.count = count;
    p.channels = channels;
    p.win_cols = win_cols;
    p.stride = (int)(win_cols * (uint32_t)size);
    const uint64_t cus = (uint64_t)device_cu_count();
    auto blocks = [&](uint32_t g) {
        const uint64_t gx = ((uint64_t)p.tiles_x + g - 1) / g;
        return gx * gx * windows;
    };
    // the largest groups that still give every CU a block
    p.group = blocks(4) >= cus ? 4 : blocks(2) >= cus ? 2 : 1;
    p.groups_x = ((uint32_t)p.tiles_x + p.group - 1) / p.group;
    // few tiles: ranges of at least 1,024 items of a window go to blocks of their own
    p.splits = 1;
    if (blocks(p.group) < cus)
        p.splits = (uint32_t)std::max<uint64_t>(
            1, std::min<uint64_t>({cus / blocks(p.group), (uint64_t)std::min(per_window, count) / 1024, 16}));
    p.partial_floats = p.splits > 1 ? (uint64_t)p.splits * channels * windows * size * size : 0;
    if (blocks(p.group) >= (1ull << 31)) return false;
    *plan = p;
    return true;
}

template <int NCH>
static hipError_t launch_draw_n(const DrawPlan& p, const DrawItem* items, const uint32_t* rects, float* partials,
                                float* image, hipStream_t stream) {
    auto k = p.group == 4 ? k_draw_tiles<NCH, 4> : p.group == 2 ? k_draw_tiles<NCH, 2> : k_draw_tiles<NCH, 1>;
    hipLaunchKernelGGL(k, dim3(p.groups_x * p.groups_x * p.windows, p.splits), dim3(kDrawWaves * 64), 0, stream, p,
                       reinterpret_cast<const float4*>(items), rects, partials, image);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.splits == 1) return e;
    const uint64_t pixels = (uint64_t)p.windows * p.size * p.size;
    hipLaunchKernelGGL(k_draw_reduce<NCH>, dim3((uint32_t)((pixels + 255) / 256)), dim3(256), 0, stream, p, partials, image);
    return hipGetLastError();
}

hipError_t launch_draw(const DrawPlan& p, const DrawItem* items, const uint32_t* rects, float* partials, float* image,
                       hipStream_t stream) {
    return p.channels == 4 ? launch_draw_n<4>(p, items, rects, partials, image, stream)
                           : launch_draw_n<5>(p, items, rects, partials, image, stream);
}

}  // namespace npa
