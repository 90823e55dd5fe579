// npa_draw.hpp - isotropic Gaussian footprints drawn as a contraction on the matrix cores (npa_draw.hip).
#pragma once

#include "npa_internal.hpp"

namespace npa {

// What one item (a particle, or a particle seen through one view) adds to pixel (x, y) of its window,
// for x0 <= x <= x0 + span and y0 <= y <= y0 + span: scale * 2^(-k2 ((x - px)^2 + (y - py)^2)) times
// its channels (c, then 1, then depth).
struct alignas(16) DrawItem {  // 48 bytes
    float px, py, k2, scale;
    float c[3], depth;
    int x0, y0;
    uint32_t span;
    uint32_t special;  // a value, or a product of scale and a channel, is not finite: drawn pixel by pixel
};

// The window's 16x16 tiles an item touches (pairs of them, where an axis has more than 127), as four
// seven-bit numbers each in a byte of its own: tx0, 127 - tx1, ty0, 127 - ty1. An item touches a group
// of tiles gx0..gx1, gy0..gy1 when every byte of its word is at most that of the group's word
// (gx1, 127 - gx0, gy1, 127 - gy0). kDrawNone touches none (tx0 = 127 and tx1 = 0 on an axis of at most
// 128 tiles whose groups span fewer).
__host__ __device__ inline uint32_t draw_rect(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return a | (127u - b) << 8 | c << 16 | (127u - d) << 24;
}
constexpr uint32_t kDrawNone = 0x7f7f7f7fu;

struct DrawPlan {
    int size, tiles_x;
    uint32_t windows, per_window, count;  // window w holds items [w * per_window, + per_window), up to count
    uint32_t channels;                    // 4 (r, g, b, weight) or 5 (and depth)
    uint32_t rect_shift;                  // 1: rectangles count pairs of tiles
    uint32_t group, groups_x, splits;     // tiles per block and axis, blocks per window and axis, item ranges
    uint32_t groups, extra;               // groups of all windows; blocks for further ranges of crowded groups
    uint32_t win_cols;                    // 4 channels: windows per image row
    int stride;                           // 4 channels: pixels per image row
    uint64_t partial_floats;              // of the splits' partial images, or of the further ranges' groups
};

// Lays out a drawing of items with footprints of about 2 * radius + 1 pixels; false beyond the grid's limits.
bool make_draw_plan(int size, int radius, uint32_t windows, uint32_t per_window, uint32_t count, uint32_t channels,
                    uint32_t win_cols, DrawPlan* plan);
// image: 4 channels [rows of windows * size][win_cols * size][4], 5 channels [windows][size][size][5].
// ws: its partials and crowd, reserved by reserve_draw.
hipError_t reserve_draw(const DrawPlan& plan, SplatWorkspace& ws, hipStream_t stream);
hipError_t launch_draw(const DrawPlan& plan, const DrawItem* items, const uint32_t* rects, SplatWorkspace& ws, float* image,
                       hipStream_t stream);

// An item's weight sum over the in-image part of its footprint, as the product of its two axes' sums, and its
// tiles. (bx, by): the pixel of its centre.
struct Footprint {
    uint32_t rect;
    float weights;
};
__device__ __forceinline__ float axis_weights(float p, float k2, int lo, int hi) {
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // four sums in flight
    for (int v = lo; v <= hi; v += 4)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float d = (float)(v + u) - p;
            const float w = __builtin_amdgcn_exp2f(-(d * d) * k2);
            s[u] += v + u <= hi ? w : 0.0f;
        }
    return (s[0] + s[1]) + (s[2] + s[3]);
}
__device__ __forceinline__ Footprint draw_footprint(float px, float py, float k2, int64_t bx, int64_t by, int64_t r, int size) {
    int64_t x0 = bx - r, x1 = bx + r, y0 = by - r, y1 = by + r;
    if (x0 < 0) x0 = 0;
    if (y0 < 0) y0 = 0;
    if (x1 > size - 1) x1 = size - 1;
    if (y1 > size - 1) y1 = size - 1;
    if (x0 > x1 || y0 > y1) return {kDrawNone, 0.0f};
    const uint32_t sh = size > 127 * 16 ? 5u : 4u;
    const uint32_t rect = draw_rect((uint32_t)x0 >> sh, (uint32_t)x1 >> sh, (uint32_t)y0 >> sh, (uint32_t)y1 >> sh);
    return {rect, axis_weights(px, k2, (int)x0, (int)x1) * axis_weights(py, k2, (int)y0, (int)y1)};
}

// Whether the item can be drawn as matrix products: its values are finite, and so is every operand
// (e(y) scale) c, which scale * c bounds (an infinite one would meet the zeros outside the footprint).
// Whether the item can be drawn as matrix products: its values are finite, and so is every operand
// (e(y) scale) c, which scale * c bounds (an infinite one would meet the zeros outside the footprint).
__device__ __forceinline__ bool draw_finite(const DrawItem& d) {
    return isfinite(d.px) && isfinite(d.py) && isfinite(d.k2) && isfinite(d.scale) && isfinite(d.scale * d.c[0]) &&
           isfinite(d.scale * d.c[1]) && isfinite(d.scale * d.c[2]) && isfinite(d.c[0]) && isfinite(d.c[1]) &&
           isfinite(d.c[2]) && isfinite(d.depth);
}


// Crowded groups of a grouped drawing, found by one block of the item kernel from a sample of the items, so
// that the drawing's blocks read what to draw: words [0, kDrawGroups) are its tickets, [kCrowdGroups, + groups)
// per group its ranges after the first | its first slot << 8, then the number of jobs (further ranges) and per job
// its group | range << 16.
constexpr uint32_t kDrawGroups = 4096;  // most groups among which crowded ones are looked for
constexpr uint32_t kCrowdMost = 256;    // most jobs
constexpr uint32_t kCrowdGroups = kDrawGroups, kCrowdJobs = 2 * kDrawGroups;
constexpr uint32_t kCrowdWords = kCrowdJobs + 1 + kCrowdMost;
constexpr uint32_t kCrowdSample = 1024;

// Whole blocks of 256 threads; it has to be done in the time of the other blocks, about 5 us. box_of(window, item,
// box): the item's footprint in whole pixels, before the image's edges. A group's items are estimated from the
// sampled footprints that touch it (of wide ones the middle groups). It is crowded, and cut into ranges of about C
// items, if it has at least 3 C, with C at least 512, the groups' mean and a P.extra-th of all; sixteen sampled
// items at least. An even drawing has none: its blocks fill every CU for the same time, and one range more would
// be a round of its own (200,000 items in four 256x256 windows, of whose 256 groups one or two seem to have twice the
// mean: 62 us, 81 us with their ranges).
template <class BoxOf>
__device__ __forceinline__ void draw_crowd(const DrawPlan& P, uint32_t* crowd, BoxOf&& box_of) {
    __shared__ uint32_t hist[kDrawGroups], sums[4], jobs[4];
    constexpr uint32_t PER = kCrowdSample / 256;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float box[PER][4];  // first and last column, first and last row
    uint32_t win[PER];
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        const uint32_t k = i * 256 + threadIdx.x;
        const uint32_t item = P.count > kCrowdSample ? (uint32_t)((uint64_t)k * P.count / kCrowdSample) : k;
        win[i] = item / P.per_window;
        box[i][0] = 1.0f;
        box[i][1] = box[i][2] = box[i][3] = 0.0f;
        if (item < P.count) box_of(win[i], item, box[i]);
    }
    for (uint32_t g = threadIdx.x; g < P.groups; g += 256) hist[g] = 0;
    __syncthreads();
    const uint32_t lg = P.group == 4 ? 6 : 5;  // pixels -> groups
    const float edge = (float)(P.size - 1);
    uint32_t hits = 0;
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        const float x0 = fmaxf(box[i][0], 0.0f), x1 = fminf(box[i][1], edge);
        const float y0 = fmaxf(box[i][2], 0.0f), y1 = fminf(box[i][3], edge);
        if (!(x0 <= x1 && y0 <= y1)) continue;
        uint32_t xa = (uint32_t)x0 >> lg, xb = (uint32_t)x1 >> lg, ya = (uint32_t)y0 >> lg, yb = (uint32_t)y1 >> lg;
        if (xb - xa > 3) {
            xa = (xa + xb) / 2 - 1;
            xb = xa + 3;
        }
        if (yb - ya > 3) {
            ya = (ya + yb) / 2 - 1;
            yb = ya + 3;
        }
        uint32_t* h = hist + (win[i] * P.groups_x + ya) * P.groups_x;
        for (uint32_t y = ya; y <= yb; ++y, h += P.groups_x)
            for (uint32_t x = xa; x <= xb; ++x, ++hits) atomicAdd(h + x, 1u);
    }
    hits = wave_sum_u32(hits);
    if (lane == 0) sums[wave] = hits;
    __syncthreads();
    // items per hit; C; ranges per hit
    const float scale = P.count > kCrowdSample ? (float)P.count / kCrowdSample : 1.0f;
    const float all = (float)(sums[0] + sums[1] + sums[2] + sums[3]) * scale;
    const float c = fmaxf(512.0f, fmaxf(all / (float)P.groups, all / (float)P.extra)), per_hit = scale / c;
    auto more_of = [&](uint32_t h) {
        const uint32_t n = (uint32_t)((float)h * per_hit);
        return h < 16 || n < 3 ? 0u : min(n, 63u);
    };
    // consecutive groups per thread, sixteen or fewer
    const uint32_t per = (P.groups + 255) / 256;
    const uint32_t g0 = min(P.groups, threadIdx.x * per), g1 = min(P.groups, g0 + per);
    uint32_t more = 0;
    for (uint32_t g = g0; g < g1; ++g) more += more_of(hist[g]);
    uint32_t incl = more;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, 64);
        if (lane >= (uint32_t)off) incl += y;
    }
    if (lane == 63) jobs[wave] = incl;
    __syncthreads();
    uint32_t at = incl - more;
    for (uint32_t w = 0; w < wave; ++w) at += jobs[w];
    for (uint32_t g = g0; g < g1; ++g) {
        const uint32_t m = min(more_of(hist[g]), P.extra - min(at, P.extra));  // (for the products' rounding)
        crowd[kCrowdGroups + g] = m | at << 8;
        for (uint32_t s = 1; s <= m; ++s) crowd[kCrowdJobs + at + s] = g | s << 16;
        at += m;
    }
    if (threadIdx.x == 255) crowd[kCrowdJobs] = min(at, P.extra);
}

}  // namespace npa
