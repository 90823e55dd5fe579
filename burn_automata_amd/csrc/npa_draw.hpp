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
    uint32_t win_cols;                    // 4 channels: windows per image row
    int stride;                           // 4 channels: pixels per image row
    uint64_t partial_floats;              // of the splits' partial images (0 without splits)
};

// Lays out a drawing of items with footprints of about 2 * radius + 1 pixels; false beyond the grid's limits.
bool make_draw_plan(int size, int radius, uint32_t windows, uint32_t per_window, uint32_t count, uint32_t channels,
                    uint32_t win_cols, DrawPlan* plan);
// image: 4 channels [rows of windows * size][win_cols * size][4], 5 channels [windows][size][size][5].
hipError_t launch_draw(const DrawPlan& plan, const DrawItem* items, const uint32_t* rects, float* partials, float* image,
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
__device__ __forceinline__ bool draw_finite(const DrawItem& d) {
    return isfinite(d.px) && isfinite(d.py) && isfinite(d.k2) && isfinite(d.scale) && isfinite(d.scale * d.c[0]) &&
           isfinite(d.scale * d.c[1]) && isfinite(d.scale * d.c[2]) && isfinite(d.c[0]) && isfinite(d.c[1]) &&
           isfinite(d.c[2]) && isfinite(d.depth);
}

}  // namespace npa
