// npa_decode.hip - Gaussian decode, the splat's and the render's items and the oriented raster on gfx950.
//
// decode_gaussians_3d  crates/burn_automata_kernels/src/gaussian.rs:53-223: a per-particle map.
//
// splat_particles_2d   crates/burn_automata_kernels/src/splat.rs:30-93, and the render loss's
// project_positions + splat_projected: the particles' footprints are prepared here and drawn by
// npa_draw.hip, deterministically.
//
// The oriented Gaussian raster: per-tile lists in depth order, composited front to back.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "npa_draw.hpp"
#include "npa_internal.hpp"

namespace npa {

// --------------------------------------------------------------- decode
__global__ __launch_bounds__(256) void k_decode(const float4* __restrict__ pos, const float* __restrict__ states,
                                                uint32_t count, uint32_t S, npa_gaussian_decode_cfg cfg,
                                                uint32_t K, float* __restrict__ pv, float* __restrict__ sh,
                                                float* __restrict__ rot, float* __restrict__ so) {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= count) return;
    const float* s = states + (uint64_t)idx * S;
    const float4 p = pos[idx];
    const uint32_t color_start = cfg.mode == NPA_DECODE_SH0_ORIENTED ? S - K * 3 : S - 3;
    for (uint32_t k = 0; k < K; ++k) {  // decode_sh gaussian.rs:134-158
        const uint32_t base = color_start + k * 3;
        for (int ch = 0; ch < 3; ++ch)
            sh[((uint64_t)idx * K + k) * 3 + ch] = clampf_(s[base + ch] + 0.5f, 0.0f, 1.0f);
    }
    float q[4] = {1.0f, 0.0f, 0.0f, 0.0f};
    if (cfg.mode == NPA_DECODE_SH0_ORIENTED) {  // normalize_quat gaussian.rs:214-223
        const uint32_t rs = color_start - 4;
        q[0] = s[rs];
        q[1] = s[rs + 1];
        q[2] = s[rs + 2];
        q[3] = s[rs + 3];
        const float norm = sqrtf(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        if (norm <= 1e-8f) {
            q[0] = 1.0f;
            q[1] = q[2] = q[3] = 0.0f;
        } else {
            for (int k = 0; k < 4; ++k) q[k] /= norm;
        }
    }
    float o[4];
    switch (cfg.mode) {  // decode_scale_opacity gaussian.rs:160-208
        case NPA_DECODE_PARTICLE_POINT: {
            const float sc = fmaxf(cfg.min_scale, 1.0e-6f);
            o[0] = o[1] = o[2] = sc;
            o[3] = 1.0f;
        } break;
        case NPA_DECODE_SH0_FIXED_SCALE: {
            const float sc = clampf_(cfg.sigma, cfg.min_scale, cfg.max_scale);
            o[0] = o[1] = o[2] = sc;
            o[3] = clampf_(cfg.opacity_scale, cfg.min_opacity, cfg.max_opacity);
        } break;
        case NPA_DECODE_SH0_LEARNED_SCALE: {
            const float scale_logit = clampf_(s[S - 5], -8.0f, 8.0f);
            const float opacity_logit = clampf_(s[S - 4], -12.0f, 12.0f);
            const float sc = clampf_(cfg.sigma * expf(scale_logit), cfg.min_scale, cfg.max_scale);
            const float sig = 1.0f / (1.0f + expf(-opacity_logit));
            const float op = clampf_(sig, cfg.min_opacity, cfg.max_opacity) * cfg.opacity_scale;
            o[0] = o[1] = o[2] = sc;
            o[3] = clampf_(op, cfg.min_opacity, cfg.max_opacity);
        } break;
        default: {
            const uint32_t anis = color_start - 8;
            const float ma = fmaxf(cfg.max_anisotropy, 1e-6f);
            const float ax = tanhf(s[anis] / ma) * cfg.max_anisotropy;
            const float ay = tanhf(s[anis + 1] / ma) * cfg.max_anisotropy;
            const float az = tanhf(s[anis + 2] / ma) * cfg.max_anisotropy;
            const float ol = tanhf(s[anis + 3] / ma) * cfg.max_anisotropy;
            o[0] = clampf_(cfg.sigma * expf(ax), cfg.min_scale, cfg.max_scale);
            o[1] = clampf_(cfg.sigma * expf(ay), cfg.min_scale, cfg.max_scale);
            o[2] = clampf_(cfg.sigma * expf(az), cfg.min_scale, cfg.max_scale);
            o[3] = clampf_(cfg.opacity_scale * expf(ol), cfg.min_opacity, cfg.max_opacity);
        } break;
    }
    reinterpret_cast<float4*>(pv)[idx] = make_float4(p.x, p.y, p.z, 1.0f);
    reinterpret_cast<float4*>(rot)[idx] = make_float4(q[0], q[1], q[2], q[3]);
    reinterpret_cast<float4*>(so)[idx] = make_float4(o[0], o[1], o[2], o[3]);
}

hipError_t launch_decode_gaussians(const float4* pos, const float* states, uint32_t count, uint32_t S,
                                   const npa_gaussian_decode_cfg& cfg, float* pv, float* sh, float* rot,
                                   float* so, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const uint32_t K = cfg.mode == NPA_DECODE_SH0_ORIENTED ? (cfg.sh_degree + 1) * (cfg.sh_degree + 1) : 1;
    hipLaunchKernelGGL(k_decode, dim3((count + 255) / 256), dim3(256), 0, stream, pos, states, count, S, cfg, K,
                       pv, sh, rot, so);
    return hipGetLastError();
}

// ------------------------------------------------------------ viewer export
// write_gaussian_from_output  crates/burn_automata/src/gpu_step.wgsl:4963-5052 (write_gaussian_main
// 4929-4936): position (z = 0 in 2D) and visibility 1; 48 SH coefficients, zero but for the DC
// triple (clamp(tail + 0.5) - 0.5) / SH_C0 of the last three state channels (4981-4990); identity
// rotation and isotropic scale max(eps * 0.12, 8e-5), or for 3D position-feature models with
// S >= 9 the rotation taking +z onto the normal in channels 4..6 and a flattened tangent-plane
// scale (4992-5045); opacity 1 in 2D, clamp(sigmoid(channel 8, or 3 when S <= 8), 0.001, 0.95) in
// 3D (5046-5051). normalize() is v / sqrt(sum v^2) and length() sqrt(x^2 + y^2 + z^2), in that
// order (the oracle's restatement evaluates the same operations). The material branch belongs to
// the adaptive rollouts and is not built.
constexpr float kShC0 = 0.28209479177387814f;  // SH_C0 gpu_step.wgsl:7
constexpr uint32_t kShCoeffs = NPA_GAUSSIAN_SH_COEFF_COUNT;

struct ExportParams {
    uint32_t total, N, S, dim;
    float eps;
    uint32_t normal_branch;
};

__device__ __forceinline__ float export_channel(const float* s, uint32_t S, uint32_t c) {  // output_state_channel
    return c < S ? s[c] : (S > 0 ? s[0] : 0.0f);
}

// One thread per particle for the 4-float records; each wave then writes its 64 particles' SH
// rows (12 float4 each) as consecutive float4s, lane l taking float4 j * 64 + l of the wave's
// block and the DC triple from the particle's lane.
__global__ __launch_bounds__(256) void k_write_gaussians(ExportParams P, const float4* __restrict__ pos,
                                                         const float* __restrict__ states, float4* __restrict__ pv,
                                                         float4* __restrict__ sh, float4* __restrict__ rot,
                                                         float4* __restrict__ so) {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    float dc[3] = {0.0f, 0.0f, 0.0f};
    if (idx < P.total) {
        const uint32_t S = P.S;
        const float* s = states + (uint64_t)idx * S;
        const float4 p = pos[idx];
        pv[idx] = make_float4(p.x, p.y, P.dim == 3 ? p.z : 0.0f, 1.0f);
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {  // output_tail_state_channel(idx, 2 - ch)
            const uint32_t off = 2u - (uint32_t)ch;
            const float tail = S > off ? export_channel(s, S, S - 1 - off) : export_channel(s, S, 0);
            const float color = clampf_(tail + 0.5f, 0.0f, 1.0f);
            dc[ch] = (color - 0.5f) / kShC0;
        }
        const float iso = fmaxf(P.eps * 0.12f, 0.00008f);
        float sc[3] = {iso, iso, iso};
        float q[4] = {1.0f, 0.0f, 0.0f, 0.0f};
        if (P.normal_branch) {
            const float n0 = export_channel(s, S, 4), n1 = export_channel(s, S, 5), n2 = export_channel(s, S, 6);
            const float nn = sqrtf(n0 * n0 + n1 * n1 + n2 * n2);
            float u0 = 0.0f, u1 = 0.0f, u2 = 1.0f;
            if (nn > 1.0e-6f && nn < 1.0e20f) {
                u0 = n0 / nn;
                u1 = n1 / nn;
                u2 = n2 / nn;
            }
            if (u2 <= -0.999999f) {
                q[0] = 0.0f;
                q[1] = 1.0f;
                q[2] = 0.0f;
                q[3] = 0.0f;
            } else {
                const float r[4] = {1.0f + u2, -u1, u0, 0.0f};
                const float rl = sqrtf(r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + r[3] * r[3]);
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = r[k] / rl;
            }
            const float density_scale = clampf_(sqrtf(4096.0f / fmaxf((float)P.N, 1.0f)), 0.4f, 2.0f);
            const float tangent =
                fmaxf(clampf_(P.eps * 0.32f * density_scale, P.eps * 0.08f, P.eps * 0.64f), 0.00008f);
            sc[0] = tangent;
            sc[1] = tangent;
            sc[2] = fmaxf(tangent * 0.18f, 0.00008f);
        }
        float opacity = 1.0f;
        if (P.dim == 3) {
            const float logit = export_channel(s, S, S > 8 ? 8u : 3u);
            opacity = clampf_(1.0f / (1.0f + expf(-logit)), 0.001f, 0.95f);
        }
        rot[idx] = make_float4(q[0], q[1], q[2], q[3]);
        so[idx] = make_float4(sc[0], sc[1], sc[2], opacity * 1.0f);
    }
    constexpr uint32_t kRow = kShCoeffs / 4;  // float4s per particle
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t first = idx - lane;  // the wave's first particle
#pragma unroll
    for (uint32_t j = 0; j < kRow; ++j) {
        const uint32_t v = j * 64 + lane;
        const uint32_t pl = v / kRow, comp = v - pl * kRow;
        const float d0 = __shfl(dc[0], (int)pl, 64), d1 = __shfl(dc[1], (int)pl, 64), d2 = __shfl(dc[2], (int)pl, 64);
        if (first + pl < P.total)
            sh[(uint64_t)(first + pl) * kRow + comp] = comp == 0 ? make_float4(d0, d1, d2, 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

hipError_t launch_write_gaussians(const float4* pos, const float* states, uint32_t total, uint32_t particle_count,
                                  uint32_t S, uint32_t dim, float eps, bool position_features, float* pv, float* sh,
                                  float* rot, float* so, hipStream_t stream) {
    if (total == 0) return hipSuccess;
    ExportParams P{total, particle_count, S, dim, eps, (dim == 3 && position_features && S >= 9) ? 1u : 0u};
    hipLaunchKernelGGL(k_write_gaussians, dim3((total + 255) / 256), dim3(256), 0, stream, P, pos, states,
                       (float4*)pv, (float4*)sh, (float4*)rot, (float4*)so);
    return hipGetLastError();
}

// ----------------------------------------------------------------- splat
constexpr int kTile = 16;

// A Gaussian weight exp(-d2 / (2 sigma^2)) (splat.rs:71, image.rs:61) is taken as 2^(-d2 * k2) with
// k2 = log2(e) / (2 sigma^2) on the hardware exp2; it differs from expf of the IEEE quotient by a
// few ulps at most.
constexpr float kLog2e = 1.44269504088896340736f;

// The entry points' limits: 65,536 tiles in all, and fewer than 2^31 (item, tile) pairs at the widest
// footprint.
static bool draw_within_limits(int size, uint64_t windows, uint64_t items, int radius) {
    const uint64_t tiles_x = (uint64_t)((size + kTile - 1) / kTile), tiles = tiles_x * tiles_x;
    const uint64_t per_axis = (uint64_t)((2 * radius + 1 + kTile - 1) / kTile + 1);
    return tiles * windows <= 65536 && items * std::min<uint64_t>(per_axis * per_axis, tiles) < (1ull << 31);
}

struct SplatParams {
    int size;
    int radius;
    float k2;
    float norm_scale;
    float lo, hi;
    int normalize, y_up;
    int S;
};

// One thread per particle: its pixel-space centre, window, normaliser and colour; the window's weight sum is
// the product of the two axes' sums (2 (2 r + 1) exponentials, not their square).
__global__ __launch_bounds__(256) void k_splat_items(SplatParams P, const float4* __restrict__ pos,
                                                     const float* __restrict__ colors,
                                                     const float* __restrict__ states, uint32_t count,
                                                     DrawItem* __restrict__ out, uint32_t* __restrict__ rects,
                                                     DrawPlan draw, uint32_t* __restrict__ crowd) {
    const float fsz = (float)P.size;
    const uint32_t planner = draw.extra ? 1u : 0u;  // the first block finds the crowded groups
    if (blockIdx.x < planner) {
        const float to_px = (fsz - 1.0f) / (P.hi - P.lo);
        draw_crowd(draw, crowd, [&](uint32_t, uint32_t i, float* box) {
            const float4 p = pos[i];
            const float x = floorf((p.x - P.lo) * to_px), y0 = (p.y - P.lo) * to_px;
            const float y = floorf(P.y_up ? fsz - 1.0f - y0 : y0), r = (float)P.radius;
            box[0] = x - r;
            box[1] = x + r;
            box[2] = y - r;
            box[3] = y + r;
        });
        return;
    }
    const uint32_t n = (blockIdx.x - planner) * blockDim.x + threadIdx.x;
    if (n >= count) return;
    const float4 p = pos[n];
    const float px = (p.x - P.lo) / (P.hi - P.lo) * (fsz - 1.0f);
    float py = (p.y - P.lo) / (P.hi - P.lo) * (fsz - 1.0f);
    if (P.y_up) py = (fsz - 1.0f) - py;
    const int64_t bx = f32_to_isize(floorf(px)), by = f32_to_isize(floorf(py));
    const Footprint f = draw_footprint(px, py, P.k2, bx, by, P.radius, P.size);
    DrawItem d;
    d.px = px;
    d.py = py;
    d.k2 = P.k2;
    d.scale = P.norm_scale / (P.normalize ? fmaxf(f.weights, 1e-8f) : 1.0f);
    if (colors) {
        for (int k = 0; k < 3; ++k) d.c[k] = colors[3 * (uint64_t)n + k];
    } else {  // infer_2d.rs:20-31
        const float* s = states + (uint64_t)n * P.S + (P.S - 3);
        for (int k = 0; k < 3; ++k) d.c[k] = clampf_(s[k] + 0.5f, 0.0f, 1.0f);
    }
    d.depth = 0.0f;
    const bool any = f.rect != kDrawNone;
    d.x0 = any ? (int)(bx - P.radius) : 0;
    d.y0 = any ? (int)(by - P.radius) : 0;
    d.span = 2u * (uint32_t)P.radius;
    d.special = draw_finite(d) ? 0u : 1u;
    out[n] = d;
    rects[n] = f.rect;
}

__global__ __launch_bounds__(1024) void k_scan_1block(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                      uint32_t count, uint32_t* __restrict__ total_out) {
    __shared__ uint32_t lds[32];
    const uint32_t per = (count + blockDim.x - 1) / blockDim.x;
    const uint32_t k0 = threadIdx.x * per;
    const uint32_t k1 = k0 + per < count ? k0 + per : count;
    uint32_t sum = 0;
    // batches of 8 independent loads (one memory round trip per batch, not per element)
    for (uint32_t k = k0; k < k1; k += 8) {
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = k + u < k1 ? in[k + u] : 0u;
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += v[u];
    }
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t x = sum;
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off, 64);
        if (lane >= (uint32_t)off) x += y;
    }
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    if (wid == 0) {
        uint32_t s = lane < nw ? lds[lane] : 0;
        for (int off = 1; off < 64; off <<= 1) {
            uint32_t y = __shfl_up(s, off, 64);
            if (lane >= (uint32_t)off) s += y;
        }
        if (lane < nw) lds[lane] = s;
    }
    __syncthreads();
    uint32_t run = (wid ? lds[wid - 1] : 0) + x - sum;
    for (uint32_t k = k0; k < k1; k += 8) {
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = k + u < k1 ? in[k + u] : 0u;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (k + u < k1) out[k + u] = run;
            run += v[u];
        }
    }
    if (threadIdx.x == 0) *total_out = lds[nw - 1];
}

// Multi-block exclusive scan: blocks of 256 threads own 1024 consecutive values each, loaded
// coalesced through LDS; each thread scans 4 consecutive values.
constexpr uint32_t kScanBlock = 1024;

__device__ __forceinline__ uint32_t block_exclusive_256(uint32_t v, uint32_t* lds8, uint32_t* total) {
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= (uint32_t)off) x += y;
    }
    if (lane == 63) lds8[wid] = x;
    __syncthreads();
    uint32_t pre = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) {
        const uint32_t t = lds8[w];
        if (w < wid) pre += t;
        all += t;
    }
    *total = all;
    return pre + x - v;
}

__global__ __launch_bounds__(256) void k_scan_partials(const uint32_t* __restrict__ in, uint32_t count,
                                                       uint32_t* __restrict__ sums) {
    __shared__ uint32_t lds8[4];
    const uint32_t base = blockIdx.x * kScanBlock;
    uint32_t v = 0;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t k = base + u * 256 + threadIdx.x;
        v += k < count ? in[k] : 0u;
    }
    uint32_t total;
    (void)block_exclusive_256(v, lds8, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void k_scan_apply(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                    uint32_t count, const uint32_t* __restrict__ offsets) {
    __shared__ uint32_t vals[kScanBlock];
    __shared__ uint32_t lds8[4];
    const uint32_t base = blockIdx.x * kScanBlock;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t k = base + u * 256 + threadIdx.x;
        vals[u * 256 + threadIdx.x] = k < count ? in[k] : 0u;
    }
    __syncthreads();
    const uint32_t a = vals[4 * threadIdx.x], b = vals[4 * threadIdx.x + 1];
    const uint32_t c = vals[4 * threadIdx.x + 2], d = vals[4 * threadIdx.x + 3];
    uint32_t total;
    const uint32_t pre = offsets[blockIdx.x] + block_exclusive_256(a + b + c + d, lds8, &total);
    __syncthreads();
    vals[4 * threadIdx.x] = pre;
    vals[4 * threadIdx.x + 1] = pre + a;
    vals[4 * threadIdx.x + 2] = pre + a + b;
    vals[4 * threadIdx.x + 3] = pre + a + b + c;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t k = base + u * 256 + threadIdx.x;
        if (k < count) out[k] = vals[u * 256 + threadIdx.x];
    }
}

void SplatWorkspace::release() {
    for (DevBuf* b : {&params, &item_start, &keys, &vals, &sorted, &ranks, &table, &totals, &offsets, &count, &flags, &scan,
                      &attrs, &partials, &crowd, &order, &decoded, &sort_temp})
        b->release();
}

hipError_t launch_splat_2d(const float4* pos, const float* colors, const float* states, uint32_t S,
                           uint32_t count, const npa_splat2d_cfg& cfg, float* image, SplatWorkspace& ws,
                           hipStream_t stream, Profiler* prof, uint32_t per_window, uint32_t windows,
                           uint32_t win_cols) {
    SplatParams P{};
    P.size = (int)cfg.image_size;
    const float fsz = (float)cfg.image_size;
    float sigma = cfg.sigma;  // splat.rs:36-46
    if (cfg.normalize_color) sigma = sigma * fsz * cfg.pixel_size / (cfg.hi - cfg.lo);
    float rf = ceilf(5.0f * sigma);
    if (!(rf >= 1.0f)) rf = rf != rf ? 1.0f : 1.0f;
    if (rf > 4096.0f) rf = 4096.0f;  // windows wider than any supported image are clipped anyway
    P.radius = (int)rf;
    P.k2 = kLog2e / (2.0f * sigma * sigma);
    P.norm_scale = 1.0f;
    if (cfg.normalize_color) {
        const float t = fsz * cfg.pixel_size / (cfg.hi - cfg.lo);
        P.norm_scale = t * t;
    }
    P.lo = cfg.lo;
    P.hi = cfg.hi;
    P.normalize = cfg.normalize_color ? 1 : 0;
    P.y_up = cfg.y_up ? 1 : 0;
    P.S = (int)S;
    if (windows == 0 || win_cols == 0 || per_window == 0) return hipErrorInvalidValue;
    if ((uint64_t)per_window * windows < count) return hipErrorInvalidValue;
    if (!draw_within_limits(P.size, windows, count, P.radius)) return hipErrorInvalidValue;
    hipError_t e;
    DrawPlan draw;
    if (!make_draw_plan(P.size, P.radius, windows, per_window, count, 4, win_cols, &draw)) return hipErrorInvalidValue;
    if ((e = ws.params.reserve((uint64_t)(count ? count : 1) * sizeof(DrawItem))) != hipSuccess) return e;
    if ((e = ws.keys.reserve((uint64_t)(count ? count : 1) * 4)) != hipSuccess) return e;
    if ((e = reserve_draw(draw, ws, stream)) != hipSuccess) return e;
    ProfScope ps(prof, NPA_KERNEL_SPLAT, stream);
    if (count) {
        hipLaunchKernelGGL(k_splat_items, dim3((count + 255) / 256 + (draw.extra ? 1 : 0)), dim3(256), 0, stream, P, pos,
                           colors, states, count, ws.params.as<DrawItem>(), ws.keys.as<uint32_t>(), draw,
                           ws.crowd.as<uint32_t>());
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return launch_draw(draw, ws.params.as<DrawItem>(), ws.keys.as<uint32_t>(), ws, image, stream);
}

// ------------------------------------------------------- projected 3D render
// project_positions (render_loss/projection.rs:11-29) + splat_projected (render_loss/image.rs:18-79)
// for up to kMaxRenderViews views at once: item v * count + n is particle n seen through view v, drawn
// into window v.
constexpr float kRenderEps = 1.0e-8f;

struct RenderParams {
    int size;
    uint32_t count;
    float ws, min_sigma, max_sigma, norm_scale;
    float basis[kMaxRenderViews][9];  // right, up, forward of each view
};

// One thread per particle-view (blockIdx.y is the view, so its basis is a uniform load): dot3 (math.rs:20-22) in
// the reference's order, the depth of projection.rs:20-21, the footprint of image.rs:41-69.
__global__ __launch_bounds__(256) void k_render_items(RenderParams P, const float4* __restrict__ pos,
                                                      const float* __restrict__ colors,
                                                      const float* __restrict__ opacities,
                                                      const float* __restrict__ sigmas, DrawItem* __restrict__ out,
                                                      uint32_t* __restrict__ rects, DrawPlan draw,
                                                      uint32_t* __restrict__ crowd) {
    const float fsz1 = (float)P.size - 1.0f;
    const uint32_t planner = draw.extra ? 1u : 0u;  // the first block finds the crowded groups
    if (blockIdx.x < planner) {
        if (blockIdx.y != 0) return;
        const float to_px = fsz1 / (2.0f * P.ws);
        draw_crowd(draw, crowd, [&](uint32_t v, uint32_t i, float* box) {
            const float* B = P.basis[v];
            const uint32_t n = i - v * P.count;
            const float4 p = pos[n];
            const float r = ceilf(5.0f * clampf_(sigmas[n], P.min_sigma, P.max_sigma));
            const float x = floorf((P.ws + (p.x * B[0] + p.y * B[1] + p.z * B[2])) * to_px);
            const float y = floorf((P.ws - (p.x * B[3] + p.y * B[4] + p.z * B[5])) * to_px);
            box[0] = x - r;
            box[1] = x + r;
            box[2] = y - r;
            box[3] = y + r;
        });
        return;
    }
    const uint32_t n = (blockIdx.x - planner) * blockDim.x + threadIdx.x;
    if (n >= P.count) return;
    const uint32_t v = blockIdx.y;
    const float* B = P.basis[v];
    const float4 p = pos[n];
    const float x = p.x * B[0] + p.y * B[1] + p.z * B[2];
    const float y = p.x * B[3] + p.y * B[4] + p.z * B[5];
    const float f = p.x * B[6] + p.y * B[7] + p.z * B[8];
    const float sigma = fmaxf(clampf_(sigmas[n], P.min_sigma, P.max_sigma), kRenderEps);
    const int64_t radius = f32_to_isize(fmaxf(ceilf(5.0f * sigma), 1.0f));
    DrawItem d;
    d.px = (x + P.ws) / (2.0f * P.ws) * fsz1;
    d.py = (P.ws - y) / (2.0f * P.ws) * fsz1;
    d.k2 = kLog2e / (2.0f * (sigma * sigma));
    const int64_t bx = f32_to_isize(floorf(d.px)), by = f32_to_isize(floorf(d.py));
    const Footprint fp = draw_footprint(d.px, d.py, d.k2, bx, by, radius, P.size);
    d.scale = P.norm_scale * clampf_(opacities[n], 0.0f, 1.0f) / fmaxf(fp.weights, kRenderEps);  // image.rs:67-69
    for (int k = 0; k < 3; ++k) d.c[k] = colors[3 * (uint64_t)n + k];
    d.depth = clampf_(0.5f + 0.5f * f / fmaxf(P.ws, kRenderEps), 0.0f, 1.0f);
    const bool any = fp.rect != kDrawNone;
    d.x0 = any ? (int)(bx - radius) : 0;
    d.y0 = any ? (int)(by - radius) : 0;
    d.span = 2u * (uint32_t)radius;
    d.special = draw_finite(d) ? 0u : 1u;
    const uint64_t i = (uint64_t)v * P.count + n;
    out[i] = d;
    rects[i] = fp.rect;
}

// view_basis (render_loss/projection.rs:31-43) with normalize3 / cross3 (render_loss/math.rs:24-39).
static void render_normalize3(const float v[3], float* out) {
    const float norm = sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    if (norm <= kRenderEps) {
        out[0] = 0.0f;
        out[1] = 0.0f;
        out[2] = 1.0f;
        return;
    }
    for (int k = 0; k < 3; ++k) out[k] = v[k] / norm;
}

static bool render_view_basis(uint32_t view, float* b /* right, up, forward */) {
    static const int axes[3][3] = {{0, 1, 2}, {0, 2, 1}, {1, 2, 0}};  // Xy, Xz, Yz
    if (view < 3) {
        for (int k = 0; k < 9; ++k) b[k] = 0.0f;
        for (int r = 0; r < 3; ++r) b[3 * r + axes[view][r]] = 1.0f;
        return true;
    }
    if (view != NPA_VIEW_ISO) return false;
    const float a[3] = {1.0f, -1.0f, 0.0f}, u[3] = {1.0f, 1.0f, 2.0f};
    render_normalize3(a, b);
    render_normalize3(u, b + 3);
    const float* r = b;
    const float* up = b + 3;
    const float c[3] = {r[1] * up[2] - r[2] * up[1], r[2] * up[0] - r[0] * up[2], r[0] * up[1] - r[1] * up[0]};
    render_normalize3(c, b + 6);
    return true;
}

hipError_t launch_render_views(const float4* pos, const float* colors, const float* opacities, const float* sigmas,
                               uint32_t count, const uint32_t* views, uint32_t nviews, const npa_render_cfg& cfg,
                               float* images, SplatWorkspace& ws, hipStream_t stream, Profiler* prof) {
    if (nviews == 0 || nviews > kMaxRenderViews || !views) return hipErrorInvalidValue;
    RenderParams P{};
    P.size = (int)cfg.image_size;
    P.count = count;
    P.ws = cfg.world_scale;
    P.min_sigma = cfg.min_sigma;
    P.max_sigma = cfg.max_sigma;
    P.norm_scale = 1.0f / (float)(count > 1 ? count : 1);  // image.rs:29
    for (uint32_t v = 0; v < nviews; ++v)
        if (!render_view_basis(views[v], P.basis[v])) return hipErrorInvalidValue;
    const uint64_t items64 = (uint64_t)count * nviews;
    if (items64 >= (1ull << 31) || (uint64_t)count * 16 >= (1ull << 32)) return hipErrorInvalidValue;
    const uint32_t items = (uint32_t)items64;
    // the widest footprint: sigma <= max(max_sigma, EPS)
    const float rmaxf = fmaxf(ceilf(5.0f * fmaxf(cfg.max_sigma, kRenderEps)), 1.0f);
    if (!(rmaxf <= 1024.0f)) return hipErrorInvalidValue;
    if (!draw_within_limits(P.size, nviews, items64, (int)rmaxf)) return hipErrorInvalidValue;
    hipError_t e;
    DrawPlan draw;
    const float typical = fminf(fmaxf(cfg.sigma, cfg.min_sigma), cfg.max_sigma);  // (each particle has its own)
    const int radius = typical > 0.0f ? (int)ceilf(5.0f * typical) : 1;
    if (!make_draw_plan(P.size, radius, nviews, count, items, 5, nviews, &draw)) return hipErrorInvalidValue;
    if ((e = ws.params.reserve((uint64_t)(items ? items : 1) * sizeof(DrawItem))) != hipSuccess) return e;
    if ((e = ws.keys.reserve((uint64_t)(items ? items : 1) * 4)) != hipSuccess) return e;
    if ((e = reserve_draw(draw, ws, stream)) != hipSuccess) return e;
    ProfScope ps(prof, NPA_KERNEL_RENDER, stream);
    if (count) {
        hipLaunchKernelGGL(k_render_items, dim3((count + 255) / 256 + (draw.extra ? 1 : 0), nviews), dim3(256), 0, stream, P,
                           pos, colors, opacities, sigmas, ws.params.as<DrawItem>(), ws.keys.as<uint32_t>(), draw,
                           ws.crowd.as<uint32_t>());
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return launch_draw(draw, ws.params.as<DrawItem>(), ws.keys.as<uint32_t>(), ws, images, stream);
}

// state_tail_render_attributes (render_loss/attributes.rs:15-87): one thread per particle.
__global__ __launch_bounds__(256) void k_render_attrs(const float* __restrict__ states, uint32_t count, uint32_t S,
                                                      npa_render_cfg cfg, float* __restrict__ colors,
                                                      float* __restrict__ opacities, float* __restrict__ sigmas,
                                                      float* __restrict__ derivatives) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const float* s = states + (uint64_t)i * S;
    for (uint32_t k = 0; k < 3; ++k) colors[3 * (uint64_t)i + k] = clampf_(s[S - 3 + k] + 0.5f, 0.0f, 1.0f);
    // growth_3d_material_opacity_channel (rollout/mod.rs:37-45)
    const int ch = S > 8 ? 8 : (S > 3 ? 3 : -1);
    float opacity = 0.95f;  // RENDER_MAX_OPACITY (render_loss.rs:23)
    if (ch >= 0) {
        const float z = s[ch] + cfg.opacity_logit_bias;
        float sg;  // sigmoid (render_loss/math.rs:11-18)
        if (z >= 0.0f) {
            sg = 1.0f / (1.0f + expf(-z));
        } else {
            const float e = expf(z);
            sg = e / (1.0f + e);
        }
        opacity = clampf_(sg, 0.001f, 0.95f);
    }
    opacities[i] = opacity;
    float sigma, derivative = 0.0f;
    switch (cfg.gaussian_decode_mode) {
        case NPA_DECODE_PARTICLE_POINT: sigma = fmaxf(cfg.min_sigma, kRenderEps); break;
        case NPA_DECODE_SH0_LEARNED_SCALE: {
            const float logit = clampf_(s[S - 5], -8.0f, 8.0f);
            const float raw = cfg.sigma * expf(logit);
            sigma = clampf_(raw, cfg.min_sigma, cfg.max_sigma);
            derivative = (raw > cfg.min_sigma && raw < cfg.max_sigma) ? raw : 0.0f;
        } break;
        default: sigma = clampf_(cfg.sigma, cfg.min_sigma, cfg.max_sigma); break;
    }
    sigmas[i] = sigma;
    if (derivatives) derivatives[i] = derivative;
}

hipError_t launch_render_attributes(const float* states, uint32_t count, uint32_t S, const npa_render_cfg& cfg,
                                    float* colors, float* opacities, float* sigmas, float* derivatives,
                                    hipStream_t stream) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_render_attrs, dim3((count + 255) / 256), dim3(256), 0, stream, states, count, S, cfg, colors,
                       opacities, sigmas, derivatives);
    return hipGetLastError();
}


// ------------------------------------------------------------------ oriented Gaussian raster
// The EWA raster of the planar Gaussian export (the image the reference's viewer draws through
// the un-vendored bevy_gaussian_splatting 8.0.1, crates/bevy_automata/src/viewer/cloud.rs:80-97),
// restating the published 3D Gaussian splatting forward pass (Kerbl et al. 2023; EWA projection,
// Zwicker et al. 2001):
//   k_raster_prep      per Gaussian: camera-frame centre, cull, Sigma = R S S^T R^T, the EWA 2D
//                      covariance + 0.3 px^2, its conic, 3-sigma radius, tile rectangle, colour
//                      (spherical harmonics or RGB), the tile count and the depth key;
//   depth order        a stable radix sort of the indices by the positive depth's float bits
//                      (rocPRIM): depth ascending, ties by index;
//   k_raster_lists     up to kRasterListMax Gaussians: a block per group of tiles lists those whose
//                      rectangles touch it, in depth order; nothing is read back;
//   or, for more, k_raster_emit (the (tile, Gaussian) items in depth order, after a prefix of the tile
//                      counts; its total read back to size the item buffers) and a stable key sort by
//                      tile (the hashgrid's counting sort) -> per-tile lists in depth order;
//   k_raster_tiles     one 256-thread block per 16x16 tile; each wave draws an 8x8 block of its pixels
//                      by itself, without barriers: of 64 Gaussians of the list it keeps those that
//                      reach the 1/255 floor on its block (a lane tests one), and each pixel composites
//                      those front to back and stops at the transmittance cut; the wave leaves when
//                      every pixel has stopped.
// Both give a tile the same Gaussians in the same order. 65,536 Gaussians (one more for the items):
// 285 us with lists at 640x480 and 228 us at 1280x1024, 341 and 322 us with items; at 4096x4096, with
// groups of 16x16 tiles, 2,691 and 2,698 us. 16,384 at 1024x768, decode included: 124 and 186 us. Past 16
// bits of Gaussians an entry would double and the lists, each as long as all Gaussians, outgrow the items.
// Bound: vector instructions, about 20 per pixel and kept Gaussian. A 3-sigma tile rectangle holds two
// to three times the pixels that its Gaussian's 1/255 contour does; testing each 8x8 block (about 30
// lane instructions a Gaussian, for the 1,280 it saves) draws 16,384 oriented Gaussians at 1024x768 in
// 71 us where evaluating every listed Gaussian in every pixel took 142 us; the frame is bit-identical.
struct RasterParams {
    float view[12];
    float fx, fy, cx, cy, limx, limy, near_plane, far_plane;
    float campos[3];
    uint32_t width, height, tiles_x, tiles_y, count, K, sh_degree, color_mode;
    uint32_t stride;  // coefficient triples per Gaussian in the input (>= K)
};

struct alignas(16) RasterSplat {  // 48 bytes
    float mx, my, qa, qb;  // qa, qb, qc: the conic scaled by -log2(e)/2, -log2(e), -log2(e)/2
    float qc, opacity, r, g;
    float b;
    uint32_t rx;  // tile columns [rx & 0xffff, rx >> 16)
    uint32_t ry;  // tile rows
    uint32_t pad;
};

constexpr uint32_t kRasterMaxAxis = 16384;  // pixels per axis: tile indices fit 16 bits
constexpr uint32_t kDepthCulled = 0x7f800000u;  // +inf: sorts after every live depth

__device__ __forceinline__ float raster_clamp(float v, float lo, float hi) { return v < lo ? lo : (v > hi ? hi : v); }

__global__ __launch_bounds__(256) void k_raster_prep(RasterParams P, const float4* __restrict__ pv,
                                                     const float* __restrict__ sh, const float4* __restrict__ rot,
                                                     const float4* __restrict__ so, RasterSplat* __restrict__ out,
                                                     uint32_t* __restrict__ ntiles, uint2* __restrict__ rects,
                                                     uint32_t* __restrict__ dkey) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.count) return;
    if (rects) rects[i] = make_uint2(0u, 0u);
    else ntiles[i] = 0;
    dkey[i] = kDepthCulled;
    const float4 p = pv[i];
    if (!(p.w > 0.0f)) return;
    const float* V = P.view;
    const float vx = V[0] * p.x + V[1] * p.y + V[2] * p.z + V[3];
    const float vy = V[4] * p.x + V[5] * p.y + V[6] * p.z + V[7];
    const float vz = V[8] * p.x + V[9] * p.y + V[10] * p.z + V[11];
    const float tx = vx, ty = -vy, tz = -vz;  // x right, y down, z forward
    if (!(tz > P.near_plane) || !(tz <= P.far_plane)) return;
    const float4 q4 = rot[i];
    float qw = q4.x, qx = q4.y, qy = q4.z, qz = q4.w;
    const float qn = sqrtf(qw * qw + qx * qx + qy * qy + qz * qz);
    if (qn > 0.0f && qn < INFINITY) {
        qw = qw / qn; qx = qx / qn; qy = qy / qn; qz = qz / qn;
    } else {
        qw = 1.0f; qx = qy = qz = 0.0f;
    }
    const float R[3][3] = {
        {1.0f - 2.0f * (qy * qy + qz * qz), 2.0f * (qx * qy - qw * qz), 2.0f * (qx * qz + qw * qy)},
        {2.0f * (qx * qy + qw * qz), 1.0f - 2.0f * (qx * qx + qz * qz), 2.0f * (qy * qz - qw * qx)},
        {2.0f * (qx * qz - qw * qy), 2.0f * (qy * qz + qw * qx), 1.0f - 2.0f * (qx * qx + qy * qy)}};
    const float4 s4 = so[i];
    const float sc[3] = {s4.x, s4.y, s4.z};
    float M[3][3], S[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) M[r][c] = R[r][c] * sc[c];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) S[r][c] = M[r][0] * M[c][0] + M[r][1] * M[c][1] + M[r][2] * M[c][2];
    const float W[3][3] = {{V[0], V[1], V[2]}, {-V[4], -V[5], -V[6]}, {-V[8], -V[9], -V[10]}};
    const float jx = raster_clamp(tx / tz, -P.limx, P.limx) * tz;
    const float jy = raster_clamp(ty / tz, -P.limy, P.limy) * tz;
    const float J[2][3] = {{P.fx / tz, 0.0f, -(P.fx * jx) / (tz * tz)}, {0.0f, P.fy / tz, -(P.fy * jy) / (tz * tz)}};
    float T[2][3], U[2][3];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) T[r][c] = J[r][0] * W[0][c] + J[r][1] * W[1][c] + J[r][2] * W[2][c];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) U[r][c] = T[r][0] * S[0][c] + T[r][1] * S[1][c] + T[r][2] * S[2][c];
    const float a = (U[0][0] * T[0][0] + U[0][1] * T[0][1] + U[0][2] * T[0][2]) + 0.3f;
    const float b = U[0][0] * T[1][0] + U[0][1] * T[1][1] + U[0][2] * T[1][2];
    const float c = (U[1][0] * T[1][0] + U[1][1] * T[1][1] + U[1][2] * T[1][2]) + 0.3f;
    const float det = a * c - b * b;
    if (!(det > 0.0f) || !(det < INFINITY)) return;
    const float mid = 0.5f * (a + c);
    const float lam = mid + sqrtf(fmaxf(0.1f, mid * mid - det));
    const float radius = ceilf(3.0f * sqrtf(lam));
    const float mx = P.cx + P.fx * tx / tz;
    const float my = P.cy + P.fy * ty / tz;
    if (!(fabsf(mx) < 1e30f) || !(fabsf(my) < 1e30f) || !(radius < 1e30f)) return;
    const uint32_t x0 = (uint32_t)raster_clamp(floorf((mx - radius) / 16.0f), 0.0f, (float)P.tiles_x);
    const uint32_t x1 = (uint32_t)raster_clamp(floorf((mx + radius) / 16.0f) + 1.0f, 0.0f, (float)P.tiles_x);
    const uint32_t y0 = (uint32_t)raster_clamp(floorf((my - radius) / 16.0f), 0.0f, (float)P.tiles_y);
    const uint32_t y1 = (uint32_t)raster_clamp(floorf((my + radius) / 16.0f) + 1.0f, 0.0f, (float)P.tiles_y);
    if (x0 >= x1 || y0 >= y1) return;
    RasterSplat o;
    o.mx = mx;
    o.my = my;
    const float L = 1.4426950408889634f;
    o.qa = (c / det) * (-0.5f * L);
    o.qb = (-b / det) * -L;
    o.qc = (a / det) * (-0.5f * L);
    o.opacity = s4.w;
    o.rx = x0 | (x1 << 16);
    o.ry = y0 | (y1 << 16);
    o.pad = 0;
    const float* coef = sh + (uint64_t)i * P.stride * 3;
    if (P.color_mode == NPA_RASTER_COLOR_RGB) {
        o.r = coef[0];
        o.g = coef[1];
        o.b = coef[2];
    } else {
        float d[3] = {p.x - P.campos[0], p.y - P.campos[1], p.z - P.campos[2]};
        const float dn = sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
#pragma unroll
        for (int k = 0; k < 3; ++k) d[k] = dn > 0.0f ? d[k] / dn : 0.0f;
        // real spherical harmonics, bands 0..3, in the 3DGS sign convention (Condon-Shortley phase)
        const float x = d[0], y = d[1], z = d[2];
        float basis[16];
        basis[0] = 0.28209479177387814f;
        if (P.sh_degree > 0) {
            basis[1] = -0.4886025119029199f * y;
            basis[2] = 0.4886025119029199f * z;
            basis[3] = -0.4886025119029199f * x;
        }
        if (P.sh_degree > 1) {
            const float xx = x * x, yy = y * y, zz = z * z;
            basis[4] = 1.0925484305920792f * (x * y);
            basis[5] = -1.0925484305920792f * (y * z);
            basis[6] = 0.31539156525252005f * (2.0f * zz - xx - yy);
            basis[7] = -1.0925484305920792f * (x * z);
            basis[8] = 0.5462742152960396f * (xx - yy);
            if (P.sh_degree > 2) {
                basis[9] = -0.5900435899266435f * y * (3.0f * xx - yy);
                basis[10] = 2.890611442640554f * (x * y) * z;
                basis[11] = -0.4570457994644658f * y * (4.0f * zz - xx - yy);
                basis[12] = 0.3731763325901154f * z * (2.0f * zz - 3.0f * xx - 3.0f * yy);
                basis[13] = -0.4570457994644658f * x * (4.0f * zz - xx - yy);
                basis[14] = 1.445305721320277f * z * (xx - yy);
                basis[15] = -0.5900435899266435f * x * (xx - 3.0f * yy);
            }
        }
        float rgb[3];
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            float acc = 0.0f;
            for (uint32_t k = 0; k < P.K; ++k) acc += basis[k] * coef[k * 3 + ch];
            acc += 0.5f;
            rgb[ch] = acc > 0.0f ? acc : 0.0f;
        }
        o.r = rgb[0];
        o.g = rgb[1];
        o.b = rgb[2];
    }
    out[i] = o;
    if (rects) rects[i] = make_uint2(o.rx, o.ry);
    else ntiles[i] = (x1 - x0) * (y1 - y0);
    dkey[i] = __float_as_uint(tz);
}

// ---- Up to kRasterListMax Gaussians: one list per group of (1 << shift)^2 tiles.
constexpr uint32_t kRasterListMax = 65536;  // an entry holds its Gaussian in 16 bits
constexpr uint32_t kRasterGroups = 512;     // at most this many groups

__global__ __launch_bounds__(256) void k_raster_order_rects(const uint2* __restrict__ rects,
                                                            const uint32_t* __restrict__ order, uint32_t count,
                                                            uint2* __restrict__ out) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < count) out[j] = rects[order[j]];
}

// One block per group: the Gaussians whose rectangles touch it, in depth order, at lists[group * count].
// An entry is the Gaussian << 16 | the group's tiles that it covers as four inclusive 4-bit bounds
// (x first, x last, y first, y last). Each wave tests a consecutive range of the depth order and
// keeps the hits as bits, then writes its entries after those of the waves before it.
// Bound: the latency of a wave's loads, kRasterAhead in flight: 16 waves test 16,384 in four batches each
// (13 us for 192 groups, against 45 us for the counts, their prefix and total, the items and their sort).
constexpr int kRasterAhead = 4;

__global__ __launch_bounds__(1024) void k_raster_lists(const uint2* __restrict__ orects,
                                                       const uint32_t* __restrict__ order, uint32_t count,
                                                       uint32_t shift, uint32_t groups_x, uint32_t* __restrict__ lists,
                                                       uint32_t* __restrict__ counts) {
    __shared__ uint64_t masks[kRasterListMax / 64];
    __shared__ uint32_t wave_hits[16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t gx = (blockIdx.x % groups_x) << shift, gy = (blockIdx.x / groups_x) << shift, side = 1u << shift;
    const uint32_t chunks = (count + 63) / 64, per = (chunks + 15) / 16;
    const uint32_t c0 = min(wave * per, chunks), c1 = min(c0 + per, chunks);
    uint32_t hits = 0;
    for (uint32_t c = c0; c < c1; c += kRasterAhead) {
        uint2 r[kRasterAhead];
#pragma unroll
        for (int u = 0; u < kRasterAhead; ++u) {
            const uint32_t j = (c + u) * 64 + lane;
            r[u] = c + u < c1 && j < count ? orects[j] : make_uint2(0u, 0u);
        }
#pragma unroll
        for (int u = 0; u < kRasterAhead; ++u) {
            const uint64_t m = __ballot((r[u].x & 0xffffu) < gx + side && (r[u].x >> 16) > gx &&
                                        (r[u].y & 0xffffu) < gy + side && (r[u].y >> 16) > gy);
            if (c + u < c1 && lane == 0) masks[c + u] = m;
            hits += (uint32_t)__popcll(m);
        }
    }
    if (lane == 0) wave_hits[wave] = hits;
    __syncthreads();
    uint32_t at = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
        at += w < wave ? wave_hits[w] : 0u;
        total += wave_hits[w];
    }
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
    uint32_t* list = lists + (uint64_t)blockIdx.x * count;
    for (uint32_t c = c0; c < c1; ++c) {
        const uint64_t m = masks[c];
        if ((m >> lane) & 1ull) {  // j < count: only such lanes hit
            const uint32_t j = c * 64 + lane;
            const uint2 r = orects[j];
            const uint32_t xa = max(r.x & 0xffffu, gx) - gx, xb = min(r.x >> 16, gx + side) - gx - 1;
            const uint32_t ya = max(r.y & 0xffffu, gy) - gy, yb = min(r.y >> 16, gy + side) - gy - 1;
            list[at + (uint32_t)__popcll(m & lanemask_lt())] = (order[j] << 16) | xa | (xb << 4) | (ya << 8) | (yb << 12);
        }
        at += (uint32_t)__popcll(m);
    }
}

// ---- More Gaussians: (tile, Gaussian) items, sorted by tile.

__global__ __launch_bounds__(256) void k_raster_gather_counts(const uint32_t* __restrict__ ntiles,
                                                              const uint32_t* __restrict__ order, uint32_t count,
                                                              uint32_t* __restrict__ out) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < count) out[j] = ntiles[order[j]];
}

// The 64-bit sum of the tile counts (the 32-bit scan total can wrap).
__global__ __launch_bounds__(1024) void k_raster_sum64(const uint32_t* __restrict__ in, uint32_t count,
                                                       unsigned long long* __restrict__ total) {
    __shared__ unsigned long long lds[16];
    unsigned long long s = 0;
    for (uint32_t k = threadIdx.x; k < count; k += blockDim.x) s += in[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (uint32_t w = 0; w < blockDim.x / 64; ++w) t += lds[w];
        *total = t;
    }
}

// kEmitLanes lanes per Gaussian write its (tile, Gaussian) items interleaved, row-major over its
// tile rectangle from start[j].
constexpr uint32_t kEmitLanes = 8;

__global__ __launch_bounds__(256) void k_raster_emit(RasterParams P, const RasterSplat* __restrict__ sp,
                                                     const uint32_t* __restrict__ order,
                                                     const uint32_t* __restrict__ start, uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t j = t / kEmitLanes;
    const uint32_t sub = (uint32_t)(t % kEmitLanes);
    if (j >= P.count) return;
    const uint32_t begin = start[j], end = start[j + 1];
    if (begin + sub >= end) return;
    const uint32_t g = order[j];
    const uint32_t rx = sp[g].rx, ry = sp[g].ry;
    const uint32_t x0 = rx & 0xffffu, x1 = rx >> 16, y0 = ry & 0xffffu;
    const uint32_t w = x1 - x0;  // >= 1: the Gaussian has items
    uint32_t x = x0 + sub, y = y0;
    while (x >= x1) {
        x -= w;
        ++y;
    }
    for (uint32_t k = begin + sub; k < end; k += kEmitLanes) {
        keys[k] = y * P.tiles_x + x;
        vals[k] = g;
        x += kEmitLanes;
        while (x >= x1) {
            x -= w;
            ++y;
        }
    }
}

// Whether a Gaussian can reach the 1/255 floor on an 8x8 pixel block whose first pixel centre is
// (x, y): the largest exponent over the block, from the edges facing the mean, against
// log2(1 / (255 opacity)).  False only where every pixel would drop it: the slack is over ten times
// the rounding of the pixels' own exponents, and a conic near singular (where the edges that do not
// face the mean could hold the maximum), an infinity or a NaN is kept for the pixels to decide.
__device__ __forceinline__ bool raster_reaches(const float4& A, const float4& B, float x, float y) {
    const float x0 = A.x - (x + 7.0f), x1 = A.x - x, y0 = A.y - (y + 7.0f), y1 = A.y - y;
    const float nx = __builtin_amdgcn_fmed3f(0.0f, x0, x1), ny = __builtin_amdgcn_fmed3f(0.0f, y0, y1);
    const float ax = fmaxf(fabsf(x0), fabsf(x1)), ay = fmaxf(fabsf(y0), fabsf(y1));
    const float qa = A.z, qb = A.w, qc = B.x;
    // along the edge dx = nx the exponent is largest at dy = -qb nx / 2 qc, along dy = ny likewise
    const float ey = __builtin_amdgcn_fmed3f(-0.5f * qb * nx * __builtin_amdgcn_rcpf(qc), y0, y1);
    const float ex = __builtin_amdgcn_fmed3f(-0.5f * qb * ny * __builtin_amdgcn_rcpf(qa), x0, x1);
    const float pa = qa * nx * nx + qb * nx * ey + qc * ey * ey;
    const float pb = qa * ex * ex + qb * ex * ny + qc * ny * ny;
    const float size = fabsf(qa) * ax * ax + fabsf(qb) * ax * ay + fabsf(qc) * ay * ay;
    const float least = __builtin_amdgcn_logf(__builtin_amdgcn_rcpf(255.0f * B.y)) - (1e-3f + 1e-5f * size);
    const bool sound = 4.0f * qa * qc - qb * qb > 4e-3f * qa * qc;  // qa, qc < 0
    const bool inside = nx == 0.0f && ny == 0.0f;
    return !(sound && !inside && pa < least && pb < least);
}

// LISTS: `lists` holds the groups' entries (k_raster_lists), of which a wave keeps its tile's; otherwise
// `lists` holds the items' Gaussians sorted by tile, from offsets[tile].
template <bool LISTS>
__global__ __launch_bounds__(256) void k_raster_tiles(RasterParams P, const RasterSplat* __restrict__ sp,
                                                      const uint32_t* __restrict__ offsets,
                                                      const uint32_t* __restrict__ lists, uint32_t shift,
                                                      uint32_t groups_x, float4* __restrict__ image) {
    __shared__ float4 la[4][68], lb[4][68];
    __shared__ float lc[4][68];
    __shared__ uint32_t waiting_g[LISTS ? 4 : 1][LISTS ? 128 : 1];
    const uint32_t tile = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t tx = tile % P.tiles_x, ty = tile / P.tiles_x;
    const uint32_t bx = tx * 16 + (wave & 1) * 8, by = ty * 16 + (wave >> 1) * 8;
    const uint32_t px = bx + (lane & 7), py = by + (lane >> 3);
    const bool inside = px < P.width && py < P.height;
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float bxc = (float)bx + 0.5f, byc = (float)by + 0.5f;
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    uint32_t pos, end, lx = 0, ly = 0;  // of the list; the tile within its group
    if constexpr (LISTS) {
        const uint32_t group = (ty >> shift) * groups_x + (tx >> shift);
        pos = 0;
        end = offsets[group];
        lists += (uint64_t)group * P.count;
        lx = tx & ((1u << shift) - 1);
        ly = ty & ((1u << shift) - 1);
    } else {
        pos = offsets[tile];
        end = offsets[tile + 1];
    }
    uint32_t ahead = pos + lane < end ? lists[pos + lane] : 0u;  // the list's next 64 entries
    uint32_t waiting = 0;
    // the next up to 64 Gaussians of the tile: lane l's in g for l < the count returned
    auto take = [&](uint32_t& g) {
        if constexpr (LISTS) {
            while (waiting < 64 && pos < end) {
                const uint32_t e = ahead;
                const bool hit = pos + lane < end && lx >= (e & 15u) && lx <= ((e >> 4) & 15u) &&
                                 ly >= ((e >> 8) & 15u) && ly <= ((e >> 12) & 15u);
                pos += 64;
                if (pos + lane < end) ahead = lists[pos + lane];
                const uint64_t m = __ballot(hit);
                if (hit) waiting_g[wave][waiting + (uint32_t)__popcll(m & lanemask_lt())] = e >> 16;
                waiting += (uint32_t)__popcll(m);
            }
            wave_fence();
            const uint32_t n = min(waiting, 64u);
            g = waiting_g[wave][lane];
            const uint32_t rest = waiting_g[wave][64 + lane];
            waiting -= n;
            wave_fence();
            if (lane < waiting) waiting_g[wave][lane] = rest;
            wave_fence();
            return n;
        } else {
            const uint32_t n = min(end - pos, 64u);
            g = ahead;
            pos += n;
            if (pos + lane < end) ahead = lists[pos + lane];
            return n;
        }
    };
    float T = 1.0f, cr = 0.0f, cg = 0.0f, cb = 0.0f;
    bool done = !inside;
    float4 A = make_float4(0.f, 0.f, 0.f, 0.f), B = A;
    float C = 0.0f;
    auto load = [&](uint32_t g) {
        const float4* s4 = reinterpret_cast<const float4*>(sp + g);
        A = s4[0];
        B = s4[1];
        C = s4[2].x;
    };
    uint32_t g;
    uint32_t have = take(g);
    if (lane < have) load(g);
    while (have && !__all(done)) {
        const bool keep = lane < have && raster_reaches(A, B, bxc, byc);
        const uint64_t kept = __ballot(keep);
        const uint32_t n = (uint32_t)__popcll(kept);
        if (keep) {
            const uint32_t at = (uint32_t)__popcll(kept & lanemask_lt());
            la[wave][at] = A;
            lb[wave][at] = B;
            lc[wave][at] = C;
        }
        if (lane < 4) {  // opacity 0: nothing drawn
            la[wave][n + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
            lb[wave][n + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
            lc[wave][n + lane] = 0.0f;
        }
        have = take(g);  // the next round's records are in flight while this one is drawn
        if (lane < have) load(g);
        wave_fence();
        // Branch-free: every lane evaluates every entry and the tests become selects (the same
        // comparisons, so NaN behaves as in a branching loop); a stopped lane keeps its values.
        for (uint32_t u0 = 0; u0 < n; u0 += 4) {
#pragma unroll
            for (uint32_t du = 0; du < 4; ++du) {
                const float4 a = la[wave][u0 + du], b = lb[wave][u0 + du];  // (mx, my, qa, qb), (qc, opacity, r, g)
                const float c = lc[wave][u0 + du];
                const float dx = a.x - pxc, dy = a.y - pyc;
                // power * log2(e), with the oracle's fused operations
                const float p2 = __builtin_fmaf(a.z * dx, dx, __builtin_fmaf(b.x * dy, dy, a.w * dx * dy));
                // the hardware 2^x: below 2^-126 alpha is far under the 1/255 floor either way
                const float alpha = fminf(0.99f, b.y * __builtin_amdgcn_exp2f(p2));
                const float next = T * (1.0f - alpha);
                const bool ok = !done && !(p2 > 0.0f) && !(alpha < 1.0f / 255.0f);
                const bool stop = ok && next < 0.0001f;
                const bool apply = ok && !stop;
                const float wgt = alpha * T;
                cr = apply ? __builtin_fmaf(b.z, wgt, cr) : cr;
                cg = apply ? __builtin_fmaf(b.w, wgt, cg) : cg;
                cb = apply ? __builtin_fmaf(c, wgt, cb) : cb;
                T = apply ? next : T;
                done = done || stop;
            }
            if (__all(done)) break;
        }
        wave_fence();
    }
    if (inside) image[(uint64_t)py * P.width + px] = make_float4(cr, cg, cb, 1.0f - T);
}

hipError_t launch_raster_gaussians(const float4* pv, const float* sh, const float4* rot, const float4* so,
                                   uint32_t count, const npa_raster_camera& cam, float* image, SplatWorkspace& ws,
                                   hipStream_t stream, Profiler* prof, uint32_t coef_stride) {
    const uint32_t K = (cam.sh_degree + 1) * (cam.sh_degree + 1);
    if (cam.width == 0 || cam.height == 0 || cam.width > kRasterMaxAxis || cam.height > kRasterMaxAxis ||
        cam.sh_degree > 3 || count >= (1u << 31) || (coef_stride != 0 && coef_stride < K))
        return hipErrorInvalidValue;
    RasterParams P{};
    for (int k = 0; k < 12; ++k) P.view[k] = cam.view[k];
    P.fx = cam.fx;
    P.fy = cam.fy;
    P.cx = cam.cx;
    P.cy = cam.cy;
    P.limx = 1.3f * fmaxf(cam.cx, (float)cam.width - cam.cx) / cam.fx;
    P.limy = 1.3f * fmaxf(cam.cy, (float)cam.height - cam.cy) / cam.fy;
    P.near_plane = cam.near_plane;
    P.far_plane = cam.far_plane;
    for (int k = 0; k < 3; ++k)  // camera centre -R^T t
        P.campos[k] = -(cam.view[k] * cam.view[3] + cam.view[4 + k] * cam.view[7] + cam.view[8 + k] * cam.view[11]);
    P.width = cam.width;
    P.height = cam.height;
    P.tiles_x = (cam.width + 15) / 16;
    P.tiles_y = (cam.height + 15) / 16;
    P.count = count;
    P.K = K;
    P.stride = coef_stride ? coef_stride : K;
    P.sh_degree = cam.sh_degree;
    P.color_mode = cam.color_mode;
    const uint32_t ntile_total = P.tiles_x * P.tiles_y;
    if (ntile_total > 65536) return hipErrorInvalidValue;  // the key sort's bin limit
    const uint64_t n1 = count ? count : 1;
    hipError_t e;
#define NPA_RES(buf, n) \
    if ((e = (buf).reserve((size_t)(n))) != hipSuccess) return e;
    NPA_RES(ws.params, n1 * sizeof(RasterSplat));
    NPA_RES(ws.item_start, (4 * n1 + 1) * 4);  // ntiles, depth keys, ordered counts, starts (+1)
    NPA_RES(ws.order, n1 * 4);
    NPA_RES(ws.keys, n1 * 4);
    // Groups of the smallest size that gives at most kRasterGroups of them (16x16 tiles at the image
    // limit, 256 of those), so that a block per group about fills the chip. Lists hold up to
    // kRasterListMax Gaussians, and take no more items than the sorted way accepts.
    uint32_t shift = 0;
    auto groups_along = [&](uint32_t tiles) { return (tiles + (1u << shift) - 1) >> shift; };
    while (groups_along(P.tiles_x) * groups_along(P.tiles_y) > kRasterGroups && shift < 4) ++shift;
    const uint32_t groups_x = groups_along(P.tiles_x), groups = groups_x * groups_along(P.tiles_y);
    const bool lists = count && count <= kRasterListMax && groups <= kRasterGroups &&
                       (uint64_t)count * ntile_total < (1ull << 31);
    uint2 *rects = nullptr, *orects = nullptr;
    if (lists) {
        NPA_RES(ws.vals, n1 * 8);
        NPA_RES(ws.sorted, n1 * 8);
        NPA_RES(ws.table, (uint64_t)groups * count * 4);
        NPA_RES(ws.totals, (uint64_t)groups * 4);
        rects = ws.vals.as<uint2>();
        orects = ws.sorted.as<uint2>();
    } else {
        NPA_RES(ws.offsets, ((uint64_t)ntile_total + 1) * 4);
        NPA_RES(ws.count, 64);
        NPA_RES(ws.scan, (2 * (n1 / kScanBlock + 1) + 2) * 4);
    }
    ProfScope ps(prof, NPA_KERNEL_RASTER, stream);
    RasterSplat* sp = ws.params.as<RasterSplat>();
    uint32_t* ntiles = ws.item_start.as<uint32_t>();
    uint32_t* dkey = ntiles + n1;
    uint32_t* ocounts = dkey + n1;
    uint32_t* start = ocounts + n1;  // n1 + 1 entries
    uint32_t* ord_a = ws.order.as<uint32_t>();
    unsigned long long* d_total64 = reinterpret_cast<unsigned long long*>(ws.count.as<uint32_t>() + 2);
    if (count) {
        hipLaunchKernelGGL(k_raster_prep, dim3((count + 255) / 256), dim3(256), 0, stream, P, pv, sh, rot, so, sp,
                           ntiles, rects, dkey);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    // depth order: stable radix sort of the indices by the depth keys' bits 0-30 (non-negative floats)
    if ((e = sort_index_by_key(dkey, ws.keys.as<uint32_t>(), ord_a, count, 31, ws.sort_temp, stream)) != hipSuccess)
        return e;
    const uint32_t* order = ord_a;
    if (lists) {
        hipLaunchKernelGGL(k_raster_order_rects, dim3((count + 255) / 256), dim3(256), 0, stream, rects, order, count,
                           orects);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(k_raster_lists, dim3(groups), dim3(1024), 0, stream, orects, order, count, shift, groups_x,
                           ws.table.as<uint32_t>(), ws.totals.as<uint32_t>());
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(k_raster_tiles<true>, dim3(ntile_total), dim3(256), 0, stream, P, sp,
                           ws.totals.as<uint32_t>(), ws.table.as<uint32_t>(), shift, groups_x,
                           reinterpret_cast<float4*>(image));
        return hipGetLastError();
    }
    if (count) {
        hipLaunchKernelGGL(k_raster_gather_counts, dim3((count + 255) / 256), dim3(256), 0, stream, ntiles, order,
                           count, ocounts);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    {  // start = exclusive prefix of the ordered counts; start[count] = total
        const uint32_t nb = (count + kScanBlock - 1) / kScanBlock;
        uint32_t* sums = ws.scan.as<uint32_t>();
        if (nb) {
            hipLaunchKernelGGL(k_scan_partials, dim3(nb), dim3(256), 0, stream, ocounts, count, sums);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k_scan_1block, dim3(1), dim3(1024), 0, stream, sums, sums + nb + 1, nb, start + count);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (nb) {
            hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(256), 0, stream, ocounts, start, count, sums + nb + 1);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k_raster_sum64, dim3(1), dim3(1024), 0, stream, ocounts, count, d_total64);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    unsigned long long total = 0;
    if ((e = hipMemcpyAsync(&total, d_total64, 8, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
    if (total >= (1ull << 31)) return hipErrorInvalidValue;  // more (tile, Gaussian) items than the sort takes
    const uint32_t items = (uint32_t)total;
    HashgridPlan plan;
    if (!make_key_sort_plan(items, ntile_total, &plan)) return hipErrorInvalidValue;
    const uint64_t i1 = items ? items : 1;
    NPA_RES(ws.keys, std::max(i1, n1) * 4);
    NPA_RES(ws.vals, i1 * 4);
    NPA_RES(ws.sorted, i1 * 4);
    NPA_RES(ws.ranks, i1 * 4);
    NPA_RES(ws.table, plan.table_entries * 4);
    NPA_RES(ws.totals, (uint64_t)ntile_total * 4);
    NPA_RES(ws.flags, 64);
#undef NPA_RES
    if (count) {
        hipLaunchKernelGGL(k_raster_emit, dim3((uint32_t)(((uint64_t)count * kEmitLanes + 255) / 256)), dim3(256), 0,
                           stream, P, sp, order, start, ws.keys.as<uint32_t>(), ws.vals.as<uint32_t>());
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    // stable counting sort of the items by tile (the scan wrote the item count to start[count])
    e = launch_key_sort(plan, ws.keys.as<uint32_t>(), ws.vals.as<uint32_t>(), start + count, items,
                        ws.ranks.as<uint32_t>(), ws.table.as<uint32_t>(), ws.totals.as<uint32_t>(),
                        ws.offsets.as<uint32_t>(), ws.sorted.as<uint32_t>(), ws.flags.as<uint32_t>(), stream);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_raster_tiles<false>, dim3(ntile_total), dim3(256), 0, stream, P, sp,
                       ws.offsets.as<uint32_t>(), ws.sorted.as<uint32_t>(), 0u, 0u, reinterpret_cast<float4*>(image));
    return hipGetLastError();
}

}  // namespace npa
