// npa_mlp.hip - the update MLP on explicit feature rows (gfx950): forward_from_features_with_eps for
// a caller's rows, and the MLP + motion scaling + 3D gates + masked Euler step of the shapes the fused
// update kernel does not serve (state widths other than 9-16, more than 128 hidden units).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "npa_internal.hpp"

namespace npa {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMlpRows = 16;  // feature rows per block
constexpr int kMlpOuts = 35;  // most outputs: 3 + 32

// Weight layout: w1 as [ceil(F / 4)][HC][4] (lane's hidden unit, four consecutive features: one
// 16-byte load), b1 [HC], w2 as [ceil(H / 4)][OC][4], b2 [OC]; HC = H rounded up to 64, OC = outputs
// rounded up to 16, zeros in every padded place.
struct MlpLayout {
    uint32_t K4, HC, H4, OC;
    uint64_t b1, w2, b2, total;
};
__host__ __device__ inline MlpLayout mlp_layout(uint32_t F, uint32_t H, uint32_t O) {
    MlpLayout l;
    l.K4 = (F + 3) / 4;
    l.HC = (H + 63) / 64 * 64;
    l.H4 = (H + 3) / 4;
    l.OC = (O + 15) / 16 * 16;
    l.b1 = (uint64_t)l.K4 * l.HC * 4;
    l.w2 = l.b1 + l.HC;
    l.b2 = l.w2 + (uint64_t)l.H4 * l.OC * 4;
    l.total = l.b2 + l.OC;
    return l;
}

__global__ __launch_bounds__(256) void k_mlp_weights(uint32_t F, uint32_t H, uint32_t O, const float* __restrict__ w1,
                                                     const float* __restrict__ b1, const float* __restrict__ w2,
                                                     const float* __restrict__ b2, float* __restrict__ wp) {
    const MlpLayout l = mlp_layout(F, H, O);
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < l.total; t += (uint64_t)gridDim.x * blockDim.x) {
        float v = 0.0f;
        if (t < l.b1) {
            const uint32_t i = (uint32_t)(t & 3), h = (uint32_t)((t >> 2) % l.HC), k = (uint32_t)((t >> 2) / l.HC) * 4 + i;
            if (h < H && k < F) v = w1[(uint64_t)h * F + k];
        } else if (t < l.w2) {
            const uint32_t h = (uint32_t)(t - l.b1);
            if (h < H) v = b1[h];
        } else if (t < l.b2) {
            const uint64_t r = t - l.w2;
            const uint32_t i = (uint32_t)(r & 3), o = (uint32_t)((r >> 2) % l.OC), h = (uint32_t)((r >> 2) / l.OC) * 4 + i;
            if (o < O && h < H) v = w2[(uint64_t)o * H + h];
        } else {
            const uint32_t o = (uint32_t)(t - l.b2);
            if (o < O) v = b2[o];
        }
        wp[t] = v;
    }
}

// Element k of a float4 (k a constant once the loops are unrolled).
__device__ __forceinline__ float f4(const float4& v, int k) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; }

// forward_update_from_features model.rs:900-940 for 16 rows per block: layer 1, ReLU and layer 2, each
// output sum starting from its bias and adding its products in index order.
//
// The weights are either packed (mlp_layout; a state's or a step's, laid out once) or raw: the caller's
// w1 [H][F], w2 [O][H], read without a workspace, so that forward_from_features stays a single launch
// that owns no memory. A wave brings its 64 units' raw weights through its own LDS tile, 16 features at
// a time (a lane reading its own unit's row from memory would touch 64 cache lines a load).
//
// Engine 0 rounds every product and every sum as the reference does. The products come from the
// matrix cores: v_mfma_f32_16x16x1_4b_f32 with a -0.0 accumulator returns a * b rounded once (K = 1:
// one product per element, and x + -0.0 = x), 16 rows x 64 hidden units per instruction, and the
// vector ALUs add them to the sums in feature order. That is one v_add per 64 products where the
// vector ALUs alone need a v_mul as well, and an operand of each side is loaded once per 64 x 16
// products. Layer 2 does the same with v_mfma_f32_4x4x1_16b_f32, whose 16 blocks are 4 row groups x
// 4 output groups (16 rows x 16 outputs). Engine 1 accumulates on the matrix cores
// (v_mfma_f32_16x16x4_f32, four features at a time).
//
// Bound: the ordered adds, one wave instruction per 64 of them, on up to 1,024 SIMDs: 16 rows x 64
// units x F features take 64 F cycles. 16 rows per block (rather than a row per lane, 64 rows) keep
// small systems on every CU: 4,096 rows are 256 blocks. Measured: forward_from_features of 32,008 rows,
// F = 66, H = 128, O = 18: 1,304 us with a thread per row reading features and weights at a stride ->
// 34.5 us; the step's MLP for 4,096 rows, F = 123, H = 256, O = 27: 67.5 us with 64 rows per block and
// v_mul + v_add -> 21.3 us.
//
// The hidden units are taken in chunks of 64 per wave, so LDS does not grow with H.
//
//   wave w of layer 1: rows 0-15, units [chunk + 64 w, + 64): lane l feeds A = row l % 16 and B = unit
//   l, and holds in register r the sum of row 4 (l / 16) + r % 4, unit 16 (r / 4) + l % 16
//   wave w of layer 2: output groups w, w + NW, ... of 16: lane l (block l / 4 = rg + 4 og) feeds A =
//   row 4 rg + l % 4 and B = output 4 og + l % 4, and holds in register r row 4 rg + r, output
//   4 og + l % 4
struct RawWeights {
    const float* w1;
    const float* b1;
    const float* w2;
    const float* b2;
};
constexpr uint32_t kTileK = 16, kTileS = kTileK + 4;  // raw w1 tile of a wave: [64 units][kTileS]

// Makes the wave's LDS writes visible to its other lanes (a wave's LDS operations are performed in
// order; the barrier keeps the compiler from moving them across).
__device__ __forceinline__ void mlp_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Adds features 4 k .. 4 k + N - 1 of 16 rows x 64 units to the sums, in order: the next product is
// on the matrix cores while the last one is added.
template <int N>
__device__ __forceinline__ void add_products(v16f& acc, const float4& a, const float4& b, const v16f& zero) {
    v16f p = __builtin_amdgcn_mfma_f32_16x16x1f32(a.x, b.x, zero, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < N; ++e) {
        v16f q = p;
        if (e + 1 < N) q = __builtin_amdgcn_mfma_f32_16x16x1f32(f4(a, e + 1), f4(b, e + 1), zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = acc[r] + p[r];
        p = q;
    }
}
template <int N>
__device__ __forceinline__ void add_products(v4f& acc, const float4& a, const float4& b, const v4f& zero) {
    v4f p[N];
#pragma unroll
    for (int e = 0; e < N; ++e) p[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(f4(a, e), f4(b, e), zero, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < N; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = acc[r] + p[e][r];
}
template <class V>
__device__ __forceinline__ void add_rest(V& acc, const float4& a, const float4& b, const V& zero, uint32_t rest) {
    if (rest == 1) add_products<1>(acc, a, b, zero);
    if (rest == 2) add_products<2>(acc, a, b, zero);
    if (rest == 3) add_products<3>(acc, a, b, zero);
}

template <int ENG, int NW, bool RAW>
__device__ __forceinline__ void mlp_rows(uint32_t F, uint32_t H, uint32_t O, const float* __restrict__ wp,
                                         const RawWeights& raw, float* tile, const float* feat, uint32_t FS, float* hid,
                                         float* ul, uint32_t US) {
    static_assert(!RAW || ENG == 0, "raw weights are read by the ordered engine");
    constexpr uint32_t CH = NW * 64, HS = CH + 4;
    constexpr int NG = (kMlpOuts + 15) / 16;          // output groups of 16
    constexpr int GW = (NG + NW - 1) / NW;            // most groups a wave holds
    const MlpLayout l = mlp_layout(F, H, O);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t li = lane % 16, lk = lane / 16;
    const float4* w1 = reinterpret_cast<const float4*>(wp);
    const float4* w2 = reinterpret_cast<const float4*>(wp + l.w2);
    v4f acc2[GW];
    const uint32_t rg = (lane / 4) % 4, og = lane / 16, o4 = 4 * og + lane % 4;
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        const uint32_t first = 16 * (wave + g * NW);
        const uint32_t o = first + (ENG == 0 ? o4 : li);
        const float bias = first >= l.OC ? 0.0f : !RAW ? wp[l.b2 + o] : o < O ? raw.b2[o] : 0.0f;
        acc2[g] = v4f{bias, bias, bias, bias};
    }
    const v16f zero16 = {-0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f,
                         -0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f, -0.0f};
    const v4f zero4 = {-0.0f, -0.0f, -0.0f, -0.0f};
    for (uint32_t hb = 0; hb < H; hb += CH) {
        const uint32_t u0 = hb + 64 * wave;  // this wave's first hidden unit
        if (u0 < H) {
            if constexpr (ENG == 0) {
                v16f acc;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint32_t u = u0 + 16 * b + li;
                    const float bias = !RAW ? wp[l.b1 + u] : u < H ? raw.b1[u] : 0.0f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[4 * b + r] = bias;
                }
                const float4* a4 = reinterpret_cast<const float4*>(feat + li * FS);
                const uint32_t full = F / 4, rest = F % 4;
                if constexpr (RAW) {
                    float* wt = tile + wave * 64 * kTileS;
                    // load i: units 4 i + lane / 16, feature lane % 16 of the tile; units past H repeat the last
                    // one (their sums are never read), features past F the last feature (never added)
                    float next[16];
                    const float* src[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const uint32_t u = u0 + 4 * i + lk;
                        src[i] = raw.w1 + (uint64_t)(u < H ? u : H - 1) * F;
                    }
                    auto fetch = [&](uint32_t k0) {
                        const uint32_t k = k0 + li < F ? k0 + li : F - 1;
#pragma unroll
                        for (int i = 0; i < 16; ++i) next[i] = src[i][k];
                    };
                    fetch(0);
                    for (uint32_t k0 = 0; k0 < F; k0 += kTileK) {
                        mlp_wave_sync();  // the tile before it has been read
#pragma unroll
                        for (int i = 0; i < 16; ++i) wt[(4 * i + lk) * kTileS + li] = next[i];
                        mlp_wave_sync();
                        fetch(k0 + kTileK);
                        const float4* b4 = reinterpret_cast<const float4*>(wt + lane * kTileS);
                        const uint32_t left = full - k0 / 4;  // whole groups of four left
                        if (left >= kTileK / 4) {
#pragma unroll
                            for (uint32_t g = 0; g < kTileK / 4; ++g) add_products<4>(acc, a4[k0 / 4 + g], b4[g], zero16);
                        } else {
                            for (uint32_t g = 0; g < left; ++g) add_products<4>(acc, a4[k0 / 4 + g], b4[g], zero16);
                            add_rest(acc, a4[full], b4[left], zero16, rest);
                        }
                    }
                } else {
                    const float4* b4 = w1 + u0 + lane;
                    float4 next[4];  // the next sixteen features' weights, in flight while these are added
                    auto fetch = [&](uint32_t k) {
#pragma unroll
                        for (uint32_t g = 0; g < 4; ++g) next[g] = b4[(uint64_t)(k + g < l.K4 ? k + g : l.K4 - 1) * l.HC];
                    };
                    fetch(0);
                    float4 tail = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    for (uint32_t k0 = 0; k0 < l.K4; k0 += 4) {
                        float4 b[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) b[g] = next[g];
                        fetch(k0 + 4);
                        __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products
                        if (full - k0 >= 4) {
#pragma unroll
                            for (uint32_t g = 0; g < 4; ++g) add_products<4>(acc, a4[k0 + g], b[g], zero16);
                        } else {
#pragma unroll
                            for (uint32_t g = 0; g < 4; ++g) {
                                if (k0 + g < full) add_products<4>(acc, a4[k0 + g], b[g], zero16);
                                if (k0 + g == full) tail = b[g];
                            }
                        }
                    }
                    add_rest(acc, a4[full], tail, zero16, rest);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    hid[(4 * lk + r % 4) * HS + 64 * wave + 16 * (r / 4) + li] = fmaxf(acc[r], 0.0f);
            } else {
                v4f acc[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float bias = wp[l.b1 + u0 + 16 * t + li];
                    acc[t] = v4f{bias, bias, bias, bias};
                }
                for (uint32_t k = 0; k < l.K4; ++k) {
                    const float a = feat[li * FS + 4 * k + lk];  // zero past F
                    const float* wk = wp + ((uint64_t)k * l.HC + u0 + li) * 4 + lk;
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, wk[64 * t], acc[t], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) hid[(4 * lk + r) * HS + 64 * wave + 16 * t + li] = fmaxf(acc[t][r], 0.0f);
            }
        }
        __syncthreads();
        const uint32_t units = H - hb < CH ? H - hb : CH;
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            const uint32_t first = 16 * (wave + g * NW);
            if (first < l.OC) {  // wave-uniform
                if constexpr (ENG == 0) {
                    const float4* a4 = reinterpret_cast<const float4*>(hid + (4 * rg + lane % 4) * HS);
                    const float4* b4 = w2 + (uint64_t)(hb / 4) * l.OC + first + o4;
                    // raw: this lane's output row (the last one in place of a padded output), units past H clamped
                    const float* wr = raw.w2 + (uint64_t)(first + o4 < O ? first + o4 : O - 1) * H;
                    auto weights = [&](uint32_t k) {  // a whole group of four units
                        if constexpr (!RAW) return b4[(uint64_t)k * l.OC];
                        const float* w = wr + hb + 4 * k;
                        return make_float4(w[0], w[1], w[2], w[3]);
                    };
                    const uint32_t full = units / 4, rest = units % 4;
                    constexpr uint32_t W = 8;
                    if (full) {
                        float4 next[W];
                        auto fetch = [&](uint32_t k) {
#pragma unroll
                            for (uint32_t e = 0; e < W; ++e) next[e] = weights(k + e < full ? k + e : full - 1);
                        };
                        fetch(0);
                        for (uint32_t k0 = 0; k0 < full; k0 += W) {
                            float4 b[W];
#pragma unroll
                            for (uint32_t e = 0; e < W; ++e) b[e] = next[e];
                            fetch(k0 + W);
                            __builtin_amdgcn_sched_barrier(0);
                            if (full - k0 >= W) {
#pragma unroll
                                for (uint32_t e = 0; e < W; ++e) add_products<4>(acc2[g], a4[k0 + e], b[e], zero4);
                            } else {
#pragma unroll
                                for (uint32_t e = 0; e < W; ++e)
                                    if (k0 + e < full) add_products<4>(acc2[g], a4[k0 + e], b[e], zero4);
                            }
                        }
                    }
                    if (rest) {
                        float4 b;
                        if constexpr (RAW) {
                            const float* w = wr + hb + 4 * full;
                            b = make_float4(w[0], rest > 1 ? w[1] : 0.0f, rest > 2 ? w[2] : 0.0f, 0.0f);
                        } else {
                            b = b4[(uint64_t)full * l.OC];
                        }
                        add_rest(acc2[g], a4[full], b, zero4, rest);
                    }
                } else {
                    // a chunk's units past H hold relu(0) = 0 and meet zero weights
                    const float* wk = wp + l.w2 + ((uint64_t)(hb / 4) * l.OC + first + li) * 4 + lk;
                    for (uint32_t k = 0; k < (units + 3) / 4; ++k)
                        acc2[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(hid[li * HS + 4 * k + lk], wk[(uint64_t)k * l.OC * 4],
                                                                       acc2[g], 0, 0, 0);
                }
            }
        }
        if (hb + CH < H) __syncthreads();  // hid is read before the next chunk fills it
    }
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        const uint32_t first = 16 * (wave + g * NW);
        if (first < l.OC) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = ENG == 0 ? 4 * rg + r : 4 * lk + r;
                ul[row * US + first + (ENG == 0 ? o4 : li)] = acc2[g][r];
            }
        }
    }
    __syncthreads();
}

// Row stride in LDS of a block's features: a multiple of 4 (16-byte reads) that is 4 modulo 8, so that
// the 16 rows of a read fall on different banks.
__host__ __device__ inline uint32_t mlp_feature_stride(uint32_t F) { return ((F + 3) / 4 | 1u) * 4; }

// A wave takes every NW-th row; features past F and rows past the last are zeros.
template <int NW>
__device__ __forceinline__ void stage_rows(const float* __restrict__ src, uint32_t rows, uint32_t F, float* feat,
                                           uint32_t FS) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t k = lane; k < FS; k += 64) {
        float v[kMlpRows / NW];
#pragma unroll
        for (int i = 0; i < kMlpRows / NW; ++i) {
            const uint32_t r = wave + NW * i;
            v[i] = r < rows && k < F ? src[(uint64_t)r * F + k] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kMlpRows / NW; ++i) feat[(wave + NW * i) * FS + k] = v[i];
    }
    __syncthreads();
}

// Motion scaling of row r's outputs (model.rs:867-898).
template <int D>
__device__ __forceinline__ void motion(const StepParams& P, const float* u, float* dx) {
    float norm = 0.0f;
#pragma unroll
    for (int a = 0; a < D; ++a) norm += u[a] * u[a];
    norm = sqrtf(norm);
#pragma unroll
    for (int a = 0; a < D; ++a) dx[a] = P.alpha * u[a] * P.motion_eps / (1.0f + norm);
}

constexpr uint32_t kMlpUlStride = 49;  // outputs of a row in LDS (48 with the padding of a group)

// forward_from_features_with_eps (model.rs:867-940) for explicit feature rows [rows][F].
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, 2) void k_mlp_forward(StepParams P, const float* __restrict__ features, uint32_t rows,
                                                         RawWeights raw, float* __restrict__ dx,
                                                         float* __restrict__ ds) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t FS = mlp_feature_stride(P.F);
    float* feat = lds;
    float* hid = feat + kMlpRows * FS;
    float* ul = hid + kMlpRows * (NW * 64 + 4);
    const uint32_t row0 = blockIdx.x * kMlpRows;
    const uint32_t n = rows - row0 < (uint32_t)kMlpRows ? rows - row0 : (uint32_t)kMlpRows;
    stage_rows<NW>(features + (uint64_t)row0 * P.F, n, P.F, feat, FS);
    float* tile = ul + (kMlpRows * kMlpUlStride + 3) / 4 * 4;
    mlp_rows<0, NW, true>(P.F, P.H, D + P.S, nullptr, raw, tile, feat, FS, hid, ul, kMlpUlStride);
    if (threadIdx.x < n) {
        float v[D], px[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int a = 0; a < D; ++a) v[a] = ul[threadIdx.x * kMlpUlStride + a];
        motion<D>(P, v, px);
        float* o = dx + 4 * (uint64_t)(row0 + threadIdx.x);
#pragma unroll
        for (int a = 0; a < 4; ++a) o[a] = px[a];
    }
    for (uint32_t t = threadIdx.x; t < n * P.S; t += NW * 64) {
        const uint32_t r = t / P.S, c = t - r * P.S;
        ds[(uint64_t)row0 * P.S + t] = ul[r * kMlpUlStride + D + c];
    }
}

// The same for networks of a few dozen products a row, of whose hidden units a wave of the kernel above
// would use a few of its 64: a thread per row, 64 rows per block, their features staged in LDS (rows read
// from memory by thread touch a cache line each) and the hidden units held there. The weights are uniform loads.
template <int D>
__global__ __launch_bounds__(64) void k_mlp_forward_narrow(StepParams P, const float* __restrict__ features, uint32_t rows,
                                                           RawWeights raw, float* __restrict__ dx,
                                                           float* __restrict__ ds) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t F = P.F, H = P.H, S = P.S, FS = F | 1u, lane = threadIdx.x;
    const uint32_t row0 = blockIdx.x * 64, n = rows - row0 < 64 ? rows - row0 : 64;
    float* hid = lds + 64 * FS;  // [H][64]
    const float* src = features + (uint64_t)row0 * F;
    uint32_t r = lane / F, k = lane % F;
    for (uint32_t t = lane; t < n * F; t += 64) {
        lds[r * FS + k] = src[t];
        r += 64 / F;
        k += 64 % F;
        if (k >= F) {
            k -= F;
            ++r;
        }
    }
    __syncthreads();
    if (lane >= n) return;
    const float* f = lds + lane * FS;
    for (uint32_t h = 0; h < H; ++h) {
        float sum = raw.b1[h];
        for (uint32_t i = 0; i < F; ++i) sum += raw.w1[h * F + i] * f[i];
        hid[h * 64 + lane] = fmaxf(sum, 0.0f);
    }
    auto output = [&](uint32_t o) {
        float u = raw.b2[o];
        for (uint32_t h = 0; h < H; ++h) u += raw.w2[o * H + h] * hid[h * 64 + lane];
        return u;
    };
    float v[D], px[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int a = 0; a < D; ++a) v[a] = output(a);
    motion<D>(P, v, px);
    float* o = dx + 4 * (uint64_t)(row0 + lane);
#pragma unroll
    for (int a = 0; a < 4; ++a) o[a] = px[a];
    for (uint32_t c = 0; c < S; ++c) ds[(uint64_t)(row0 + lane) * S + c] = output(D + c);
}

// The update of the particles of 16 compact feature rows [rows][F]: MLP, motion scaling, 3D gates
// (model.rs:806-837) and the masked Euler step (step.rs:4-55). A row's first S features are its
// particle's state.
template <int D, int ENG, int NW>
__global__ __launch_bounds__(NW * 64, 2) void k_mlp_euler(StepParams P, const float* __restrict__ features,
                                                       const uint32_t* __restrict__ perm,
                                                       const uint32_t* __restrict__ act_rows,
                                                       const uint32_t* __restrict__ row_count,
                                                       const float* __restrict__ wp, StepIO io) {
    extern __shared__ __align__(16) float lds[];
    __shared__ uint32_t particle[kMlpRows];
    __shared__ float gate[kMlpRows], mask[kMlpRows];
    const uint32_t rows = *row_count;
    const uint32_t row0 = blockIdx.x * kMlpRows;
    if (row0 >= rows) return;  // whole block
    const uint32_t n = rows - row0 < (uint32_t)kMlpRows ? rows - row0 : (uint32_t)kMlpRows;
    const uint32_t FS = mlp_feature_stride(P.F), S = P.S;
    float* feat = lds;
    float* hid = feat + kMlpRows * FS;
    float* ul = hid + kMlpRows * (NW * 64 + 4);
    float4 pos = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t i = 0;
    const bool lead = threadIdx.x < n;  // the row's position, gates and mask
    if (lead) {
        const uint32_t s = act_rows[row0 + threadIdx.x];
        const uint32_t b = s / P.N, local = perm[s];
        i = b * P.N + local;
        pos = io.pos[i];
        particle[threadIdx.x] = i;
        mask[threadIdx.x] = io.mask ? io.mask[i] : hash_mask(local, b, P.N, P.update_prob, P.step_index, P.base_seed);
    }
    stage_rows<NW>(features + (uint64_t)row0 * P.F, n, P.F, feat, FS);
    mlp_rows<ENG, NW, false>(P.F, P.H, D + S, wp, RawWeights{}, nullptr, feat, FS, hid, ul, kMlpUlStride);
    if (lead) {
        const float* st = feat + threadIdx.x * FS;
        float v[D], dx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int a = 0; a < D; ++a) v[a] = ul[threadIdx.x * kMlpUlStride + a];
        motion<D>(P, v, dx);
        float sg = 1.0f;
        if (P.gates3d) {
            const float liveness = st[3], sd = S > 7 ? st[7] : st[0];
            sg = clampf_((4.0f - liveness) * 2.0f, 0.0f, 1.0f);
            float mg = 0.0f;
            if (!(pos.w >= 0.5f)) mg = sg * clampf_((fabsf(sd) - 0.01f) / 0.02f, 0.0f, 1.0f);
#pragma unroll
            for (int a = 0; a < D; ++a) dx[a] *= mg;
        }
        gate[threadIdx.x] = sg;
        const float m = mask[threadIdx.x];
        float pn[4] = {pos.x, pos.y, pos.z, pos.w};
        constexpr int MEM = D == 3 ? 4 : 2;
#pragma unroll
        for (int a = 0; a < MEM; ++a) pn[a] += P.dt * dx[a] * m;
        if (P.g.boundary == 0) {
#pragma unroll
            for (int a = 0; a < D; ++a) pn[a] = wrap_axis(pn[a], a, P.g);
        }
        io.out_pos[i] = make_float4(pn[0], pn[1], pn[2], pn[3]);
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < n * S; t += NW * 64) {
        const uint32_t r = t / S, c = t - r * S;
        float dsc = ul[r * kMlpUlStride + D + c];
        if (P.gates3d) dsc *= gate[r];
        float next = feat[r * FS + c] + P.dt * dsc * mask[r];
        if (clamped_channel(D, S, c)) next = clampf_(next, -8.0f, 24.0f);
        io.out_states[(uint64_t)particle[r] * S + c] = next;
    }
}

size_t mlp_weight_floats(const StepParams& p) { return (size_t)mlp_layout(p.F, p.H, (uint32_t)p.g.dim + p.S).total; }

hipError_t launch_mlp_weights(const StepParams& p, const float* w1, const float* b1, const float* w2, const float* b2,
                              float* wp, hipStream_t stream) {
    const size_t n = mlp_weight_floats(p);
    const uint32_t blocks = (uint32_t)std::min<size_t>((n + 255) / 256, 1024);
    hipLaunchKernelGGL(k_mlp_weights, dim3(blocks), dim3(256), 0, stream, p.F, p.H, (uint32_t)p.g.dim + p.S, w1, b1, w2,
                       b2, wp);
    return hipGetLastError();
}

// Two waves serve up to 128 hidden units in one chunk, four more of them.
static int mlp_waves(const StepParams& p) { return p.H <= 128 ? 2 : 4; }
static uint32_t mlp_lds_bytes(const StepParams& p, int waves, bool raw) {
    const uint32_t rows = (uint32_t)kMlpRows * (mlp_feature_stride(p.F) + (uint32_t)waves * 64 + 4 + kMlpUlStride);
    return ((rows + 3) / 4 * 4 + (raw ? (uint32_t)waves * 64 * kTileS : 0u)) * 4;
}

// Networks of at most 400 products a row on rows that fill the chip: 600,000 rows of F = 6, H = 8 take 20 us with a
// thread per row and 135 us with sixteen rows per block, of F = 66, H = 4 174 and 315 us. Above, or with few rows,
// the rows' own chain sets the time (4,000 rows of F = 66, H = 4: 21 and 14 us; 60,000 of F = 18, H = 32: 29 and 24 us),
// and wide rows leave too few waves (600,000 of F = 123, H = 2: 502 and 455 us).
static bool mlp_narrow(const StepParams& p, uint32_t rows) {
    return rows > 16384 && p.F <= 72 && (uint64_t)(p.F + p.g.dim + p.S) * p.H <= 400;
}

hipError_t launch_mlp_forward(const StepParams& p, const float* features, uint32_t rows, const StepIO& io,
                              float* dx, float* ds, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const int nw = mlp_waves(p);
    const bool narrow = mlp_narrow(p, rows);
    auto k = narrow ? (p.g.dim == 2 ? k_mlp_forward_narrow<2> : k_mlp_forward_narrow<3>)
             : p.g.dim == 2 ? (nw == 2 ? k_mlp_forward<2, 2> : k_mlp_forward<2, 4>)
                            : (nw == 2 ? k_mlp_forward<3, 2> : k_mlp_forward<3, 4>);
    const uint32_t per = narrow ? 64u : (uint32_t)kMlpRows, threads = narrow ? 64u : (uint32_t)nw * 64;
    const uint32_t lds = narrow ? 64 * ((p.F | 1u) + p.H) * 4 : mlp_lds_bytes(p, nw, true);
    // a launch holds fewer than 2^32 threads
    constexpr uint32_t kMost = 1u << 26;
    for (uint32_t first = 0; first < rows; first += std::min(rows - first, kMost)) {
        const uint32_t n = std::min(rows - first, kMost);
        hipLaunchKernelGGL(k, dim3((n - 1) / per + 1), dim3(threads), lds, stream, p,
                           features + (uint64_t)first * p.F, n, RawWeights{io.w1, io.b1, io.w2, io.b2},
                           dx + 4 * (uint64_t)first, ds + (uint64_t)first * p.S);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int D, int ENG>
static hipError_t launch_mlp_euler_e(const StepParams& p, Workspace& ws, const StepIO& io, hipStream_t stream,
                                     Profiler* prof) {
    const int nw = mlp_waves(p);
    return launch_timed(prof, NPA_KERNEL_MLP, nw == 2 ? k_mlp_euler<D, ENG, 2> : k_mlp_euler<D, ENG, 4>,
                        dim3((p.T + kMlpRows - 1) / kMlpRows), dim3(nw * 64), mlp_lds_bytes(p, nw, false), stream, p,
                        ws.features.as<float>(), ws.perm.as<uint32_t>(), ws.act_rows.as<uint32_t>(),
                        ws.wl_count.as<uint32_t>() + 1, ws.wpad.as<float>(), io);
}

hipError_t launch_mlp_euler(const StepParams& p, Workspace& ws, const StepIO& io, hipStream_t stream, Profiler* prof) {
    if (p.g.dim == 2)
        return p.mlp_engine == NPA_MLP_VALU ? launch_mlp_euler_e<2, 0>(p, ws, io, stream, prof)
                                            : launch_mlp_euler_e<2, 1>(p, ws, io, stream, prof);
    return p.mlp_engine == NPA_MLP_VALU ? launch_mlp_euler_e<3, 0>(p, ws, io, stream, prof)
                                        : launch_mlp_euler_e<3, 1>(p, ws, io, stream, prof);
}

}  // namespace npa
