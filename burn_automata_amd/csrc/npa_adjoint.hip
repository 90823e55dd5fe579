// npa_adjoint.hip - the perception adjoint (reverse mode of perceive_with_options) on gfx950.
//
// Reference: perceive_adjoint_with_options, crates/burn_automata_kernels/src/reference/adjoint.rs.
// The reference walks every particle idx once and scatters into the adjoint arrays of idx and of
// its neighbours j. Here every particle gathers instead: the neighbour relation is symmetric
// with equal multiplicity (for_each_neighbor accepts j for idx exactly when it accepts idx for j:
// the same cell offsets negated, the same r^2 < eps^2 test on the negated delta), so a particle
// k receives, over its own neighbour list, every term the reference adds into k - both the
// terms of the pairs where k is the neighbour j of idx = that neighbour, and the terms where k
// is idx. No atomics; the result is deterministic and equals the reference's up to rounding.
//
//   the forward density pass   rho, volumes and each particle's accepted neighbours    forward.rs:145-160
//   k_adj_prep     per particle: the forward state-gradient sums and moment matrix, then the
//                  adjoint of moment correction / scaling / log-norm (raw-gradient adjoint,
//                  moment adjoint) and of the density gradient                adjoint.rs:168-397
//   k_adj_gather   per particle: blurred-state, state-gradient, hybrid-moment and
//                  density-gradient pair terms in both roles; identity and position rows;
//                  the particle's density adjoint                             adjoint.rs:27-348
//   k_adj_density_kernel  the density kernel's position terms                 adjoint.rs:399-418
//
// Notation for the pair of the receiving particle k and its neighbour j: d = p_j - p_k, r = |d|,
// n = d / r, x = eps^2 - r^2, f = 3 K5 (eps - r)^2, h = -3 K5 x, v = 1 / rho; rg the raw-gradient
// adjoint, fb the blurred-feature adjoint, M the moment adjoint plus its transpose, rda the raw
// density-gradient adjoint. The spiky gradient is f n and its delta adjoint, which is linear and
// even in the pair's direction, takes q to (f q + h (q.n) n) / r. Both roles of a pair then sum to
//   state_k  += fb_k-terms:  v_k W fb_j  -  v_k f (rg_j.n)            (k as the neighbour of j)
//             -              rg_k . (v_j f n)                          (k as idx)
//   pos_k    += (f q + h (q.n) n) / r  -  f X n - h (n.X n) n / 2  +  6 K6 x^2 A d
//       q = sum_c (s_k - s_j)_c (v_k rg_j + v_j rg_k)_c + rda_j - rda_k,   X = v_k M_j + v_j M_k,
//       A = v_k fb_j.s_k + v_j fb_k.s_j + dens_k + dens_j     (the dens terms in the last pass)
//   dens_k   -= v_k^2 (W fb_j.s_k - f (rg_j.n).(s_k - s_j) + f r (n.M_j n) / 2)
// so that the sums over channels are taken once per pair, and whatever is constant over k's
// neighbours is applied once per particle.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "npa_internal.hpp"
#include "npa_neighbors.hpp"

namespace npa {

// log_normalize_adjoint  normalize.rs:71-91 (adds into in_adj)
template <int D>
__device__ __forceinline__ void log_normalize_adjoint(const float* in, const float* out_adj, float* in_adj) {
    const float E = 1.0e-6f;
    float s = in[0] * in[0];
#pragma unroll
    for (int k = 1; k < D; ++k) s += in[k] * in[k];
    const float norm = fmaxf(sqrtf(s + E * E), E);
    const float lp = npa_log1pf(norm);
    const float scale = lp / norm;
    const float dscale = (norm / (1.0f + norm) - lp) / (norm * norm);
    float dot = in[0] * out_adj[0];
#pragma unroll
    for (int k = 1; k < D; ++k) dot += in[k] * out_adj[k];
    const float radial = dscale * dot / norm;
#pragma unroll
    for (int k = 0; k < D; ++k) in_adj[k] += scale * out_adj[k] + radial * in[k];
}

struct AdjointArgs {
    const float4* srec;
    const int4* scoord;
    const uint32_t* bo;
    const uint32_t* perm;
    const uint32_t* act_rows;   // compact row -> slot (every particle has a row)
    const uint32_t* row_count;
    const uint32_t* nb_base;    // accepted neighbours by compact row (the density pass)
    const uint64_t* nb_mask;
    const uint32_t* nb_count;
    const float4* svol;   // slot order: position, 1 / rho
    const float* sstate;  // [T][SS] sorted, padded
    const float* fadj;    // [T][F] particle order
    float* rows;          // [T][4 * slice]: what a neighbour gathers of a particle, see AdjRow
    float* side;          // [T][kSide<D>]: M (upper triangle), then rda
    float4* dpos;         // slot order: position, density adjoint
    float4* ppos;         // slot order: position adjoint before the density-kernel terms
    float* state_adj;     // [T][S] particle order (output)
    float4* pos_adj;      // [T] particle order (output)
};

// Four lanes serve a particle, lane q owning its channels q * CPL .. + CPL - 1. Its gathered row holds
// for each lane the slice [s CPL][fb CPL][rg CPL * D] padded to whole float4s, with float4 v of lane
// q at v * 4 + q, so that the four lanes of a load read 64 consecutive bytes.
template <int D, int SM>
struct AdjRow {
    static constexpr int L = 4, CPL = SM / L;
    static constexpr int USED = CPL * (2 + D), NV = (USED + 3) / 4;
    static constexpr int FLOATS = NV * 16;
    float v[NV * 4];
    __device__ __forceinline__ void load(const float* __restrict__ rows, uint32_t slot, uint32_t q) {
        const float4* p = reinterpret_cast<const float4*>(rows + (uint64_t)slot * FLOATS) + q;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const float4 x = p[4 * k];
            v[4 * k] = x.x;
            v[4 * k + 1] = x.y;
            v[4 * k + 2] = x.z;
            v[4 * k + 3] = x.w;
        }
    }
    __device__ __forceinline__ void store(float* __restrict__ rows, uint32_t slot, uint32_t q) const {
        float4* p = reinterpret_cast<float4*>(rows + (uint64_t)slot * FLOATS) + q;
#pragma unroll
        for (int k = 0; k < NV; ++k) p[4 * k] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    }
    __device__ __forceinline__ float s(int u) const { return v[u]; }
    __device__ __forceinline__ float fb(int u) const { return v[CPL + u]; }
    __device__ __forceinline__ float rg(int u, int a) const { return v[2 * CPL + u * D + a]; }
};
template <int D>
constexpr int kSide = D == 3 ? 12 : 8;

// Sum over a quad, the same pairing in every lane (lane ^ 2, then lane ^ 1).
__device__ __forceinline__ float quad_swap2(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_swap1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_sum(float v) {
    v += quad_swap2(v);
    v += quad_swap1(v);
    return v;
}
// Lane q of a quad gets the quad's sum of v[q].
__device__ __forceinline__ float quad_scatter(const float (&v)[4], uint32_t q) {
    const bool hi = (q & 2u) != 0, odd = (q & 1u) != 0;
    const float y0 = (hi ? v[2] : v[0]) + quad_swap2(hi ? v[0] : v[2]);
    const float y1 = (hi ? v[3] : v[1]) + quad_swap2(hi ? v[1] : v[3]);
    return (odd ? y1 : y0) + quad_swap1(odd ? y0 : y1);
}
template <int J>
__device__ __forceinline__ uint32_t quad_slot(uint32_t slot) {
    return (uint32_t)__float_as_int(group_bcast<4, J>(__int_as_float((int)slot)));
}

// The pair quantities of the notation above; f, h and n are zero for the self pair and for coincident
// particles (spiky_gradient_kernel and its adjoint, kernels.rs:81-126) and for a lane without an entry.
template <int D>
struct AdjPair {
    float d[3], n[D];
    float x, r, ir, f, h;
    __device__ __forceinline__ void set(const GridParams& g, const float* pk, const float4& rec, bool other) {
        d[0] = delta_axis(pk[0], rec.x, 0, g);
        d[1] = delta_axis(pk[1], rec.y, 1, g);
        d[2] = 0.0f;
        float r2 = d[0] * d[0];
        r2 += d[1] * d[1];
        if constexpr (D == 3) {
            d[2] = delta_axis(pk[2], rec.z, 2, g);
            r2 += d[2] * d[2];
        }
        x = g.eps2 - r2;
        const bool ok = other && r2 > 0.0f;
        // r and 1 / r from the hardware's reciprocal square root, each refined once. It takes a subnormal
        // for zero, so the squares of distances below 2^-50 are scaled by 2^64, exactly, around it.
        const bool tiny = r2 < 0x1p-100f;
        const float z = ok ? (tiny ? r2 * 0x1p64f : r2) : 1.0f;
        float y = __builtin_amdgcn_rsqf(z);
        y = fmaf(0.5f * y, fmaf(-z * y, y, 1.0f), y);
        const float w = z * y;
        r = fmaf(fmaf(-w, w, z), 0.5f * y, w);
        r = tiny ? r * 0x1p-32f : r;
        y = tiny ? y * 0x1p32f : y;
        ir = y;
        const float t = g.eps - r, k = ok ? 3.0f * g.k5 : 0.0f;
        f = k * (t * t);
        h = -(k * x);
#pragma unroll
        for (int a = 0; a < D; ++a) n[a] = ok ? d[a] * y : 0.0f;
    }
};

// Walks the accepted neighbours of 16 particles per wave in rounds of four list entries per particle:
// lane q holds entry 4 r + q of its particle's list. `rounds(n)` takes the lists' first n rounds.
template <int D, class Rounds>
__device__ __forceinline__ void adj_walk(const StepParams& P, const AdjointArgs& A, PerceiveLists<16>& lists, uint32_t row,
                                         bool active, uint32_t b, const float* pi, const int* ci, uint32_t& cnt,
                                         Rounds&& rounds) {
    const uint32_t lane = threadIdx.x, t = lane / 4, q = lane % 4;
    // Entry e of a particle's whole list falls to lane e % 4 wherever the lists have to be emptied in
    // between (which depends on the wave's other particles): a flush before the end takes whole rounds
    // and keeps up to three entries, so the sums' order, and with it the result, is always the same.
    auto flush = [&](bool last) {
        __syncthreads();  // list writes of every lane are visible
        const uint32_t keep = last ? 0u : cnt % 4;
        cnt -= keep;
        const uint32_t kept = q < keep ? lists.slot[cnt + q][t] : 0u;
        const uint32_t n = wave_max_u32(active ? (cnt + 3) / 4 : 0u);
        if (n) rounds(n);
        __syncthreads();  // every lane has read the lists before they are refilled
        if (q < keep) lists.slot[q][t] = kept;
        cnt = keep;
    };
    append_accepted<D, 4>(P, A.srec, A.scoord, A.bo, A.nb_base, A.nb_mask, A.nb_count, row, active, b, pi, ci, lane, t, q,
                          lists, cnt, [&]() { flush(false); });
    flush(true);
}

// One wave per 16 particles over their lists of accepted neighbours: a walk over the 3^D cells'
// candidates runs its body for all 16 particles whenever one of them accepts, about three times as
// often. Lane q takes the pair quantities of every fourth entry, and all four lanes that entry's sums for
// their channels. Bound: VALU issue and the rows' gathers, at two waves per SIMD (the 2D system below)
// or one (the 3D system). Measured on 8 x 4,096 2D particles, 41 neighbours each, S = 16: 176 -> 27 us;
// 2 x 8,192 3D particles, 65 neighbours, S = 24: 438 -> 39 us.
template <int D, int SM>
__global__ __launch_bounds__(64) void k_adj_prep(StepParams P, AdjointArgs A) {
    using Row = AdjRow<D, SM>;
    constexpr int CPL = Row::CPL, NM = D * (D + 1) / 2;
    __shared__ PerceiveLists<16> lists;
    constexpr uint32_t CAP = PerceiveLists<16>::CAP;
    const uint32_t lane = threadIdx.x, t = lane / 4, q = lane % 4, c0 = q * CPL;
    const uint32_t nrows = *A.row_count, S = P.S;
    for (uint32_t it = blockIdx.x; it * 16 < nrows; it += gridDim.x) {
        const uint32_t row = it * 16 + t;
        const bool active = row < nrows;
        const uint32_t s = A.act_rows[active ? row : it * 16];
        const uint32_t b = s / P.N;
        const uint64_t pk = (uint64_t)b * P.N + A.perm[s];
        const float* fa = A.fadj + pk * P.F;
        float pi[3];
        int ci[3];
        load_rec<D>(A.srec, A.scoord, s, pi, ci);
        Row out;
#pragma unroll
        for (int k = 0; k < Row::NV * 4; ++k) out.v[k] = 0.0f;
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            out.v[u] = A.sstate[(uint64_t)s * SM + c0 + u];
            out.v[CPL + u] = c0 + u < S ? fa[S + c0 + u] : 0.0f;
        }
        float raw[CPL * D], mom[NM], rawd[D];
#pragma unroll
        for (int k = 0; k < CPL * D; ++k) raw[k] = 0.0f;
#pragma unroll
        for (int k = 0; k < NM; ++k) mom[k] = 0.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) rawd[a] = 0.0f;
        if (P.state_grad || P.density_grad) {
            uint32_t cnt = 0;
            adj_walk<D>(P, A, lists, row, active, b, pi, ci, cnt, [&](uint32_t rounds) {
                struct Fetch {
                    uint32_t slot;
                    bool has;
                    float4 rec;
                    float sv[4][CPL];
                };
                auto fetch = [&](uint32_t r, Fetch& F) {
                    const uint32_t e = 4 * r + q;
                    F.has = active && e < cnt;
                    F.slot = F.has ? lists.slot[e < CAP ? e : CAP - 1][t] : s;
                    F.rec = A.svol[F.slot];
                    const uint32_t js[4] = {quad_slot<0>(F.slot), quad_slot<1>(F.slot), quad_slot<2>(F.slot),
                                            quad_slot<3>(F.slot)};
                    if (P.state_grad) {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int u = 0; u < CPL; ++u) F.sv[j][u] = A.sstate[(uint64_t)js[j] * SM + c0 + u];
                    }
                };
                auto compute = [&](const Fetch& F) {
                    AdjPair<D> p;
                    p.set(P.g, pi, F.rec, F.has && F.slot != s);
                    float g[D];
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        rawd[a] = fmaf(p.f, p.n[a], rawd[a]);
                        g[a] = F.rec.w * p.f * p.n[a];
                    }
                    if (!P.state_grad) return;
                    int m = 0;
#pragma unroll
                    for (int a = 0; a < D; ++a)
#pragma unroll
                        for (int c = a; c < D; ++c, ++m) mom[m] = fmaf(p.d[a], g[c], mom[m]);
                    auto entry = [&](auto J) {
                        constexpr int j = decltype(J)::value;
                        float cg[D];
#pragma unroll
                        for (int a = 0; a < D; ++a) cg[a] = group_bcast<4, j>(g[a]);
#pragma unroll
                        for (int u = 0; u < CPL; ++u) {
                            const float diff = F.sv[j][u] - out.v[u];
#pragma unroll
                            for (int a = 0; a < D; ++a) raw[u * D + a] = fmaf(diff, cg[a], raw[u * D + a]);
                        }
                    };
                    entry(std::integral_constant<int, 0>{});
                    entry(std::integral_constant<int, 1>{});
                    entry(std::integral_constant<int, 2>{});
                    entry(std::integral_constant<int, 3>{});
                };
                Fetch X, Y;  // the next round's loads are out while a round is summed
                fetch(0, X);
                for (uint32_t r = 0; r < rounds; r += 2) {
                    fetch(r + 1, Y);
                    compute(X);
                    if (r + 1 >= rounds) break;
                    fetch(r + 2, X);
                    compute(Y);
                }
            });
        }
        if (!active) continue;
        float* side = A.side + (uint64_t)s * kSide<D>;
        uint32_t cur = 2 * S;
        if (P.state_grad) {
            float moment[D * D], inv[D * D];
            int m = 0;
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int c = a; c < D; ++c, ++m) {
                    moment[a * D + c] = quad_sum(mom[m]);
                    moment[c * D + a] = moment[a * D + c];
                }
            if (P.hybrid) safe_inverse<D>(moment, inv);
            const float scale = P.state_scale;
            float inv_adj[D * D];
#pragma unroll
            for (int k = 0; k < D * D; ++k) inv_adj[k] = 0.0f;
#pragma unroll
            for (int u = 0; u < CPL; ++u) {
                const uint32_t c = c0 + u;
                if (c >= S) continue;
                float corr[D];
#pragma unroll
                for (int a = 0; a < D; ++a) corr[a] = raw[u * D + a];
                if (P.hybrid) {
                    float mc[D];
#pragma unroll
                    for (int o = 0; o < D; ++o) {
                        mc[o] = 0.0f;
#pragma unroll
                        for (int ia = 0; ia < D; ++ia) mc[o] += corr[ia] * inv[ia * D + o];
                    }
#pragma unroll
                    for (int a = 0; a < D; ++a) corr[a] = mc[a];
                }
                float nin[D], cadj[D], ga[D];
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    nin[a] = corr[a] * scale;
                    ga[a] = fa[cur + c * D + a];
                    cadj[a] = 0.0f;
                }
                if (P.log_norm_grad) log_normalize_adjoint<D>(nin, ga, cadj);
                else
#pragma unroll
                    for (int a = 0; a < D; ++a) cadj[a] = ga[a];
#pragma unroll
                for (int a = 0; a < D; ++a) cadj[a] *= scale;
                if (P.hybrid) {
#pragma unroll
                    for (int ia = 0; ia < D; ++ia) {
                        float radj = 0.0f;
#pragma unroll
                        for (int o = 0; o < D; ++o) {
                            radj += cadj[o] * inv[ia * D + o];
                            inv_adj[ia * D + o] += raw[u * D + ia] * cadj[o];
                        }
                        out.v[2 * CPL + u * D + ia] = radj;
                    }
                } else {
#pragma unroll
                    for (int a = 0; a < D; ++a) out.v[2 * CPL + u * D + a] = cadj[a];
                }
            }
            if (P.hybrid) {  // inverse_matrix_adjoint  adjoint.rs:447-468, inv_adj summed over the quad
                float madj[D * D];
#pragma unroll
                for (int k = 0; k < D * D; ++k) inv_adj[k] = quad_sum(inv_adj[k]);
#pragma unroll
                for (int rr = 0; rr < D; ++rr)
#pragma unroll
                    for (int cc = 0; cc < D; ++cc) {
                        float v = 0.0f;
#pragma unroll
                        for (int ir = 0; ir < D; ++ir)
#pragma unroll
                            for (int ic = 0; ic < D; ++ic) v += inv[ir * D + rr] * inv_adj[ir * D + ic] * inv[cc * D + ic];
                        madj[rr * D + cc] = 0.0f - v;
                    }
                if (q == 0) {
                    m = 0;
#pragma unroll
                    for (int a = 0; a < D; ++a)
#pragma unroll
                        for (int c = a; c < D; ++c, ++m) side[m] = madj[a * D + c] + madj[c * D + a];
                }
            }
            cur += S * D;
        }
        if (P.density_grad) {  // adjoint.rs:350-397
            const float scale = P.dgrad_scale;
            float nin[D], radj[D], da[D];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                nin[a] = quad_sum(rawd[a]) * scale;
                radj[a] = 0.0f;
                da[a] = fa[cur + a];
            }
            if (P.log_norm_dgrad) {
                log_normalize_adjoint<D>(nin, da, radj);
#pragma unroll
                for (int a = 0; a < D; ++a) radj[a] *= scale;
            } else {
#pragma unroll
                for (int a = 0; a < D; ++a) radj[a] = da[a] * scale;
            }
            if (q == 0) {
#pragma unroll
                for (int a = 0; a < D; ++a) side[NM + a] = radj[a];
            }
        }
        out.store(A.rows, s, q);
    }
}

// Every pair term of both roles but the density kernel's, by the receiving particle. The channels'
// sums of a pair are added across the quad once per value (quad_scatter: the sums of four entries
// arrive in the lanes that own them), and the position terms are evaluated once per pair rather than in
// every lane. Measured as k_adj_prep: 461 -> 38 us (2D), 976 -> 62 us (3D).
template <int D, int SM>
__global__ __launch_bounds__(64) void k_adj_gather(StepParams P, AdjointArgs A) {
    using Row = AdjRow<D, SM>;
    constexpr int CPL = Row::CPL, NM = D * (D + 1) / 2, NS = kSide<D> / 4;
    __shared__ PerceiveLists<16> lists;
    constexpr uint32_t CAP = PerceiveLists<16>::CAP;
    const uint32_t lane = threadIdx.x, t = lane / 4, q = lane % 4, c0 = q * CPL;
    const uint32_t nrows = *A.row_count, S = P.S;
    const bool sg = P.state_grad != 0, hybrid = sg && P.hybrid, dg = P.density_grad != 0;
    for (uint32_t it = blockIdx.x; it * 16 < nrows; it += gridDim.x) {
        const uint32_t row = it * 16 + t;
        const bool active = row < nrows;
        const uint32_t s = A.act_rows[active ? row : it * 16];
        const uint32_t b = s / P.N;
        float pi[3];
        int ci[3];
        load_rec<D>(A.srec, A.scoord, s, pi, ci);
        Row own;
        own.load(A.rows, s, q);
        const float vk = A.svol[s].w;
        float sv[CPL], B[CPL], T[CPL];
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            sv[u] = vk * own.s(u);
            B[u] = 0.0f;
            T[u] = 0.0f;
        }
        float mk[NM], rk[D], pa[D], G[D];
#pragma unroll
        for (int m = 0; m < NM; ++m) mk[m] = hybrid ? A.side[(uint64_t)s * kSide<D> + m] : 0.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            rk[a] = dg ? A.side[(uint64_t)s * kSide<D> + NM + a] : 0.0f;
            pa[a] = 0.0f;
            G[a] = 0.0f;
        }
        float dsum = 0.0f, msum = 0.0f;  // sum f (rg_j.n).(s_k - s_j) over this lane's channels; f r n.M_j n
        uint32_t cnt = 0;
        adj_walk<D>(P, A, lists, row, active, b, pi, ci, cnt, [&](uint32_t rounds) {
            auto slot_of = [&](uint32_t r, bool& has) {
                const uint32_t e = 4 * r + q;
                has = active && e < cnt;
                return has ? lists.slot[e < CAP ? e : CAP - 1][t] : s;
            };
            bool has;
            uint32_t slot = slot_of(0, has);
            float4 rec = A.svol[slot], sd[NS];
#pragma unroll
            for (int k = 0; k < NS; ++k) sd[k] = reinterpret_cast<const float4*>(A.side)[(uint64_t)slot * NS + k];
            Row R0, R1;
            R0.load(A.rows, quad_slot<0>(slot), q);
            for (uint32_t r = 0; r < rounds; ++r) {
                bool has_n;
                const uint32_t slot_n = slot_of(r + 1, has_n);
                const float4 rec_n = A.svol[slot_n];
                float4 sd_n[NS];
#pragma unroll
                for (int k = 0; k < NS; ++k) sd_n[k] = reinterpret_cast<const float4*>(A.side)[(uint64_t)slot_n * NS + k];
                AdjPair<D> p;
                p.set(P.g, pi, rec, has && slot != s);
                const float x2 = has ? P.g.k6 * (p.x * p.x) : 0.0f, W = x2 * p.x, vj = rec.w;
                float sn[D];
#pragma unroll
                for (int a = 0; a < D; ++a) sn[a] = p.f * p.n[a];
                float tot[1 + D][4];
                auto entry = [&](auto J, const Row& R) {
                    constexpr int j = decltype(J)::value;
                    const float Wj = group_bcast<4, j>(W), vjj = group_bcast<4, j>(vj);
                    float cn[D], gj[D], hk[D], wad = 0.0f, wk = 0.0f;
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        cn[a] = group_bcast<4, j>(sn[a]);
                        gj[a] = 0.0f;
                        hk[a] = 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < CPL; ++u) {
                        wad = fmaf(R.fb(u), sv[u], wad);
                        wk = fmaf(own.fb(u), R.s(u), wk);
                        B[u] = fmaf(Wj, R.fb(u), B[u]);
                        if (sg) {
                            const float diff = own.s(u) - R.s(u), dv = vk * diff;
                            float tc = R.rg(u, 0) * cn[0];
#pragma unroll
                            for (int a = 1; a < D; ++a) tc = fmaf(R.rg(u, a), cn[a], tc);
                            T[u] += tc;
                            dsum = fmaf(tc, diff, dsum);
#pragma unroll
                            for (int a = 0; a < D; ++a) {
                                gj[a] = fmaf(R.rg(u, a), dv, gj[a]);
                                hk[a] = fmaf(own.rg(u, a), diff, hk[a]);
                            }
                        }
                    }
                    tot[0][j] = fmaf(vjj, wk, wad);
#pragma unroll
                    for (int a = 0; a < D; ++a) tot[1 + a][j] = fmaf(vjj, hk[a], gj[a]);
                };
                // the next entry's row is loaded while one is summed
                R1.load(A.rows, quad_slot<1>(slot), q);
                entry(std::integral_constant<int, 0>{}, R0);
                R0.load(A.rows, quad_slot<2>(slot), q);
                entry(std::integral_constant<int, 1>{}, R1);
                R1.load(A.rows, quad_slot<3>(slot), q);
                entry(std::integral_constant<int, 2>{}, R0);
                R0.load(A.rows, quad_slot<0>(slot_n), q);
                entry(std::integral_constant<int, 3>{}, R1);
                // this lane's entry: the channel sums of its pair
                const float al = 6.0f * x2 * quad_scatter(tot[0], q);
                float qv[D], qn = 0.0f;
                const float* sj = reinterpret_cast<const float*>(sd);
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    qv[a] = sg ? quad_scatter(tot[1 + a], q) : 0.0f;
                    if (dg) qv[a] += sj[NM + a] - rk[a];
                    qn = fmaf(qv[a], p.n[a], qn);
                    G[a] = fmaf(vj, sn[a], G[a]);
                }
                const float fi = p.f * p.ir, hi = p.h * p.ir * qn;
#pragma unroll
                for (int a = 0; a < D; ++a) pa[a] += fmaf(fi, qv[a], fmaf(hi, p.n[a], al * p.d[a]));
                if (hybrid) {
                    float Xn[D], Mn[D], nXn = 0.0f, nMn = 0.0f;
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        Xn[a] = 0.0f;
                        Mn[a] = 0.0f;
#pragma unroll
                        for (int c = 0; c < D; ++c) {
                            const int lo = a < c ? a : c, hi2 = a < c ? c : a;
                            const int m = D == 2 ? lo + hi2 : (lo == 0 ? hi2 : lo + hi2 + 1);
                            Mn[a] = fmaf(sj[m], p.n[c], Mn[a]);
                            Xn[a] = fmaf(fmaf(vk, sj[m], vj * mk[m]), p.n[c], Xn[a]);
                        }
                        nXn = fmaf(Xn[a], p.n[a], nXn);
                        nMn = fmaf(Mn[a], p.n[a], nMn);
                    }
                    const float hx = 0.5f * p.h * nXn;
#pragma unroll
                    for (int a = 0; a < D; ++a) pa[a] -= fmaf(p.f, Xn[a], hx * p.n[a]);
                    msum = fmaf(p.f * p.r, nMn, msum);
                }
                slot = slot_n;
                has = has_n;
                rec = rec_n;
#pragma unroll
                for (int k = 0; k < NS; ++k) sd[k] = sd_n[k];
            }
        });
        if (!active) continue;
        const uint64_t pk = (uint64_t)b * P.N + A.perm[s];
        const float* fa = A.fadj + pk * P.F;
        float bs = 0.0f;  // sum W fb_j.s_k over this lane's channels
#pragma unroll
        for (int u = 0; u < CPL; ++u) bs = fmaf(own.s(u), B[u], bs);
        const float dens = quad_sum(dsum - bs - 0.5f * msum) * (vk * vk);
#pragma unroll
        for (int a = 0; a < D; ++a) {
            pa[a] = quad_sum(pa[a]);
            G[a] = quad_sum(G[a]);
            if (P.position_features) pa[a] += fa[P.F - D + a];  // adjoint.rs:118-122
        }
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            if (c0 + u >= S) continue;
            float acc = fa[c0 + u] + vk * (B[u] - T[u]);  // the identity rows (adjoint.rs:68-71) and both roles
            if (sg) {
#pragma unroll
                for (int a = 0; a < D; ++a) acc = fmaf(-own.rg(u, a), G[a], acc);
            }
            A.state_adj[pk * S + c0 + u] = acc;
        }
        if (q == 0) {
            A.ppos[s] = make_float4(pa[0], pa[1], D == 3 ? pa[D - 1] : 0.0f, 0.0f);
            A.dpos[s] = make_float4(pi[0], pi[1], D == 3 ? pi[2] : 0.0f, dens);
        }
    }
}

// accumulate_density_kernel_position_adjoint (adjoint.rs:399-418), gathered: 16 lanes per particle
// take its recorded chunks sixteen slots at a time. Bound: the round trips of the chunks' records.
// Measured as k_adj_prep: 57 us with a thread per particle and 24 us with one chunk in flight -> 17 us
// (2D), 181 -> 21 us (3D).
template <int D>
__global__ __launch_bounds__(256) void k_adj_density_kernel(StepParams P, AdjointArgs A) {
    constexpr uint32_t MAXC = max_chunks(D);
    const uint32_t row = (blockIdx.y * gridDim.x + blockIdx.x) * 16 + threadIdx.x / 16, l = threadIdx.x % 16;
    if (row >= *A.row_count) return;  // whole 16-lane groups leave together
    const uint32_t s = A.act_rows[row];
    const uint32_t b = s / P.N;
    const float4 own = A.dpos[s];
    const float pk[3] = {own.x, own.y, own.z};
    float pa[3] = {0.0f, 0.0f, 0.0f};
    auto add = [&](const float4& o, bool test) {
        float d[3];
        d[0] = delta_axis(pk[0], o.x, 0, P.g);
        d[1] = delta_axis(pk[1], o.y, 1, P.g);
        d[2] = 0.0f;
        float r2 = d[0] * d[0];
        r2 += d[1] * d[1];
        if constexpr (D == 3) {
            d[2] = delta_axis(pk[2], o.z, 2, P.g);
            r2 += d[2] * d[2];
        }
        if (test && !(r2 < P.g.eps2)) return;
        const float x = P.g.eps2 - r2;
        const float w = 6.0f * P.g.k6 * (x * x) * (o.w + own.w);
#pragma unroll
        for (int a = 0; a < D; ++a) pa[a] = fmaf(w, d[a], pa[a]);
    };
    const uint32_t nc = A.nb_count[row];
    if (nc <= MAXC) {
        // three chunks at a time, the next three's records and these chunks' first sixteen slots (all that
        // most cells hold) in flight together
        constexpr int U = 3;
        uint64_t mask[U];
        uint32_t base[U];
        auto fetch = [&](uint32_t c0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t c = c0 + u;
                mask[u] = c < nc ? A.nb_mask[(uint64_t)row * MAXC + c] : 0ull;
                base[u] = c < nc ? A.nb_base[(uint64_t)row * MAXC + c] : 0u;
            }
        };
        fetch(0);
        for (uint32_t c = 0; c < nc; c += U) {
            uint64_t m[U];
            uint32_t at[U];
            float4 o[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                m[u] = mask[u] >> l;
                at[u] = base[u] + l;
                o[u] = m[u] & 1ull ? A.dpos[at[u]] : own;  // the particle itself adds nothing (d = 0)
            }
            fetch(c + U);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                add(o[u], false);
#pragma unroll
                for (uint32_t i = 1; i < 4; ++i)
                    if ((m[u] >> (16 * i)) & 1ull) add(A.dpos[at[u] + 16 * i], false);
            }
        }
    } else {  // more chunks than were recorded: test the candidates of the 3^D cells
        float pi[3];
        int ci[3];
        load_rec<D>(A.srec, A.scoord, s, pi, ci);
        for (int k = 0; k < (D == 3 ? 27 : 9); ++k) {
            const int64_t n0 = (int64_t)ci[0] + k % 3 - 1, n1 = (int64_t)ci[1] + (k / 3) % 3 - 1;
            const int64_t n2 = D == 3 ? (int64_t)ci[2] + k / 9 - 1 : 0;
            uint32_t beg = 0, end = 0;
            bool filter = false;
            if (!cell_range(P, A.bo, b, n0, n1, n2, beg, end, filter)) continue;
            for (uint32_t j = beg + l; j < end; j += 16) {
                if (filter) {
                    float pj[3];
                    int cj[3];
                    load_rec<D>(A.srec, A.scoord, j, pj, cj);
                    if ((int64_t)cj[0] != n0 || (int64_t)cj[1] != n1 || (D == 3 && (int64_t)cj[2] != n2)) continue;
                }
                add(A.dpos[j], true);
            }
        }
    }
#pragma unroll
    for (int a = 0; a < D; ++a) {
        pa[a] = quad_sum(pa[a]);
        pa[a] += __shfl_xor(pa[a], 4, 16);
        pa[a] += __shfl_xor(pa[a], 8, 16);
    }
    if (l == 0) {
        const float4 p0 = A.ppos[s];
        A.pos_adj[(uint64_t)b * P.N + A.perm[s]] = make_float4(p0.x + pa[0], p0.y + pa[1], D == 3 ? p0.z + pa[2] : 0.0f, 0.0f);
    }
}

template <int D, int SM>
static hipError_t launch_adjoint_t(const StepParams& p, const AdjointArgs& a, hipStream_t stream) {
    // a launch's row of blocks holds fewer than 2^32 threads: past 2^24 particles a block of the pair kernels takes
    // several sixteens, and the density kernel's blocks have more rows
    const uint32_t sixteens = (p.T + 15) / 16;
    const dim3 waves(std::min(sixteens, 1u << 20)), blocks(waves.x, (sixteens + waves.x - 1) / waves.x);
    hipLaunchKernelGGL((k_adj_prep<D, SM>), waves, dim3(64), 0, stream, p, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_adj_gather<D, SM>), waves, dim3(64), 0, stream, p, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_adj_density_kernel<D>, blocks, dim3(256), 0, stream, p, a);
    return hipGetLastError();
}

template <int D>
static hipError_t launch_adjoint_d(const StepParams& p, const AdjointArgs& a, hipStream_t stream) {
    switch (p.SS) {
        case 4: return launch_adjoint_t<D, 4>(p, a, stream);
        case 8: return launch_adjoint_t<D, 8>(p, a, stream);
        case 16: return launch_adjoint_t<D, 16>(p, a, stream);
        case 24: return launch_adjoint_t<D, 24>(p, a, stream);
        default: return launch_adjoint_t<D, 32>(p, a, stream);
    }
}

template <int D>
static size_t row_floats(uint32_t SS) {
    switch (SS) {
        case 4: return AdjRow<D, 4>::FLOATS;
        case 8: return AdjRow<D, 8>::FLOATS;
        case 16: return AdjRow<D, 16>::FLOATS;
        case 24: return AdjRow<D, 24>::FLOATS;
        default: return AdjRow<D, 32>::FLOATS;
    }
}

hipError_t launch_perceive_adjoint(const StepParams& p_in, Workspace& ws, AdjointWorkspace& aw, const float* fadj,
                                   float* state_adj, float4* pos_adj, int grid_blocks, hipStream_t stream) {
    if (p_in.T == 0) return hipSuccess;
    const uint64_t T = p_in.T;
    if (T * 8 >= (1ull << 32)) return hipErrorInvalidValue;
    StepParams p = p_in;
    p.dir_n = ws.dir_n.as<uint32_t>();
    p.dir_e = ws.dir_e.as<int4>();
    const bool d3 = p.g.dim == 3;
    hipError_t e;
    if ((e = aw.rows.reserve(T * (d3 ? row_floats<3>(p.SS) : row_floats<2>(p.SS)) * 4)) != hipSuccess) return e;
    if ((e = aw.side.reserve(T * (d3 ? kSide<3> : kSide<2>) * 4)) != hipSuccess) return e;
    if ((e = aw.dpos.reserve(T * 16)) != hipSuccess) return e;
    if ((e = aw.ppos.reserve(T * 16)) != hipSuccess) return e;
    if ((e = launch_density(p, ws, nullptr, grid_blocks, stream, nullptr)) != hipSuccess) return e;
    AdjointArgs a{};
    a.srec = ws.srec.as<float4>();
    a.scoord = ws.scoord.as<int4>();
    a.bo = ws.bin_offsets.as<uint32_t>();
    a.perm = ws.perm.as<uint32_t>();
    a.act_rows = ws.act_rows.as<uint32_t>();
    a.row_count = ws.wl_count.as<uint32_t>() + 1;
    a.nb_base = ws.nb_base.as<uint32_t>();
    a.nb_mask = ws.nb_mask.as<uint64_t>();
    a.nb_count = ws.nb_count.as<uint32_t>();
    a.svol = ws.svol.as<float4>();
    a.sstate = ws.sstate.as<float>();
    a.fadj = fadj;
    a.rows = aw.rows.as<float>();
    a.side = aw.side.as<float>();
    a.dpos = aw.dpos.as<float4>();
    a.ppos = aw.ppos.as<float4>();
    a.state_adj = state_adj;
    a.pos_adj = pos_adj;
    return d3 ? launch_adjoint_d<3>(p, a, stream) : launch_adjoint_d<2>(p, a, stream);
}

void AdjointWorkspace::release() {
    for (DevBuf* b : {&rows, &side, &dpos, &ppos}) b->release();
}

}  // namespace npa
