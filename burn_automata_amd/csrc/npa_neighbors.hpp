// npa_neighbors.hpp - neighbour-cell lookups shared by the neighbour passes (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "npa_internal.hpp"

namespace npa {

// A neighbour cell's run is walked in chunks of kNbChunk consecutive slots; the density pass
// records one accept mask per chunk.
constexpr int kNbChunk = 64;

__device__ __forceinline__ int readlane_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Candidate slots of neighbour cell (n0, n1, n2) of system b: in Particle mode the cell's own run
// of its split bin (no coordinate test needed) or, for an unsplit bin, the whole bin with
// `filter` set; in Grid mode the cell's bin. False when the cell holds no particle.
__device__ __forceinline__ bool cell_range(const StepParams& P, const uint32_t* __restrict__ bo, uint32_t b,
                                           int64_t n0, int64_t n1, int64_t n2, uint32_t& beg, uint32_t& end,
                                           bool& filter) {
    uint32_t cell;
    if (!cell_index(n0, n1, n2, P.g, &cell)) return false;
    const uint64_t bin = (uint64_t)b * P.g.cells + cell;
    filter = false;
    if (P.g.mode != 1) {
        beg = bo[bin];
        end = bo[bin + 1];
        return beg < end;
    }
    // the bin's directory size, its first entry and its end: all that a bin of one cell (most
    // bins) needs
    const int4* e = P.dir_e + bin * kDirGroups;
    const uint32_t nd = P.dir_n[bin];
    const int4 e0 = e[0];
    const uint32_t last = bo[bin + 1];
    if (nd == 0) return false;
    if (nd > kDirGroups) {
        beg = bo[bin];
        end = last;
        filter = true;
        return true;
    }
    if (nd == 1) {
        if ((int64_t)e0.x != n0 || (int64_t)e0.y != n1 || (int64_t)e0.z != n2) return false;
        beg = (uint32_t)e0.w;
        end = last;
        return true;
    }
    // several cells: the directory entries are loaded four at a time (each half's loads issued
    // together); a run ends where the next entry's run starts, the last one at the bin's end
    bool found = false;
    int hit_k = -1;
#pragma unroll
    for (uint32_t h = 0; h < kDirGroups; h += 4) {
        if (h >= nd) break;
        int4 ek[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) ek[k] = h + k < nd ? e[h + k] : make_int4(0, 0, 0, 0);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool hit = !found && h + k < nd && (int64_t)ek[k].x == n0 && (int64_t)ek[k].y == n1 &&
                             (int64_t)ek[k].z == n2;
            if (hit) {
                beg = (uint32_t)ek[k].w;
                hit_k = (int)(h + k);
                found = true;
            }
        }
    }
    if (found) end = (uint32_t)hit_k + 1 < nd ? (uint32_t)e[hit_k + 1].w : last;
    return found;
}

// cell_range for NU cells of one lane at once: every cell's directory loads (its size, first
// entry and end; a Grid-mode cell's start and end) are issued before the first is used, so the
// lookups cost one memory round trip instead of NU. A cell not wanted, outside a clamped grid or
// empty gets beg = end = 0. Bins of several cells (rare) finish through cell_range.
template <int NU>
__device__ __forceinline__ void cell_ranges(const StepParams& P, const uint32_t* __restrict__ bo, uint32_t b,
                                            const int64_t (&n)[NU][3], const bool (&want)[NU], uint32_t (&beg)[NU],
                                            uint32_t (&end)[NU], bool (&filter)[NU]) {
    uint64_t bin[NU];
    bool ok[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        uint32_t cell = 0;
        ok[u] = want[u] && cell_index(n[u][0], n[u][1], n[u][2], P.g, &cell);
        bin[u] = (uint64_t)b * P.g.cells + cell;
        beg[u] = 0;
        end[u] = 0;
        filter[u] = false;
    }
    if (P.g.mode != 1) {
        uint32_t lo[NU], hi[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            lo[u] = ok[u] ? bo[bin[u]] : 0u;
            hi[u] = ok[u] ? bo[bin[u] + 1] : 0u;
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            beg[u] = lo[u];
            end[u] = hi[u];
        }
        return;
    }
    uint32_t nd[NU], last[NU];
    int4 e0[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        nd[u] = ok[u] ? P.dir_n[bin[u]] : 0u;
        e0[u] = ok[u] ? P.dir_e[bin[u] * kDirGroups] : make_int4(0, 0, 0, 0);
        last[u] = ok[u] ? bo[bin[u] + 1] : 0u;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        if (nd[u] == 1) {
            if ((int64_t)e0[u].x == n[u][0] && (int64_t)e0[u].y == n[u][1] && (int64_t)e0[u].z == n[u][2]) {
                beg[u] = (uint32_t)e0[u].w;
                end[u] = last[u];
            }
        } else if (nd[u] != 0) {
            uint32_t bb = 0, ee = 0;
            bool ff = false;
            if (cell_range(P, bo, b, n[u][0], n[u][1], n[u][2], bb, ee, ff)) {
                beg[u] = bb;
                end[u] = ee;
                filter[u] = ff;
            }
        }
    }
}

// The candidate runs of the 3^D neighbour cells of cell (c0, c1, c2) of system b, looked up in
// parallel: lane k < 3^D takes neighbour k in the reference's visit order (k = (dz+1)*9 +
// (dy+1)*3 + (dx+1): dz, then dy, then dx). found: the cell holds particles.
template <int D>
__device__ __forceinline__ void neighbor_runs(const StepParams& P, const uint32_t* __restrict__ bo, uint32_t b,
                                              int c0, int c1, int c2, uint32_t lane, uint32_t& beg, uint32_t& end,
                                              bool& filter, bool& found) {
    constexpr uint32_t NC = D == 3 ? 27 : 9;
    beg = end = 0;
    filter = false;
    found = false;
    if (lane >= NC) return;
    const int dx = (int)(lane % 3) - 1, dy = (int)((lane / 3) % 3) - 1, dz = D == 3 ? (int)(lane / 9) - 1 : 0;
    found = cell_range(P, bo, b, (int64_t)c0 + dx, (int64_t)c1 + dy, (int64_t)c2 + dz, beg, end, filter);
}

// Value of lane (group base + j) for groups of L consecutive lanes (L = 1, 2 or 4), via DPP.
// quad_perm reads a valid lane for every lane, so bound_ctrl (zero for an invalid source lane)
// never applies; with it set the compiler folds the permutation into the consuming VALU
// instruction (v_mul_f32_dpp, v_add_f32_dpp) instead of issuing a separate move.
template <int L, int J>
__device__ __forceinline__ float group_bcast(float v) {
    if constexpr (L == 1) {
        return v;
    } else if constexpr (L == 2) {
        constexpr int c = J == 0 ? (0 | (0 << 2) | (2 << 4) | (2 << 6)) : (1 | (1 << 2) | (3 << 4) | (3 << 6));
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), c, 0xf, 0xf, true));
    } else {
        constexpr int c = J | (J << 2) | (J << 4) | (J << 6);
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), c, 0xf, 0xf, true));
    }
}

// OR of a 64-bit value over each group of L consecutive lanes (L = 1, 2 or 4), via DPP.
template <int L>
__device__ __forceinline__ uint64_t group_or(uint64_t m) {
    if constexpr (L == 1) return m;
    uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
    constexpr int swap1 = 1 | (0 << 2) | (3 << 4) | (2 << 6);  // quad_perm [1,0,3,2]
    lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, swap1, 0xf, 0xf, true);
    hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, swap1, 0xf, 0xf, true);
    if constexpr (L == 4) {
        constexpr int swap2 = 2 | (3 << 2) | (0 << 4) | (1 << 6);  // quad_perm [2,3,0,1]
        lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, swap2, 0xf, 0xf, true);
        hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, swap2, 0xf, 0xf, true);
    }
    return ((uint64_t)hi << 32) | lo;
}

// Per-wave accepted-neighbour lists of the neighbour passes: the sorted slots of each target's accepted
// candidates, appended in visit order (cells dz, dy, dx; slots ascending), so walking a list front
// to back is the reference's neighbour order. kListBytes of LDS per wave for any targets-per-item.
constexpr int kListBytes = 12288;

template <int TPI>
struct PerceiveLists {
    static constexpr int CAP = kListBytes / (4 * TPI);
    uint32_t slot[CAP][TPI];
};

// Bits k of a 64-bit chunk mask with k % L == q.
template <int L>
__device__ __forceinline__ uint64_t residue_mask(uint32_t q) {
    if constexpr (L == 1) return ~0ull;
    else if constexpr (L == 2) return 0x5555555555555555ull << q;
    else return 0x1111111111111111ull << q;
}

// Appends each target's accepted candidates to its list in visit order: from the accept masks the
// density pass recorded (the same test on the same candidates), or, where a target of the wave has
// more chunks than were recorded, by testing the candidates here. Lane q of the L lanes of target t
// holds its position pi, cell ci and compact row; `flush` consumes the lists and empties them (cnt = 0)
// before one would overflow. The caller flushes what is left at the end.
template <int D, int L, class Lists, class Flush>
__device__ __forceinline__ void append_accepted(const StepParams& P, const float4* __restrict__ srec,
                                                const int4* __restrict__ scoord, const uint32_t* __restrict__ bo,
                                                const uint32_t* __restrict__ nb_base,
                                                const uint64_t* __restrict__ nb_mask,
                                                const uint32_t* __restrict__ nb_count, uint32_t row, bool active,
                                                uint32_t b, const float* pi, const int* ci, uint32_t lane, uint32_t t,
                                                uint32_t q, Lists& lists, uint32_t& cnt, Flush&& flush) {
    constexpr uint32_t MAXC = max_chunks(D), CAP = Lists::CAP;
    static_assert(CAP >= (uint32_t)kNbChunk, "an emptied list takes a whole chunk");
    const uint64_t my_residue = residue_mask<L>(q);
    // Phase A. The density pass recorded each target's accepted candidates per chunk, in visit
    // order; the lists are built from those masks (RB chunk records loaded per batch).
    const uint32_t nct = active ? nb_count[row] : 0u;
    const bool recorded = !__ballot(nct > MAXC);
    constexpr int RB = 2;  // chunk records loaded per batch
    for (uint32_t cb = 0; recorded && __ballot(cb < nct); cb += RB) {
        uint4 rc[RB];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            const uint32_t c = cb + (uint32_t)u;
            if (c < nct) {
                const uint64_t mk = nb_mask[(uint64_t)row * MAXC + c];
                rc[u] = make_uint4(nb_base[(uint64_t)row * MAXC + c], 0u, (uint32_t)mk, (uint32_t)(mk >> 32));
            } else {
                rc[u] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            const uint32_t c = cb + (uint32_t)u;
            const uint64_t acc = ((uint64_t)rc[u].w << 32) | rc[u].z;  // 0 past the target's chunks
            const uint32_t add = (uint32_t)__popcll(acc);
            if (__ballot(cnt + add > CAP)) flush();
            uint64_t mine = acc & my_residue;
            while (mine) {
                const uint32_t k = (uint32_t)__builtin_ctzll(mine);
                mine &= mine - 1;
                const uint32_t pos = cnt + (uint32_t)__popcll(acc & ((1ull << k) - 1ull));
                lists.slot[pos][t] = rc[u].x + k;
            }
            cnt += add;
        }
    }
    // Otherwise (a target with more chunks than were recorded): the coordinate groups of the
    // item, then each group's neighbour cells in order, testing the candidates here.
    uint64_t pending = recorded ? 0ull : __ballot(active);
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int l0 = readlane_i(ci[0], leader), l1 = readlane_i(ci[1], leader);
        const int l2 = D == 3 ? readlane_i(ci[2], leader) : 0;
        const uint32_t lb = (uint32_t)readlane_i((int)b, leader);
        const bool same = active && ci[0] == l0 && ci[1] == l1 && (D == 2 || ci[2] == l2) && b == lb;
        const uint64_t group = __ballot(same) & pending;
        pending &= ~group;
        const bool in_group = (group >> lane) & 1ull;
        uint32_t nb_beg, nb_end;
        bool nb_filter, nb_found;
        neighbor_runs<D>(P, bo, lb, l0, l1, l2, lane, nb_beg, nb_end, nb_filter, nb_found);
        for (uint64_t cells = __ballot(nb_found); cells; cells &= cells - 1) {
            const int nk = __ffsll((unsigned long long)cells) - 1;  // ascending = visit order
            const int64_t n0 = (int64_t)l0 + nk % 3 - 1, n1 = (int64_t)l1 + (nk / 3) % 3 - 1;
            const int64_t n2 = D == 3 ? (int64_t)l2 + nk / 9 - 1 : 0;
            const uint32_t beg = (uint32_t)readlane_i((int)nb_beg, nk);
            const uint32_t end = (uint32_t)readlane_i((int)nb_end, nk);
            const bool filter = readlane_i((int)nb_filter, nk) != 0;
            for (uint32_t base = beg; base < end; base += kNbChunk) {
                const uint32_t m = end - base < (uint32_t)kNbChunk ? end - base : (uint32_t)kNbChunk;
                // batches of 4 candidates per lane: loads first (index clamped to
                // the chunk, so every load is in bounds), then branch-free tests. The boundary and the
                // bin's filter are chosen per chunk: tested by candidate the compiler turns both into
                // selects for every one of them (a step of 60,000 particles, 730 neighbours each, S = 8: 1,108 us,
                // now 987).
                uint64_t acc = 0;
                auto tests = [&](auto periodic, auto filtered) {
#pragma unroll 1
                    for (int i0 = 0; i0 < kNbChunk / L; i0 += 4) {
                        if ((uint32_t)(i0 * L) >= m) break;  // wave-uniform
                        float4 rc[4];
                        int4 cc[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint32_t k = q + (uint32_t)((i0 + u) * L);
                            const uint32_t kc = k < m ? k : m - 1;
                            rc[u] = srec[base + kc];
                            if constexpr (D == 3 && filtered) cc[u] = scoord[base + kc];
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint32_t k = q + (uint32_t)((i0 + u) * L);
                            const float4 r = rc[u];
                            bool ok = in_group & (k < m);
                            if constexpr (filtered && D == 2)
                                ok = ok & ((int64_t)__float_as_int(r.z) == n0) & ((int64_t)__float_as_int(r.w) == n1);
                            if constexpr (filtered && D == 3)
                                ok = ok & ((int64_t)cc[u].x == n0) & ((int64_t)cc[u].y == n1) & ((int64_t)cc[u].z == n2);
                            const float d0 = delta_axis_as<periodic>(pi[0], r.x, 0, P.g);
                            const float d1 = delta_axis_as<periodic>(pi[1], r.y, 1, P.g);
                            float r2 = d0 * d0;
                            r2 += d1 * d1;
                            if constexpr (D == 3) {
                                const float d2 = delta_axis_as<periodic>(pi[2], r.z, 2, P.g);
                                r2 += d2 * d2;
                            }
                            acc |= (ok & (r2 < P.g.eps2)) ? (1ull << (k & 63u)) : 0ull;
                        }
                    }
                };
                if (P.g.boundary == 0) {
                    if (filter) tests(std::true_type{}, std::true_type{});
                    else tests(std::true_type{}, std::false_type{});
                } else {
                    if (filter) tests(std::false_type{}, std::true_type{});
                    else tests(std::false_type{}, std::false_type{});
                }
                acc = group_or<L>(acc);
                const uint32_t add = (uint32_t)__popcll(acc);
                if (__ballot(cnt + add > CAP)) flush();
                uint64_t mine = acc & my_residue;
                while (mine) {
                    const uint32_t k = (uint32_t)__builtin_ctzll(mine);
                    mine &= mine - 1;
                    const uint32_t pos = cnt + (uint32_t)__popcll(acc & ((1ull << k) - 1ull));
                    lists.slot[pos][t] = base + k;
                }
                cnt += add;
            }
        }
    }
}

}  // namespace npa
