// CSR fill of a FullGridCellList's neighbour lists with rows that come out sorted
// (PrecomputedNeighborhoodSearch, src/nhs_precomputed.jl:187-206; sorteach!,
// src/vector_of_vectors.jl:177-212) on gfx950: one wavefront per non-empty query cell.
//
// The candidates of a cell, the points of the cells around it, are brought into the order of their
// original indices once, by a bitonic network over up to 2048 keys in registers.  Every query of
// the cell then takes the candidates 64 at a time in that order, and a step appends its accepted
// ones to the row with one contiguous store: a row is ascending as it is written.
//
// VALU issue bounds it: 2 M points with 113 neighbours each and 729 candidates a cell, Float32,
// spend 345 us on the network and a dozen instructions per 64 pairs on the test and the store; the
// stores themselves are 140 us.  The fill by k_cells and the separate sort of the rows took 1300 us
// (Float64 1590), this takes 1130 (1530); 512,000 points at r = 3.2 spacings 528 -> 417 (654 -> 492),
// at 2.5 254 -> 202 (300 -> 235).  The wavefronts in flight decide: with the candidates' coordinates
// staged in LDS, which costs half of them, it took 1350 to 1680 us.
#pragma once

#include "pn_lists.h"
#include "pn_runs.h"

namespace pn {

constexpr int FILL_CAP = 32 * WAVE;  // most candidates of a cell

// inv[sorted_idx[p]] = p
static __global__ __launch_bounds__(256) void k_invert(const int32_t* __restrict__ sorted_idx,
                                                const DevStatus* __restrict__ st, int32_t* __restrict__ inv) {
    const int n = st->n_binned;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) inv[sorted_idx[p]] = p;
}

// Status of a list count: st[0] as k_reset_status leaves it; st[1] the grid's own, with n_ordered for
// k_list_counts.
static __global__ void k_list_status(const DevStatus* __restrict__ grid_st, DevStatus* __restrict__ st) {
    DevStatus s = {};
    s.first_bad = s.bad_now = ~0ull;
    st[0] = s;
    s = *grid_st;
    s.n_ordered = 0;
    st[1] = s;
}

// Clears the counts of a list count's rows and counts, among FILL_SAMPLES pairs of neighbouring sorted
// positions spread over the grid's points, those whose original indices differ by two at most (in the
// same launch, which it does not lengthen; one of its own took 7 us).
constexpr int FILL_SAMPLES = 4096;
static __global__ __launch_bounds__(256) void k_list_counts(int32_t* __restrict__ counts, int64_t n,
                                                            const int32_t* __restrict__ sorted_idx,
                                                            DevStatus* __restrict__ st) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < FILL_SAMPLES) {  // whole wavefronts
        const int n_binned = st[1].n_binned;
        bool near = false;
        if (n_binned >= 2) {
            const int p = (int)(t * (n_binned - 1) / FILL_SAMPLES);
            const int64_t step = (int64_t)sorted_idx[p + 1] - sorted_idx[p];
            near = step >= -2 && step <= 2;
        }
        const int in_wave = __popcll(__ballot(near));
        if ((threadIdx.x & (WAVE - 1)) == 0) atomicAdd(&st[1].n_ordered, in_wave);
    }
    for (int64_t i = t; i < n; i += (int64_t)gridDim.x * blockDim.x) counts[i] = 0;
}

__device__ __forceinline__ float lane_value(float v, int l) {
    return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

struct FillArgs {
    const int32_t* inv;  // sorted position of an original index
    const int32_t* row_ptr;
    int32_t* col;
    int base;
};

// The original indices of a cell's candidates (at most 64 K) in ascending order into s_key; INT32_MAX
// after the last.
template <int D, int K>
__device__ __forceinline__ void sort_candidates(const SetView& Gs, const RunPieces<D, false>& pc, int* s_key) {
    const int lane = threadIdx.x & (WAVE - 1);  // the mask tells the compiler the network's directions
    int v[1][K];
    typename RunPieces<D, false>::Walk walk;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int m = lane + WAVE * j;
        v[0][j] = INT32_MAX;
        if (WAVE * j < pc.M) {  // wave-uniform
            const int p = pc.position(walk, min(WAVE * j + WAVE, pc.M) - 1, m);
            if (m < pc.M) v[0][j] = Gs.sorted_idx[p];
        }
    }
    bitonic_sizes<K, 1, 2>(v, lane);
#pragma unroll
    for (int j = 0; j < K; ++j) s_key[WAVE * j + lane] = v[0][j];
}

template <int D, class TC, class TR>
__global__ __launch_bounds__(WAVE, 6) void k_fill_sorted(Geom g, SetView Q, SetView Gs, TR r2, FillArgs a, int n_keys,
                                                         int nblocks) {
    constexpr int NQ = sizeof(TC) == 4 ? 14 : 6;  // scalar registers: 12 and 9, 16 and 8 lose 5 to 20 %
    extern __shared__ int s_key[];  // as many keys as the network sorts
    const int lane = threadIdx.x;
    const TC* qc = (const TC*)Q.coords;
    const TC* gc = (const TC*)Gs.coords;
    const int n_work = Q.st->n_nonempty;
    const int xcd = blockIdx.x & 7, per_xcd = nblocks >> 3;
    const int wchunk = (n_work + 7) >> 3;
    const int w_end = min(n_work, (xcd + 1) * wchunk);
    for (int w = xcd * wchunk + (int)(blockIdx.x >> 3); w < w_end; w += per_xcd) {
        const int cell = Q.nonempty[w];
        RunDesc rd;
        rd.n0 = g.n[0];
        rd.n1 = g.n[1];
        const int yz = cell / rd.n0;
        rd.row = yz * rd.n0;
        rd.ca = rd.cb = cell - rd.row;
        RunPieces<D, false> pc;
        pc.set(g, Gs, rd);
        pc.M = min(pc.M, n_keys);  // the caller sized n_keys for the fullest cell
        __syncthreads();
        if (pc.M <= 4 * WAVE) sort_candidates<D, 4>(Gs, pc, s_key);
        else if (pc.M <= 8 * WAVE) sort_candidates<D, 8>(Gs, pc, s_key);
        else if (pc.M <= 16 * WAVE) sort_candidates<D, 16>(Gs, pc, s_key);
        else sort_candidates<D, 32>(Gs, pc, s_key);
        __syncthreads();
        const int qs = Q.start[cell], qe = Q.start[cell + 1];
        for (int q0 = qs; q0 < qe; q0 += NQ) {
            const int nq = min(NQ, qe - q0);
            // the queries in scalar registers: coordinates, next slot of the row, its end
            TC x[NQ][D];
            int at[NQ], end[NQ];
            {
                const int k = q0 + min(lane, nq - 1);
                const int64_t i = Q.sorted_idx[k];
                const int at_l = a.row_ptr[i], end_l = a.row_ptr[i + 1];
                TC x_l[D];
#pragma unroll
                for (int d = 0; d < D; ++d) x_l[d] = qc[(int64_t)d * Q.cap + k];
#pragma unroll
                for (int u = 0; u < NQ; ++u) {
                    at[u] = __builtin_amdgcn_readlane(at_l, u);
                    end[u] = __builtin_amdgcn_readlane(end_l, u);
#pragma unroll
                    for (int d = 0; d < D; ++d) x[u][d] = lane_value(x_l[d], u);
                }
            }
            auto load = [&](int m0, int& key, TC (&y)[D]) {
                key = s_key[m0 + lane];
                const bool valid = key != INT32_MAX;
                const int p = valid ? a.inv[key] : 0;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const TC c = gc[(int64_t)d * Gs.cap + p];
                    y[d] = valid ? c : (TC)NAN;  // never within the radius
                }
            };
            int key;
            TC y[D];
            load(0, key, y);
#pragma unroll 1
            for (int m0 = 0; m0 < pc.M; m0 += WAVE) {
                int key_n = 0;
                TC y_n[D] = {};
                if (m0 + WAVE < pc.M) load(m0 + WAVE, key_n, y_n);
                const int value = key + a.base;
#pragma unroll
                for (int u = 0; u < NQ; ++u) {
                    if (u < nq) {
                        TR pd = (TR)(x[u][0] - y[0]);
                        TR d2 = pd * pd;
#pragma unroll
                        for (int d = 1; d < D; ++d) {
                            pd = (TR)(x[u][d] - y[d]);
                            const TR p2 = pd * pd;
                            d2 = d2 + p2;
                        }
                        const unsigned long long mask = __builtin_amdgcn_ballot_w64(d2 <= r2);
                        if (mask) {
                            const unsigned slot = __builtin_amdgcn_mbcnt_hi(
                                (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
                            // a row that would overflow: coordinates moved after the count
                            const int n = max(min((int)__builtin_popcountll(mask), end[u] - at[u]), 0);
                            if (d2 <= r2 && slot < (unsigned)n) (a.col + at[u])[slot] = value;
                            at[u] += n;
                        }
                    }
                }
                key = key_n;
#pragma unroll
                for (int d = 0; d < D; ++d) y[d] = y_n[d];
            }
        }
    }
}

}  // namespace pn
