// Neighbour traversal by runs of query points (foreach_point_neighbor, hot loop
// src/nhs_grid.jl:519-575) on gfx950: one wavefront per run of up to 32 query points that are
// consecutive in the sorted order and lie in one x-row of cells.
//
// The cells around a run are 3^(D-1) x-rows, each one contiguous range of the sorted order (two
// with a periodic box).  Testing every candidate against every query in the reference's unfused
// arithmetic is nine VALU instructions per 64 pairs; here the matrix cores sort out all but the
// neighbours first, at one instruction per 64 pairs:
//   * Coordinates relative to the run's centre, scaled so that the search radius lies in [1, 2),
//     are split into two Float16 values each (22 bits).  |x_c|^2 + |x_q|^2 - r^2 - 2 x_c . x_q is
//     then one product of 16 terms, and v_mfma_f32_32x32x16_f16 evaluates it for 32 candidates x
//     32 queries.  Lane l holds query l & 31 against half of the candidates.
//   * Its error is below PREFILTER_EPS ((2 |x_q| + r)^2 + r^2) (splits 2^-22 per factor, 16
//     products summed with at most 2^-23 each).  With that margin subtracted, a set sign bit means
//     "maybe a neighbour" and a clear one "certainly not".  A lane collects 16 sign bits of a
//     32-candidate tile in one word, an instruction each.
//   * The pair body then runs over the set bits: one lane, one query, its sums in registers.  It
//     recomputes d^2 in the reference's arithmetic
//         p = convert(T_r, x_i - y_j), d2 = ((p1*p1 + p2*p2) + p3*p3), accept iff d2 <= r*r
//     (src/nhs_grid.jl:547-555, built with -ffp-contract=off), so neighbour sets are exact.
// A run's cells together have candidates that are two cells or more in x from a query's own cell.
// They are further away than r but for the rounding of the cell arithmetic, where the reference
// does not look at them: a pair that close to r is accepted only if its cells are adjacent.  After
// coordinates moved without a new binning a run is one cell, so that the cells of the binning
// decide, as in the reference.  The device says so (DevStatus::moved): a captured traversal may be
// replayed over coordinates that moved since its capture.
// Points for which the estimate cannot be trusted (a query outside its cell after an in-place
// move, a candidate whose other image in a periodic box may be as near) are kept as "maybe" for every pair.
//
// A run has up to 64 lanes for its queries: two per query, four for up to 16 and eight for up to
// 8 queries, which share the query's candidates; their sums are combined in a fixed order, so
// results are deterministic.
#pragma once

#include "pn_sph.h"
#include "pn_traverse.h"

#include <type_traits>

namespace pn {

constexpr int RUN = 32;       // most queries of a run
constexpr int RUN_SPAN = 32;  // cells in x that a run may cover: keeps the split values in range
// A run ends where the next query is this many cells further in x.  Two runs stage fewer candidates
// than one from a gap of 4 cells on, but each starts with a chain of loads of some 5 us: at 4, the
// few points of a thin row made a small cloud wait for eight runs of one (19,200 points in 2D, r = 2.3
// spacings: interact! 21 -> 13 us, count 13.3 -> 9.2; 90,000 at r = 2.8: 25.4 -> 21.0; without such
// rows the same).
constexpr int RUN_GAP = 12;
constexpr float PREFILTER_EPS = 3.8146973e-06f;  // 2^-18
// Squared lengths that decide a pair alone: "certainly not" and "maybe" (|x|^2 stays below 1500,
// and REJECT + MAYBE < 0).
constexpr float PREFILTER_REJECT = 16000.0f, PREFILTER_MAYBE = -60000.0f;

// Scale of the estimate: r * s in [1, 2), s a power of two.
struct RunScale {
    float s;
    float rt;      // r * s
    float per_mg;  // periodic box: additional margin for the subtraction over its length
    // pairs two cells apart have d^2 > r^2 (1 - cell_rel): the rounding of the cell arithmetic
    double cell_rel;
};

// How the sorted positions are cut into runs.
struct RunSplit {
    int n;     // points that the host expects; the kernels read their number on the device
    int most;  // queries of a run, a power of two up to RUN
    int lg_parts;  // 2^lg_parts wavefronts share the runs of a window of `most` positions
    int span;  // cells of a run
    unsigned magic0, magic1;  // floor((2^32 - 1) / cells) in x and y (no batch table)
    int cell64;  // cells are computed in Float64
};

using f32x16 = float __attribute__((ext_vector_type(16)));
using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
using f16x2 = _Float16 __attribute__((ext_vector_type(2)));
using f32x2 = float __attribute__((ext_vector_type(2)));
using u32x4 = unsigned __attribute__((ext_vector_type(4)));

// Float16 splits of a and b, (hi of a, hi of b) and (lo of a, lo of b): hi + lo is the value to
// 22 bits.
__device__ __forceinline__ uint2 split16x2(float a, float b) {
    const f32x2 v = {a, b};
    const f16x2 h = __builtin_convertvector(v, f16x2);
    const f32x2 r = {a - (float)h[0], b - (float)h[1]};
    const f16x2 l = __builtin_convertvector(r, f16x2);
    return uint2{__builtin_bit_cast(unsigned, h), __builtin_bit_cast(unsigned, l)};
}

// One run: queries at sorted positions [q0, q0 + nq) in cells ca .. cb (0-based x) of the x-row
// whose cell x = 0 has index row; cy and cz are the row's 0-based cell coordinates.
struct RunDesc {
    int q0, nq, row, ca, cb, n0, n1, cy, cz;
    double minc[3];
};

// x / n for x < 2^31 and magic = floor((2^32 - 1) / n): the product's high word is the quotient or
// one less (scalar instructions only where x is uniform).
__device__ __forceinline__ unsigned div_magic(unsigned x, unsigned n, unsigned magic) {
    const unsigned q = (unsigned)(((unsigned long long)x * magic) >> 32);
    return x - q * n >= n ? q + 1 : q;
}

// Calls fn(w, part) for the work items of this workgroup: window w holds the sorted positions from
// w * most on, part is which of its 2^lg_parts wavefronts this one is.  An XCD takes consecutive
// windows, the last XCD its own from the last to the first.  Those are the cloud's outer layer in the
// slowest dimension, and one that the cells cut thin has few points a row: its runs cover up to 32
// cells and take some times as long as others, and started last they kept the chip waiting (us, all
// ascending / as here, lattices whose last layer is thin: 512,000 points at r = 2.4 spacings count
// 100 / 69, density 153 / 97; 1 M at 3.2 count 236 / 146, density 401 / 276, interact! 626 / 448).  Other
// clouds lose 1 to 2 % to the scalar registers that this and the device's number of points take (1.14 M
// points in 64 clouds count 116 / 118, 1 M points density 161 / 162, pressure 188 / 190; all of it computed
// again for each window instead: more spills).
// sp.n shares the windows out, so that no load waits for n, the number of points on the device (0.3 us
// of a launch); where n is larger, the windows behind follow in turn.
template <class Fn>
__device__ __forceinline__ void for_windows(int n, int nblocks, const RunSplit& sp, Fn&& fn) {
    const int n_win = (sp.n + sp.most - 1) / sp.most;
    const int xcd = blockIdx.x & 7, chunk = (n_win + 7) >> 3;
    const int w0 = min(n_win, xcd * chunk), nw = min(n_win, w0 + chunk) - w0;
    for (int k = (int)(blockIdx.x >> 3);; k += nblocks >> 3) {
        const int i = k >> sp.lg_parts, part = k & ((1 << sp.lg_parts) - 1);
        int w;
        if (i < nw) {
            w = w0 + (xcd == 7 ? nw - 1 - i : i);
        } else {
            w = n_win + (i - nw) * 8 + xcd;
            if ((int64_t)w * sp.most >= n) break;
        }
        fn(w, part);
    }
}

// Calls fn(RunDesc) for the runs of window w that are this part's, every 2^lg_parts-th: the window of
// `most` (at most RUN) sorted positions is cut where the x-row changes, where a run would cover more
// than `span` cells (one where the coordinates moved since the binning) and at gaps.
template <int D, class Fn>
__device__ __forceinline__ void for_runs(const Geom& g, const SetView& Q, int w, int part, int n, int moved,
                                         const RunSplit& sp, Fn&& fn) {
    const int lane = threadIdx.x;
    const int p0 = w * sp.most, mask = (1 << sp.lg_parts) - 1;
    int turn = part;
    const int key_l = Q.keys[min((int64_t)p0 + lane, Q.cap - 1)];  // lanes from cnt on are not looked at
    const int cnt = min(sp.most, n - p0);
    asm volatile("" : "+s"(moved));  // not waited for before the keys are on their way
    const int span = moved ? 1 : sp.span;
    const int step = key_l - __shfl_up(key_l, 1, WAVE);
    RunDesc rd;
    rd.n0 = g.n[0];
    rd.n1 = g.n[1];
#pragma unroll
    for (int d = 0; d < 3; ++d) rd.minc[d] = g.minc[d];
    for (int i = 0; i < cnt;) {
        const int key = __builtin_amdgcn_readlane(key_l, i);
        unsigned yz;
        if (g.table) {
            const GeomEntry* e = &g.table[cloud_of_cell(g, key)];
            const int4 dims = *(const int4*)e;  // n[3], cell_off
            rd.n0 = dims.x;
            rd.n1 = dims.y;
#pragma unroll
            for (int d = 0; d < 3; ++d) rd.minc[d] = e->minc[d];
            yz = (unsigned)(key - dims.w) / (unsigned)rd.n0;
            rd.row = dims.w + (int)yz * rd.n0;
            rd.cz = D >= 3 ? (int)(yz / (unsigned)rd.n1) : 0;
        } else {
            yz = div_magic((unsigned)key, (unsigned)rd.n0, sp.magic0);
            rd.row = (int)yz * rd.n0;
            rd.cz = D >= 3 ? (int)div_magic(yz, (unsigned)rd.n1, sp.magic1) : 0;
        }
        rd.cy = (int)yz - rd.cz * rd.n1;
        const int cx = key_l - rd.row;
        rd.ca = key - rd.row;
        const bool cut = lane > i && (lane >= cnt || cx >= min(rd.n0, rd.ca + span) || step >= RUN_GAP);
        const int end = __builtin_ctzll(__builtin_amdgcn_ballot_w64(cut));  // cnt < 64 at the latest
        rd.q0 = p0 + i;
        rd.nq = end - i;
        rd.cb = __builtin_amdgcn_readlane(cx, end - 1);
        if (turn == 0) fn(rd);
        turn = (turn - 1) & mask;
        i = end;
    }
}

// The candidates of a run: pieces of the sorted order, lane u holding the first element and the
// offset to sorted positions of piece u.
template <int D, bool PER>
struct RunPieces {
    static constexpr int R = Rows<D>::R;
    static constexpr int RP = PER ? 2 * R : R;
    int pre_l, rdel_l, M;

    __device__ __forceinline__ void set(const Geom& g, const SetView& Gs, const RunDesc& rd) {
        const int lane = threadIdx.x;
        int rb = 0, rlen = 0;
        if (lane < RP) {
            const int t = PER ? lane >> 1 : lane, piece = PER ? lane & 1 : 0;
            const int dy = D >= 2 ? (t % 3) - 1 : 0, dz = D >= 3 ? (t / 3) - 1 : 0;
            int row, lo = rd.ca - 1, hi = rd.cb + 2;  // cells [lo, hi) of the row
            if constexpr (!PER) {
                row = rd.row + (dy + dz * rd.n1) * rd.n0;
            } else {
                // 0-based periodic cells are 1 .. per; a run leaves two of them out, so its window
                // wraps on one side at most
                auto wrap = [](int c, int per) { return c < 1 ? c + per : (c > per ? c - per : c); };
                const int yy = D >= 2 ? wrap(rd.cy + dy, g.per[1]) : 0, zz = D >= 3 ? wrap(rd.cz + dz, g.per[2]) : 0;
                row = (yy + zz * rd.n1) * rd.n0;
                const int per = g.per[0];
                const bool left = lo < 1, right = hi > per + 1;
                if (piece == 0) {
                    if (left) {
                        lo = per;
                        hi = per + 1;
                    } else if (right) {
                        hi = per + 1;
                    }
                } else {
                    hi = left ? hi : (right ? 2 : 1);
                    lo = 1;
                }
            }
            rb = Gs.start[row + lo];
            rlen = Gs.start[row + hi] - rb;
        }
        // inclusive prefix sums over the first 32 lanes (DPP row shifts, then row 0's last into row 1)
        int sum = rlen;
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, true);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, true);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, true);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x118, 0xf, 0xf, true);
        if constexpr (RP >= 16) sum += __builtin_amdgcn_update_dpp(0, sum, 0x142, 0xa, 0xf, false);
        M = __builtin_amdgcn_readlane(sum, RP - 1);
        pre_l = sum - rlen;
        rdel_l = rb - pre_l;
    }

    // A walk over the elements in ascending order: the piece reached, its first element past the
    // end and its offset, wave-uniform.
    struct Walk {
        int u = -1, end = 0, del = 0;
    };

    // Sorted position of element m; the wavefront's elements are ascending, not below those of the
    // walk's last call, and at most mhi.  Called with every lane active.
    __device__ __forceinline__ int position(Walk& w, int mhi, int m) const {
        int del = w.del;
        while (w.end <= mhi) {  // piece u + 1 starts at w.end
            ++w.u;
            w.del = __builtin_amdgcn_readlane(rdel_l, w.u);
            del = m >= w.end ? w.del : del;
            w.end = __builtin_amdgcn_readlane(pre_l, w.u + 1);
        }
        return m + del;
    }
};

// p[i] with a 32-bit byte offset (one address register beside the uniform base).
template <class T>
__device__ __forceinline__ T load32(const T* p, unsigned i) {
    return *(const T*)((const char*)p + (size_t)(i * (unsigned)sizeof(T)));
}

// Coordinates relative to a run's centre, and the operands of the estimate.  Both hold, for lane l
// with half = l >> 5, the 8 of 16 factors of row (candidate) or column (query) l & 31:
//     candidate   half 0: [xh yh xl yl xh yh 256 256]   half 1: [zh nh zl nl zh nh 256 256]
//     query       half 0: [xh yh xh yh xl yl mh  ml ]   half 1: [zh 256 zh 256 zl 0 0 0]
// of T_c = 16 t_c, -2 T_q, n = |t_c|^2 and m = |t_q|^2 - r^2 - margin, so the product is
// 256 (|t_c - t_q|^2 - r^2 - margin) (without the products of two low parts).
template <int D, class TC, bool PER>
struct RunFrame {
    TC o[D];
    float hq[D];   // bound on |t_d| of the run's queries
    float hc[D];   // ... of the candidates that can be neighbours
    float len[D];  // periodic box
    float near[D];  // ... up to this |t_d| a candidate's image is the nearest to every query within r
    float s, rt, per_mg;

    __device__ __forceinline__ void set(const Geom& g, const RunDesc& rd, const RunScale& sc) {
        s = sc.s;
        rt = sc.rt;
        per_mg = sc.per_mg;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const double lo = d == 0 ? (double)rd.ca : (double)(d == 1 ? rd.cy : rd.cz);
            const double half = d == 0 ? 0.5 * (double)(rd.cb - rd.ca + 1) : 0.5;
            o[d] = (TC)(rd.minc[d] + (lo + half) * g.csd[d]);
            hq[d] = (float)(half * g.csd[d]) * s + 0.01f * rt;
            hc[d] = hq[d] + 1.01f * rt;
            len[d] = PER ? (float)g.box[d] * s : 0.0f;
            // another image of a candidate at t is len - |t| from the centre, so at least
            // len - |t| - hq from a query: further than r.  Half the length alone is not enough
            // where the box has three cells.
            near[d] = fminf(0.499f * len[d], len[d] - hq[d] - 1.01f * rt);
        }
    }

    // T = 16 t of a point; false (PER): the nearest image is not certain
    __device__ __forceinline__ bool relative(const TC (&x)[D], float (&t)[D]) const {
        bool sure = true;
        const float s16 = 16.0f * s;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            t[d] = (float)(x[d] - o[d]) * s16;
            if constexpr (PER) {
                const float l16 = 16.0f * len[d];
                sure = sure && fabsf(t[d]) <= 4.0f * l16;
                t[d] = __builtin_fmaf(-l16, rintf(t[d] / l16), t[d]);
                sure = sure && fabsf(t[d]) <= 16.0f * near[d];
            }
        }
        return sure;
    }

    // The candidate's operand words.  valid = false: never a neighbour.
    // Returns |t|^2; a point far outside (its coordinates moved since the binning) may give any
    // estimate.
    struct Operand {
        uint2 xy, zn;
    };
    __device__ __forceinline__ float candidate(const TC (&x)[D], bool valid, bool& maybe, Operand& op) const {
        float t[3] = {0.0f, 0.0f, 0.0f};
        float tt[D];
        const bool sure = relative(x, tt);
        float n = tt[0] * tt[0];
#pragma unroll
        for (int d = 1; d < D; ++d) n = __builtin_fmaf(tt[d], tt[d], n);
#pragma unroll
        for (int d = 0; d < D; ++d) t[d] = tt[d];
        n *= 0x1p-8f;
        maybe = PER && valid && !sure;
        if constexpr (PER) {
            n = maybe ? PREFILTER_MAYBE : n;
#pragma unroll
            for (int d = 0; d < D; ++d) t[d] = maybe ? 0.0f : t[d];
        }
        n = valid ? n : PREFILTER_REJECT;
        op.xy = split16x2(t[0], t[1]);
        op.zn = split16x2(t[2], n);
        return n;
    }

    // The query operand; margin: subtracted from m (mg receives it).  Returns false where
    // every pair of the query is "maybe" (its coordinates are not where its cell says).
    struct Query {
        f16x8 op;
        float mg;
        bool sure;
    };
    __device__ __forceinline__ Query query(const TC (&x)[D], bool with_margin) const {
        Query q;
        float t[3] = {0.0f, 0.0f, 0.0f};
        float tt[D];
        q.sure = relative(x, tt);
        float n = 0.0f;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            q.sure = q.sure && fabsf(tt[d]) <= 16.0f * hq[d];
            n = __builtin_fmaf(tt[d], tt[d], n);
        }
        n *= 0x1p-8f;
        const float reach = 2.0f * __builtin_amdgcn_sqrtf(n) + rt;
        q.mg = PREFILTER_EPS * (reach * reach + rt * rt) + per_mg;
        const float m = q.sure ? n - rt * rt - (with_margin ? q.mg : 0.0f) : 0.0f;
#pragma unroll
        for (int d = 0; d < D; ++d) t[d] = q.sure ? -2.0f * tt[d] : 0.0f;
        const bool upper = threadIdx.x >= 32;
        const uint2 xy = split16x2(t[0], t[1]), zm = split16x2(t[2], m);
        unsigned w[4];
        w[0] = w[1] = upper ? (zm.x & 0xffffu) | 0x5c000000u : xy.x;  // 0x5c00: 256
        w[2] = upper ? zm.y & 0xffffu : xy.y;
        w[3] = upper ? 0u : (zm.x >> 16) | (zm.y & 0xffff0000u);
        q.op = __builtin_bit_cast(f16x8, w);
        return q;
    }
};

// Place in a block of 64 candidates of the one that lane l loads and holds the operand of: lanes
// 0 .. 31 hold the rows of its first tile of 32, the others those of the second.  Result i (0 .. 15)
// of half h is the product of row 8 (i / 4) + 4 h + i % 4, and element 2 i + h of a tile is put
// there: a query's neighbours, which come in stretches, are shared evenly by its two lanes.
__device__ __forceinline__ int block_place(int l) {
    return (l & 32) + ((l >> 3) & 3) * 8 + (l & 3) * 2 + ((l >> 2) & 1);
}

// Operands of a block's two tiles from the words of its lanes: the first needs the xy words of
// lanes 0 .. 31 in the lower half and their zn words in the upper half, the second the same of
// lanes 32 .. 63, which is one exchange of halves per word.
struct TileOperands {
    f16x8 t[2];
    __device__ __forceinline__ TileOperands(uint2 xy, uint2 zn) {
        const auto a = __builtin_amdgcn_permlane32_swap(xy.x, zn.x, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(xy.y, zn.y, false, false);
        t[0] = __builtin_bit_cast(f16x8, u32x4{a[0], b[0], a[0], 0x5c005c00u});
        t[1] = __builtin_bit_cast(f16x8, u32x4{a[1], b[1], a[1], 0x5c005c00u});
    }
};

template <class Query>
__device__ __forceinline__ f32x16 tile_products(const f16x8& tile, const Query& q) {
    f32x16 zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(tile, q.op, zero, 0, 0, 0);
}

// (w << 16) | sign bits of v, bit i that of v[i].
__device__ __forceinline__ unsigned sign_bits(unsigned w, const f32x16& v) {
#pragma unroll
    for (int i = 15; i >= 0; --i) w = __builtin_amdgcn_alignbit(w, __float_as_uint(v[i]), 31);
    return w;
}

// Whether the lower half of w is zero, as one 16-bit compare.
__device__ __forceinline__ bool low16_zero(unsigned w) {
    unsigned long long m;
    asm("v_cmp_eq_u16 %0, 0, %1" : "=s"(m) : "v"(w));
    return __builtin_amdgcn_inverse_ballot_w64(m);
}

// The lanes of a run: queries per copy of the columns (32, 16 or 8) and the candidates that a
// copy takes (all, every second or every fourth of a lane's 16 of a tile).
struct RunLanes {
    int cols, query, mask;
    __device__ __forceinline__ explicit RunLanes(int nq) {
        const int l = threadIdx.x & 31;
        cols = nq > 16 ? 32 : (nq > 8 ? 16 : 8);
        query = l & (cols - 1);
        const int copy = l / cols;
        mask = (cols == 32 ? 0xffff : (cols == 16 ? 0x5555 : 0x1111)) << copy;
    }
};

// compute_periodic_distance (src/neighborhood_search.jl:428-436): where d2 > r^2 and some
// |pos_diff_d| > 0.49 L_d, pos_diff -= L .* round.(pos_diff ./ L) (half to even) and d2 again;
// elsewhere every round is 0.
template <int D, class TR>
__device__ __forceinline__ TR run_periodic_fix(const TR (&box)[D], TR (&pd)[D], TR d2, TR r2) {
    bool need = false;
#pragma unroll
    for (int d = 0; d < D; ++d) need = need || (fabs(pd[d]) > (TR)0.49 * box[d]);
    need = need && (d2 > r2);
    if (need) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const TR k = rint(pd[d] / box[d]);
            const TR sh = box[d] * k;
            pd[d] = pd[d] - sh;
        }
        d2 = pd[0] * pd[0];
#pragma unroll
        for (int d = 1; d < D; ++d) {
            const TR p2 = pd[d] * pd[d];
            d2 = d2 + p2;
        }
    }
    return d2;
}

// pos_diff and d^2 of a pair in the reference's arithmetic.
template <int D, class TC, class TR, bool PER>
__device__ __forceinline__ TR run_distance(const TC (&x)[D], const Pack<TC, D>& y, const TR (&box)[D], TR r2,
                                           TR (&pd)[D]) {
#pragma unroll
    for (int d = 0; d < D; ++d) pd[d] = (TR)(x[d] - y.v[d]);
    TR d2 = pd[0] * pd[0];
#pragma unroll
    for (int d = 1; d < D; ++d) {
        const TR p2 = pd[d] * pd[d];
        d2 = d2 + p2;
    }
    if constexpr (PER) d2 = run_periodic_fix<D, TR>(box, pd, d2, r2);
    return d2;
}

// 0-based cell in x of a coordinate, in cell_key's arithmetic.  (The empty asm keeps parts of the
// division out of the registers of the pair loop around this rare call.)
template <class TCELL, class TC, bool PER>
__device__ __forceinline__ int run_cell_x(const Geom& g, double minc, TC x) {
    TCELL lo = (TCELL)minc, size = (TCELL)g.csd[0];
    asm volatile("" : "+v"(lo), "+v"(size), "+v"(x));
    const TCELL f = floor(((TCELL)x - lo) / size);
    if constexpr (!PER) return (int)f;
    const int64_t a = (int64_t)((uint64_t)floor_to_int64(f) - 1ull);
    const int64_t m = a % (int64_t)g.per[0];
    return (int)(m < 0 ? m + g.per[0] : m) + 1;
}

// Whether a candidate's cell in x (as of the binning) is adjacent to cell cq.
template <class TC, bool PER>
__device__ __forceinline__ bool run_adjacent(const Geom& g, const RunDesc& rd, int cell64, int cq, TC xc) {
    int d;
    if (sizeof(TC) == 8 || cell64) d = cq - run_cell_x<double, TC, PER>(g, rd.minc[0], xc);
    else d = cq - run_cell_x<float, TC, PER>(g, rd.minc[0], xc);
    d = d < 0 ? -d : d;
    return d <= 1 || (PER && d == g.per[0] - 1) || rd.ca == rd.cb;
}

// A lane's queue of candidates in LDS: words of (byte offset of its first candidate of a tile << 16)
// | 16 bits, bit i for the candidate 2 i places further, in rows of 64 lanes, ending with two zeros.
template <class Rec>
struct LaneQueue {
    unsigned word, next;
    const unsigned* row;  // where next comes from
    __device__ __forceinline__ explicit LaneQueue(const unsigned (*q)[WAVE]) {
        word = q[0][threadIdx.x];
        next = q[1][threadIdx.x];
        row = &q[1][threadIdx.x];
    }
    // The next candidate's byte offset; a used up word is replaced and the one after it loaded.
    __device__ __forceinline__ unsigned pop() {
        const unsigned at = (word >> 16) + (unsigned)__builtin_ctz(word) * (unsigned)(2 * sizeof(Rec));
        word &= word - 1;
        const bool used = low16_zero(word);
        word = used ? next : word;
        row = used ? row + WAVE : row;
        next = *row;
        return at;
    }
};

// Counting (CountF).  Nothing but the signs and the smallest |estimate| of a block of 64 candidates
// is looked at; the pairs that the estimate does not decide (within the margin of the search
// radius: ties of a lattice, one pair in some thousand elsewhere) are queued and tested exactly.
template <int D, class TC, class TR, bool PER>
__global__ __launch_bounds__(WAVE, 4) void k_runs_count(Geom g, SetView Q, SetView Gs, TR r2, CountF f, int nblocks,
                                                        RunScale sc, RunSplit sp) {
    using Rec = Pack<TC, D>;
    constexpr int NB = 6144 / (WAVE * (int)sizeof(Rec)), CAP = NB * WAVE;
    constexpr int G = 1;  // blocks of candidates whose loads are in flight together (2 measured no faster)
    __shared__ Rec s_c[CAP];
    __shared__ unsigned s_q[2 * NB + 2][WAVE];
    const int lane = threadIdx.x, place = block_place(lane);
    const TC* __restrict__ gc = (const TC*)Gs.coords;
    const TC* __restrict__ qcrd = (const TC*)Q.coords;
    TR box[D];
#pragma unroll
    for (int d = 0; d < D; ++d) box[d] = (TR)g.box[d];
    const TR r2_in = r2 - r2 * (TR)sc.cell_rel;  // up to this x distance squared cells are adjacent
    const int n = Q.st->n_binned, moved = Gs.st->moved;
    for_windows(n, nblocks, sp, [&](int w, int part) {
        for_runs<D>(g, Q, w, part, n, moved, sp, [&](const RunDesc& rd) {
            const RunLanes ln(rd.nq);
            const bool qact = ln.query < rd.nq;
            const int qpos = rd.q0 + (qact ? ln.query : 0);
            RunPieces<D, PER> pc;
            pc.set(g, Gs, rd);
            RunFrame<D, TC, PER> fr;
            fr.set(g, rd, sc);
            TC xq[D];
#pragma unroll
            for (int d = 0; d < D; ++d) xq[d] = qcrd[(int64_t)d * Q.cap + qpos];
            const auto qr = fr.query(xq, false);
            const float mg = 256.0f * (qr.mg + sc.rt * sc.rt * (float)sc.cell_rel);
            // |t|^2 of a candidate that can be a neighbour of a query in its place
            float nmax = 0.0f;
#pragma unroll
            for (int d = 0; d < D; ++d) nmax = __builtin_fmaf(fr.hc[d], fr.hc[d], nmax);
            const unsigned some = qact ? (unsigned)ln.mask : 0u;  // the lane's candidates of a tile
            int count = 0;
            typename RunPieces<D, PER>::Walk walk;
            for (int p0 = 0; p0 < pc.M; p0 += CAP) {
                const int pe = min(p0 + CAP, pc.M);
                int qn = 0;
                for (int b0 = p0; b0 < pe; b0 += G * WAVE) {
                    TC cx[G][D];
#pragma unroll
                    for (int gi = 0; gi < G; ++gi) {
                        const int m0 = b0 + gi * WAVE;
                        if (m0 < pe) {
                            const int mhi = min(m0 + WAVE, pe) - 1;
                            const unsigned src = (unsigned)pc.position(walk, mhi, min(m0 + place, mhi));
#pragma unroll
                            for (int d = 0; d < D; ++d) cx[gi][d] = load32(gc + (int64_t)d * Gs.cap, src);
                        }
                    }
#pragma unroll
                    for (int gi = 0; gi < G; ++gi) {
                        const int m0 = b0 + gi * WAVE;
                        if (m0 >= pe) break;
                        const bool valid = m0 + place < pe;
                        bool maybe;
                        typename RunFrame<D, TC, PER>::Operand op;
                        const float nn = fr.candidate(cx[gi], valid, maybe, op);
                        // a candidate moved far away since the binning (or not a number): no neighbour
                        // of a query in its place, tested exactly for the others
                        const bool far = !(nn <= nmax);
                        if (__builtin_amdgcn_ballot_w64(far)) {
                            if (far) {
                                op.xy = uint2{0u, 0u};
                                op.zn = split16x2(0.0f, PREFILTER_REJECT);
                            }
                        }
                        const bool exact = __builtin_amdgcn_ballot_w64((PER && maybe) || !qr.sure);
                        Rec pk;
#pragma unroll
                        for (int d = 0; d < (D == 3 ? 4 : D); ++d) pk.v[d] = d < D ? cx[gi][d] : (TC)0;
                        if (!valid) pk.v[0] = (TC)INFINITY;
                        const int e0 = m0 - p0;
                        s_c[e0 + place] = pk;
                        const TileOperands tiles(op.xy, op.zn);
                        unsigned bits = 0;
#pragma unroll
                        for (int t = 1; t >= 0; --t) {
                            const f32x16 v = tile_products(tiles.t[t], qr);
                            bits = sign_bits(bits, v);
                            float least = INFINITY;
#pragma unroll
                            for (int i = 0; i < 16; i += 2) least = fminf(fminf(fabsf(v[i]), fabsf(v[i + 1])), least);
                            if (exact || __builtin_amdgcn_ballot_w64(least <= mg)) {
                                f32x16 u;
#pragma unroll
                                for (int i = 0; i < 16; ++i) u[i] = fabsf(v[i]) - mg;
                                unsigned open = sign_bits(0u, u);
                                if (exact) {
                                    // "maybe" candidates lie far below any estimate (256 (|t_c - t_q|^2 - r^2) >
                                    // -1024 with r < 2); a query out of its place has all pairs open
#pragma unroll
                                    for (int i = 0; i < 16; ++i) u[i] = v[i] + 1100.0f;
                                    open |= qr.sure ? sign_bits(0u, u) : 0xffffu;
                                }
                                bits &= ~open;
                                open &= some;
                                if (open) {
                                    const unsigned first = (unsigned)((e0 + 32 * t + (lane >> 5)) * (int)sizeof(Rec));
                                    s_q[qn][lane] = (first << 16) | open;
                                    ++qn;
                                }
                            }
                        }
                        count += __builtin_popcount(bits & (some | (some << 16)));
                    }
                }
                if (__builtin_amdgcn_ballot_w64(qn != 0)) {
                    s_q[qn][lane] = 0;
                    s_q[qn + 1][lane] = 0;
                    __syncthreads();
                    LaneQueue<Rec> q(s_q);
                    auto test = [&](const Rec& y) {
                        TR pd[D];
                        const TR d2 = run_distance<D, TC, TR, PER>(xq, y, box, r2, pd);
                        bool in = d2 <= r2;
                        if (in && pd[0] * pd[0] > r2_in)
                            in = run_adjacent<TC, PER>(g, rd, sp.cell64, Q.keys[qpos] - rd.row, y.v[0]);
                        count += in;
                    };
                    auto record = [&](unsigned at) { return *(const Rec*)((const char*)s_c + at); };
                    while (q.word) {
                        const Rec y0 = record(q.pop());
                        const bool two = q.word != 0;
                        Rec y1;
                        if (two) y1 = record(q.pop());
                        test(y0);
                        if (two) test(y1);
                    }
                }
                __syncthreads();
            }
            count += __shfl_xor(count, 32, WAVE);
            if (ln.cols <= 16) count += __shfl_xor(count, 16, WAVE);
            if (ln.cols <= 8) count += __shfl_xor(count, 8, WAVE);
            if (lane < ln.cols && qact) f.write(Q.sorted_idx[qpos], Empty{}, count);
        });
    });
}

// fn(f), with a smoothing kernel's kind as a constant (no branch per pair).
template <class F, class = void>
struct HasKernel : std::false_type {};
template <class F>
struct HasKernel<F, std::void_t<decltype(std::declval<F>().kern.kind)>> : std::true_type {};
template <class F, class Fn>
__device__ __forceinline__ void with_kernel(const F& f, Fn&& fn) {
    if constexpr (HasKernel<F>::value) {
        F fk = f;
        if (f.kern.kind == KERNEL_CUBIC_SPLINE) {
            fk.kern.kind = KERNEL_CUBIC_SPLINE;
            fn(fk);
        } else {
            fk.kern.kind = KERNEL_WENDLAND_C2;
            fn(fk);
        }
    } else {
        fn(f);
    }
}

// Candidates (in blocks of 64) staged in LDS at a time, by the bytes that one of them takes: about
// 9 KB per wavefront.  More would spare parts (a query's lanes wait for each other at the end of
// each), less leaves room for more wavefronts.  Measured at 1M points, us with 3 / 4 / 5 / 6 blocks:
// density (16 bytes) 174 / 154 / 152 / 154, pressure (20) 205 / 187 / 177 / 188, TrixiParticles
// interact! (36) 432 / 456 / 511 / 544 and 831 with 2 in Float64 (80), 898 / 947 / 1255 / 1413.
template <class TC, class TR, class F, int D>
struct RunShape {
    static constexpr bool packed = D == 3 && F::kFields > 0 && std::is_same<TC, TR>::value;
    static constexpr int bytes = (int)sizeof(Pack<TC, D>) + (F::kFields - (packed ? 1 : 0)) * (int)sizeof(TR) +
                                 (F::kIndex ? 4 : 0);
    static constexpr int fit = 9000 / (WAVE * bytes + 512);  // records and two queue rows per block
    static constexpr int NB = fit > 2 ? fit : 2;
};

// Pair functors.  A run's candidates are staged in LDS, NB blocks of 64 at a time (more: in
// interleaved parts, so that every part holds some of each query's neighbours), a lane's words
// with set bits are queued in LDS, and then every lane walks its own queue.
template <int D, class TC, class TR, class F, bool PER, int NB = RunShape<TC, TR, F, D>::NB>
__global__ __launch_bounds__(WAVE, (sizeof(TR) == 8 ? 3 : 4)) void k_runs(Geom g, SetView Q, SetView Gs, TR r2, F f, int nblocks, RunScale sc,
                                               RunSplit sp) {
    constexpr int NF = F::kFields;
    constexpr int CAP = NB * WAVE, NT = NB * 2;
    constexpr int G = sizeof(TR) == 8 ? 1 : 2;  // blocks whose loads are in flight together
    using Acc = typename F::Acc;
    using QS = typename F::QState;
    // 3D: the first field rides in the padding slot of the candidate record
    constexpr bool kPackF = D == 3 && NF > 0 && std::is_same<TC, TR>::value;
    constexpr int FOFF = kPackF ? 1 : 0, NFL = NF - FOFF;
    __shared__ Pack<TC, D> s_c[CAP];
    __shared__ TR s_f[NFL > 0 ? NFL : 1][NFL > 0 ? CAP : 1];
    __shared__ int s_j[F::kIndex ? CAP : 1];
    __shared__ unsigned s_q[NT + 2][WAVE];  // LaneQueue
    const int lane = threadIdx.x, place = block_place(lane);
    const TC* __restrict__ gc = (const TC*)Gs.coords;
    const TC* __restrict__ qcrd = (const TC*)Q.coords;
    const TR* __restrict__ fs = (const TR*)f.fsorted;
    TR box[D];
#pragma unroll
    for (int d = 0; d < D; ++d) box[d] = (TR)g.box[d];
    const TR r2_in = r2 - r2 * (TR)sc.cell_rel;  // up to this x distance squared cells are adjacent
    const int n = Q.st->n_binned, moved = Gs.st->moved;
    for_windows(n, nblocks, sp, [&](int w, int part) {
        for_runs<D>(g, Q, w, part, n, moved, sp, [&](const RunDesc& rd) {
            const RunLanes ln(rd.nq);
            const bool qact = ln.query < rd.nq;
            const int qpos = rd.q0 + (qact ? ln.query : 0);
            const int cxq = Q.keys[qpos] - rd.row;
            RunPieces<D, PER> pc;
            pc.set(g, Gs, rd);
            RunFrame<D, TC, PER> fr;
            fr.set(g, rd, sc);
            TC xq[D];
#pragma unroll
            for (int d = 0; d < D; ++d) xq[d] = qcrd[(int64_t)d * Q.cap + qpos];
            const int64_t orig = Q.sorted_idx[qpos];
            const QS qst = f.query(orig);
            const auto qr = fr.query(xq, true);
            const unsigned some = qact ? (unsigned)ln.mask : 0u;  // the lane's candidates of a tile
            const unsigned mask = 0xffff0000u | some, all = qr.sure ? 0u : some;
            Acc acc = f.init(), acc1 = f.init();  // of the first and the second pair of a step
            // part c of the np parts holds the groups c, c + np, ... of gran elements
            const int np = (pc.M + CAP - 1) / CAP;
            const int gran = np <= 8 ? 1 : 16;
            const int ngroups = (pc.M + gran - 1) / gran;
            for (int c = 0; c < np; ++c) {
                const int nel = ((ngroups - c + np - 1) / np) * gran;
                auto element = [&](int e) {  // element of the run's candidates at place e of the part
                    return np == 1 ? e : (gran == 1 ? e * np + c : ((e >> 4) * np + c) * 16 + (e & 15));
                };
                int qn = 0;  // words in this lane's queue
                typename RunPieces<D, PER>::Walk walk;
                for (int b0 = 0; b0 < nel; b0 += G * WAVE) {
                    Pack<TC, D> pk[G];
                    TR fv[G][NF > 0 ? NF : 1];
                    int jv[G];
                    bool val[G];
#pragma unroll
                    for (int gi = 0; gi < G; ++gi) {
                        const int e0 = b0 + gi * WAVE;
                        if (e0 < nel) {
                            const int mhi = min(element(min(e0 + WAVE, nel) - 1), pc.M - 1);
                            const int m = element(e0 + place);
                            val[gi] = e0 + place < nel && m < pc.M;
                            const unsigned src = (unsigned)pc.position(walk, mhi, min(m, mhi));
#pragma unroll
                            for (int d = 0; d < (D == 3 ? 4 : D); ++d) pk[gi].v[d] = (TC)0;
#pragma unroll
                            for (int d = 0; d < D; ++d) pk[gi].v[d] = load32(gc + (int64_t)d * Gs.cap, src);
                            if constexpr (NF > 0) {
#pragma unroll
                                for (int fi = 0; fi < NF; ++fi) fv[gi][fi] = load32(fs + (int64_t)fi * f.fstride, src);
                            }
                            if constexpr (F::kIndex) jv[gi] = load32(Gs.sorted_idx, src);
                        }
                    }
#pragma unroll
                    for (int gi = 0; gi < G; ++gi) {
                        const int e0 = b0 + gi * WAVE;
                        if (e0 >= nel) break;
                        TC cx[D];
#pragma unroll
                        for (int d = 0; d < D; ++d) cx[d] = pk[gi].v[d];
                        bool maybe;
                        typename RunFrame<D, TC, PER>::Operand op;
                        fr.candidate(cx, val[gi], maybe, op);
                        if constexpr (kPackF) pk[gi].v[3] = fv[gi][0];
                        if (!val[gi]) pk[gi].v[0] = (TC)INFINITY;  // for queries that look at every pair
                        s_c[e0 + place] = pk[gi];
                        if constexpr (NFL > 0) {
#pragma unroll
                            for (int fi = FOFF; fi < NF; ++fi) s_f[fi - FOFF][e0 + place] = fv[gi][fi];
                        }
                        if constexpr (F::kIndex) s_j[e0 + place] = jv[gi];
                        const TileOperands tiles(op.xy, op.zn);
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const f32x16 v = tile_products(tiles.t[t], qr);
                            const unsigned first = (unsigned)((e0 + 32 * t + (lane >> 5)) * (int)sizeof(Pack<TC, D>));
                            const unsigned word = (sign_bits(first, v) & mask) | all;
                            if (word & 0xffffu) {
                                s_q[qn][lane] = word;
                                ++qn;
                            }
                        }
                    }
                }
                s_q[qn][lane] = 0;
                s_q[qn + 1][lane] = 0;
                __syncthreads();
                with_kernel(f, [&](const F& fk) {
                    LaneQueue<Pack<TC, D>> q(s_q);
                    auto evaluate = [&](Acc& a, unsigned at, const Pack<TC, D>& pk) {
                        TR pd[D];
                        const TR d2 = run_distance<D, TC, TR, PER>(xq, pk, box, r2, pd);
                        bool in = d2 <= r2;
                        if (in && pd[0] * pd[0] > r2_in) in = run_adjacent<TC, PER>(g, rd, sp.cell64, cxq, pk.v[0]);
                        if (in) {
                            const unsigned slot = at / (unsigned)sizeof(Pack<TC, D>);
                            TR fj[NF > 0 ? NF : 1];
                            if constexpr (kPackF) fj[0] = pk.v[3];
                            if constexpr (NFL > 0) {
#pragma unroll
                                for (int fi = FOFF; fi < NF; ++fi) fj[fi] = s_f[fi - FOFF][slot];
                            }
                            int j = 0;
                            if constexpr (F::kIndex) j = s_j[slot];
                            fk.template pair<TR, D>(a, qst, pd, d2, j, fj, nullptr);
                        }
                    };
                    auto record = [&](unsigned at) { return *(const Pack<TC, D>*)((const char*)s_c + at); };
                    // two pairs per step: both records are on their way before the first is used, and each
                    // has sums of its own (shorter chains of additions, as accurate as the cell kernel's)
                    while (q.word) {
                        const unsigned a0 = q.pop();
                        const Pack<TC, D> p0 = record(a0);
                        const bool two = q.word != 0;
                        unsigned a1;
                        Pack<TC, D> p1;
                        if (two) {
                            a1 = q.pop();
                            p1 = record(a1);
                        }
                        evaluate(acc, a0, p0);
                        if (two) evaluate(acc1, a1, p1);
                    }
                });
                __syncthreads();
            }
            f.combine(acc, acc1);
            f.combine(acc, shfl_acc(acc, lane ^ 32));
            if (ln.cols <= 16) f.combine(acc, shfl_acc(acc, lane ^ 16));
            if (ln.cols <= 8) f.combine(acc, shfl_acc(acc, lane ^ 8));
            if (lane < ln.cols && qact) f.write(orig, qst, acc);
        });
    });
}

}  // namespace pn
