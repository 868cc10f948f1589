// Build kernels of the MI355X neighbourhood-search engine (gfx950, wave64):
// initialize!/update! with ParallelUpdate semantics (src/nhs_grid.jl:255-281) as a
// counting sort of the selected points by linear cell index.
//      k_bin       cell key per point + bounds check + wave-aggregated histogram
//      k_scan_*    exclusive scan of the histogram -> cell_start, non-empty cell list
//      k_scatter   point -> provisional slot in its cell segment
//      k_canon     deterministic order inside each cell (original index ascending),
//                  one thread per sorted slot, and the cell-sorted coordinate planes
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pn {

constexpr int WAVE = 64;

// Geometry of one cloud's grid inside a batch: its cells occupy the linear range
// [cell_off, cell_off + n0*n1*n2) of the concatenated cell table.
struct GeomEntry {
    int n[3];
    int cell_off;
    double minc[3];
};

// Grid geometry.  minc and cs are exact in the cell-computation type.  A batch of
// independent clouds (same radius, own boxes) sets `table`: point p belongs to cloud
// cloud_of_point[p], whose cells start at cell_offsets[cloud].
struct Geom {
    int nd;
    int n[3];      // cells per dimension, 1 for unused dimensions
    int ncells;    // total cells (all clouds)
    double minc[3];
    double cs;      // search radius
    double csd[3];  // cell size per dimension: the search radius, or box size / per with a periodic box
    int periodic;   // a PeriodicBox is set (src/nhs_grid.jl:102-125)
    int per[3];     // periodic cells per dimension
    double box[3];  // periodic box size
    const GeomEntry* table;
    const int32_t* cloud_of_point;
    const int32_t* cell_offsets;  // n_clouds + 1
    int n_clouds;
    int hash;       // SpatialHashingCellList: keys are hash buckets of unbounded cells
    int list_size;  // its number of buckets (== ncells)
    unsigned long long list_magic;  // floor((2^64 - 1) / list_size), for the bucket reduction
};

// Cloud of a linear cell index in a batch (binary search over cell_offsets).
__device__ __forceinline__ int cloud_of_cell(const Geom& g, int c) {
    int lo = 0, hi = g.n_clouds;  // cell_offsets[lo] <= c < cell_offsets[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (g.cell_offsets[mid] <= c) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Cells per dimension (x, y) of the grid holding cell c: the batch entry of its cloud, or
// gn0, gn1 (the single grid's, read once from the kernel arguments by the caller).  The
// entry is read as one 8-byte load, so the compiler cannot fold the two sources into one
// load through a private copy of the kernel arguments.
__device__ __forceinline__ void grid_dims_xy(const Geom& g, int c, int gn0, int gn1, int& n0, int& n1) {
    if (g.table) {
        const int2 e = *(const int2*)&g.table[cloud_of_cell(g, c)].n[0];
        n0 = e.x;
        n1 = e.y;
    } else {
        n0 = gn0;
        n1 = gn1;
    }
}

// Device-side status of one binning pass.
struct DevStatus {
    unsigned long long first_bad;  // smallest selection position out of bounds
    unsigned long long total64;    // sum of all counts, 64-bit (overflow guard)
    int max_count;                 // largest cell population
    int n_nonempty;                // number of non-empty cells
    int n_binned;                  // number of binned points (low 32 bits of the sum)
    int n_ordered;                 // work items appended by k_order_work; k_list_counts
    // k_bin's minimum, moved to first_bad and set back to ~0 by the scan, so that the next binning
    // finds it ready without a launch of its own
    unsigned long long bad_now;
    int moved;  // the coordinate planes were gathered again since (k_regather)
    int n_octets;  // aligned groups of eight cells (in x, but for the ends of rows) that hold points; 0: not counted
};

// Host copy of a binning's status in pinned, coherent host memory.  The scan (or k_build_small),
// the last of a binning to change the fields the host checks, stores the status there and
// then raises `seq` with a system-scope release, so the host can raise the binning's
// errors while the scatter and the in-cell ordering still run.
struct StatusMailbox {
    DevStatus status;
    unsigned long long seq;
};

// Read-only view of a binned point set used by the traversal.
struct SetView {
    const int32_t* start;       // C + 1 cell offsets
    const int32_t* nonempty;    // non-empty cell ids
    const int32_t* sorted_idx;  // original index per sorted position
    const int32_t* keys;        // cell per sorted position (NULL for a SpatialHashingCellList)
    const void* coords;         // D planes of cap entries, cell-sorted
    int64_t cap;
    const DevStatus* st;
    // SpatialHashingCellList only (else NULL), as of the last binning: per non-empty bucket the
    // cell of one of its points (3 int32), and bucket_mixed[b] == bucket_epoch when its points
    // lie in more than one cell (entries of earlier binnings hold earlier epochs)
    const int32_t* bucket_cell;
    const int32_t* bucket_mixed;
    int bucket_epoch;
};

// Workgroups are dispatched round-robin over the 8 XCDs.  Remap so that each XCD
// works on a contiguous range of cells: neighbouring cells share stencil rows, which
// then hit the same L2.  The launch size must be a multiple of 8.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
    const int per = nblocks >> 3;
    return (bid & 7) * per + (bid >> 3);
}

// ------------------------------------------------------------------------------------
// Build kernels
// ------------------------------------------------------------------------------------

static __global__ void k_reset_status(DevStatus* st) {
    st->first_bad = ~0ull;
    st->total64 = 0ull;
    st->max_count = 0;
    st->n_nonempty = 0;
    st->n_binned = 0;
    st->n_ordered = 0;
    st->bad_now = ~0ull;
    st->moved = 0;
    st->n_octets = 0;
}

static __global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

// floor_to_int (src/util.jl:19-34) of an already floored value: NaN and values >= 2^63
// saturate to typemax(Int64), values <= -2^63 to typemin(Int64).
template <class T>
__device__ __forceinline__ int64_t floor_to_int64(T f) {
    if (!(f < (T)9223372036854775808.0)) return INT64_MAX;  // NaN too
    if (f <= (T)-9223372036854775808.0) return INT64_MIN;
    return (int64_t)f;
}

// Cell key of point p: (x - min) / cs in TCELL, floor, 1-based cell must lie in
// 2:(n_d - 1) (src/cell_lists/full_grid.jl:84-94, :187-213).  With f = floor(q) the
// condition reads 1 <= f <= n_d - 2; NaN and +-Inf fail both comparisons, matching the
// saturating floor_to_int (src/util.jl:19-34) whose saturated values are out of range.
// With a periodic box the 1-based cell floor_to_int(q) + 1 is wrapped to
// mod(cell - 2, per) + 2 in Int64 arithmetic (src/nhs_grid.jl:609-628), so every
// coordinate, NaN included, lands in 2:per+1; that must still lie in 2:(n_d - 1).
template <int D, class TC, class TCELL>
__device__ __forceinline__ int cell_key(const int (&n)[3], const double (&minc)[3], const double (&cs)[3],
                                        const Geom& g, const TC* __restrict__ xp, bool& ok) {
    int key = 0, stride = 1;
    ok = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        TCELL q = ((TCELL)xp[d] - (TCELL)minc[d]) / (TCELL)cs[d];
        TCELL f = floor(q);
        int c0;
        bool in;
        if (!g.periodic) {
            in = (f >= (TCELL)1) && (f <= (TCELL)(n[d] - 2));
            c0 = in ? (int)f : 0;
        } else {
            // (floor_to_int(q) + 1) - 2 with Int64 wrap, floored mod per
            const int64_t a = (int64_t)((uint64_t)floor_to_int64(f) - 1ull);
            int64_t r = a % (int64_t)g.per[d];
            if (r < 0) r += g.per[d];
            c0 = (int)r + 1;  // 0-based index of the 1-based cell r + 2
            in = c0 <= n[d] - 2;
            c0 = in ? c0 : 0;
        }
        ok = ok && in;
        key += c0 * stride;
        stride *= n[d];
    }
    return key;
}

// mod(c - 2, n) + 2 in wrapping Int64 arithmetic (periodic_cell_index, src/nhs_grid.jl:609-620).
__device__ __forceinline__ int64_t hash_wrap(int64_t c, int n) {
    int64_t m = (int64_t)((uint64_t)c - 2ull) % (int64_t)n;
    if (m < 0) m += n;
    return m + 2;
}

// Cell of a point under a SpatialHashingCellList: floor_to_int.(x ./ cell_size), no corner
// and no +1 (nonperiodic_cell_coords, src/nhs_grid.jl:636-638).  ok is false when a cell
// coordinate does not fit in Int32 (NaN and infinities included): the reference's
// coordinates_flattened (src/cell_lists/spatial_hashing.jl:170-183) throws InexactError there.
// With a PeriodicBox the cell is wrapped, mod.(c .- 2, n_periodic) .+ 2 (periodic_cell_index,
// src/nhs_grid.jl:609-620), which always fits: no error then, as in the reference.
template <int D, class TC, class TCELL, bool PER>
__device__ __forceinline__ void hash_cell_p(const Geom& g, const TC* __restrict__ xp, int64_t (&c)[3], bool& ok) {
    ok = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) c[d] = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const TCELL q = (TCELL)xp[d] / (TCELL)g.csd[d];
        const TCELL f = floor(q);
        if constexpr (PER) {
            c[d] = hash_wrap(floor_to_int64(f), g.per[d]);
        } else {
            ok = ok && (f >= (TCELL)-2147483648.0) && (f <= (TCELL)2147483647.0);
            c[d] = ok ? (int64_t)f : 0;
        }
    }
}

template <int D, class TC, class TCELL>
__device__ __forceinline__ void hash_cell(const Geom& g, const TC* __restrict__ xp, int64_t (&c)[3], bool& ok) {
    if (g.periodic) hash_cell_p<D, TC, TCELL, true>(g, xp, c, ok);
    else hash_cell_p<D, TC, TCELL, false>(g, xp, c, ok);
}

// spatial_hash (src/cell_lists/spatial_hashing.jl:150-164, Ihmsen et al. 2011) in Julia's
// wrapping Int64 arithmetic, 0-based: mod(xor(i * 73856093, j * 19349663, k * 83492791), L),
// the floored mod of the signed hash.  For a negative hash h, mod(h, L) = L - 1 - (~h mod L)
// (~h = -h - 1 >= 0).  x mod L for x < 2^63 is a Barrett reduction with
// magic = floor((2^64 - 1) / L): q = mulhi(x, magic) > x / L - 3/2, so r = x - q L lies in
// [0, 3L/2) and one conditional subtraction ends it (a 64-bit division is a long software
// routine here).
template <int D>
__device__ __forceinline__ int spatial_hash(const int64_t (&c)[3], const Geom& g) {
    uint64_t h = (uint64_t)c[0] * 73856093ull;
    if (D >= 2) h ^= (uint64_t)c[1] * 19349663ull;
    if (D >= 3) h ^= (uint64_t)c[2] * 83492791ull;
    const uint64_t L = (uint64_t)g.list_size;
    const bool neg = (int64_t)h < 0;
    const uint64_t x = neg ? ~h : h;
    uint64_t r = x - __umul64hi(x, g.list_magic) * L;
    r = r >= L ? r - L : r;
    return (int)(neg ? L - 1 - r : r);
}

__device__ __forceinline__ int64_t sel_point(int64_t a, int64_t sel_first, const int32_t* sel_list) {
    return sel_list ? (int64_t)sel_list[a] : sel_first + a;
}

// 0-based cell of point p (ok: it lies in the grid).
template <int D, class TC, class TCELL>
__device__ __forceinline__ int point_key(const Geom& g, const TC* __restrict__ y, int64_t p, bool& ok) {
    if (g.hash) {
        int64_t c[3];
        hash_cell<D, TC, TCELL>(g, y + (int64_t)D * p, c, ok);
        return spatial_hash<D>(c, g);
    }
    if (g.table) {
        const GeomEntry e = g.table[g.cloud_of_point[p]];
        return e.cell_off + cell_key<D, TC, TCELL>(e.n, e.minc, g.csd, g, y + (int64_t)D * p, ok);
    }
    return cell_key<D, TC, TCELL>(g.n, g.minc, g.csd, g, y + (int64_t)D * p, ok);
}

// One thread per selected point.  Lanes of a wavefront whose keys form a run (common:
// inputs are usually close to cell order) share one atomic on the histogram; the slot
// of each point inside its cell segment is the atomic's old value plus its run offset.
template <int D, class TC, class TCELL>
__global__ __launch_bounds__(256) void k_bin(Geom g, const TC* __restrict__ y, int64_t sel_first,
                                             const int32_t* __restrict__ sel_list, int64_t n_sel,
                                             int32_t* __restrict__ keys, int32_t* __restrict__ slots,
                                             int32_t* __restrict__ counts, DevStatus* st) {
    const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & (WAVE - 1);
    int key = -1;
    if (a < n_sel) {
        int64_t p = sel_point(a, sel_first, sel_list);
        bool ok;
        const int k = point_key<D, TC, TCELL>(g, y, p, ok);
        if (ok) key = k;
        else atomicMin(&st->bad_now, (unsigned long long)a);
        keys[a] = key;
    }
    const int prev = __shfl_up(key, 1, WAVE);
    const bool head = (lane == 0) || (key != prev);
    const unsigned long long hm = __ballot(head);
    const unsigned long long above = lane == 63 ? 0ull : (hm >> (lane + 1)) << (lane + 1);
    const int next = above ? __ffsll((long long)above) - 1 : WAVE;
    int base = 0;
    if (head && key >= 0) base = atomicAdd(&counts[key], next - lane);
    const unsigned long long upto = hm & ((2ull << lane) - 1ull);
    const int hl = 63 - __clzll((long long)upto);
    base = __shfl(base, hl, WAVE);
    if (a < n_sel && key >= 0) slots[a] = base + (lane - hl);
}

// Scan of a histogram of C int32 counts, 2048 items per block (256 threads x 8).
// Packed 64-bit value per cell: low word = count, high word = (count > 0); the high
// word's prefix is the position in the non-empty cell list.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ unsigned long long pack_cell(int32_t c) {
    return (unsigned long long)(uint32_t)c | ((unsigned long long)(c > 0) << 32);
}

__device__ __forceinline__ unsigned long long wave_incl_scan(unsigned long long v, int lane) {
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        unsigned long long t = __shfl_up(v, o, WAVE);
        if (lane >= o) v += t;
    }
    return v;
}

// Block-wide exclusive scan of one value per thread (sh: one entry per wave).
__device__ __forceinline__ unsigned long long block_excl_scan(unsigned long long v, unsigned long long* sh,
                                                              unsigned long long& total) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x >> 6;
    unsigned long long inc = wave_incl_scan(v, lane);
    if (lane == WAVE - 1) sh[w] = inc;
    __syncthreads();
    unsigned long long off = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < SCAN_THREADS / WAVE; ++i) {
        unsigned long long s = sh[i];
        if (i < w) off += s;
        total += s;
    }
    __syncthreads();
    return off + inc - v;
}

static __global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const int32_t* __restrict__ counts, int64_t C,
                                                              unsigned long long* __restrict__ block_sums,
                                                              DevStatus* st) {
    __shared__ unsigned long long sh[SCAN_THREADS / WAVE];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned long long s = 0;
    int mx = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        int64_t c = base + i;
        int32_t v = c < C ? counts[c] : 0;
        s += pack_cell(v);
        mx = max(mx, v);
    }
    unsigned long long total;
    block_excl_scan(s, sh, total);
    static_assert(SCAN_ITEMS == 8, "a thread's cells are an octet");
    const int octets = __popcll(__ballot(s != 0));
    // block max of the populations; block sums and maxima go to k_scan_top (no same-address
    // atomics: with millions of cells or buckets they serialised the pass)
    __shared__ int shm[SCAN_THREADS / WAVE], sho[SCAN_THREADS / WAVE];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, WAVE));
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        shm[threadIdx.x >> 6] = mx;
        sho[threadIdx.x >> 6] = octets;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int m = shm[0], oct = sho[0];
#pragma unroll
        for (int i = 1; i < SCAN_THREADS / WAVE; ++i) {
            m = max(m, shm[i]);
            oct += sho[i];
        }
        block_sums[blockIdx.x] = total;
        block_sums[gridDim.x + blockIdx.x] = (unsigned long long)(uint32_t)m | (unsigned long long)oct << 32;
    }
}

// The status of a binning whose packed counts sum to `sum`; in pinned host memory too when mb.
__device__ __forceinline__ void publish_status(DevStatus* st, StatusMailbox* mb, unsigned long long seq,
                                               unsigned long long bad, unsigned long long total64, int max_count,
                                               unsigned long long sum, int n_octets = 0) {
    DevStatus s;
    s.first_bad = bad;
    s.total64 = total64;
    s.max_count = max_count;
    s.n_nonempty = (int)(uint32_t)(sum >> 32);
    s.n_binned = (int)(uint32_t)(sum & 0xffffffffull);
    s.n_ordered = 0;
    s.bad_now = ~0ull;
    s.moved = 0;
    s.n_octets = n_octets;
    *st = s;
    if (mb) {
        mb->status = s;
        __hip_atomic_store(&mb->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Single workgroup: exclusive scan of the block sums (block_sums[0, nblocks)), writes the
// totals, the 64-bit sum of all counts, the largest count and the number of octets (block maxima and
// octets at block_sums[nblocks, 2 nblocks)).
static __global__ __launch_bounds__(SCAN_THREADS) void k_scan_top(unsigned long long* __restrict__ block_sums,
                                                           int64_t nblocks, int32_t* __restrict__ start,
                                                           int64_t C, DevStatus* st, StatusMailbox* mb,
                                                           unsigned long long seq) {
    __shared__ unsigned long long sh[SCAN_THREADS / WAVE];
    __shared__ unsigned long long sh_sum[SCAN_THREADS / WAVE];
    __shared__ int sh_max[SCAN_THREADS / WAVE], sh_oct[SCAN_THREADS / WAVE];
    unsigned long long carry = 0, sum64 = 0;
    int mx = 0, oct = 0;
    for (int64_t b0 = 0; b0 < nblocks; b0 += SCAN_THREADS) {
        int64_t b = b0 + threadIdx.x;
        unsigned long long v = b < nblocks ? block_sums[b] : 0ull;
        if (b < nblocks) {
            sum64 += v & 0xffffffffull;
            const unsigned long long mo = block_sums[nblocks + b];
            mx = max(mx, (int)(uint32_t)mo);
            oct += (int)(uint32_t)(mo >> 32);
        }
        unsigned long long total;
        unsigned long long ex = block_excl_scan(v, sh, total);
        if (b < nblocks) block_sums[b] = carry + ex;
        carry += total;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum64 += __shfl_xor(sum64, o, WAVE);
        mx = max(mx, __shfl_xor(mx, o, WAVE));
        oct += __shfl_xor(oct, o, WAVE);
    }
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        sh_sum[threadIdx.x >> 6] = sum64;
        sh_max[threadIdx.x >> 6] = mx;
        sh_oct[threadIdx.x >> 6] = oct;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        int m = 0, n_octets = 0;
#pragma unroll
        for (int i = 0; i < SCAN_THREADS / WAVE; ++i) {
            tot += sh_sum[i];
            m = max(m, sh_max[i]);
            n_octets += sh_oct[i];
        }
        start[C] = (int32_t)(uint32_t)(carry & 0xffffffffull);
        publish_status(st, mb, seq, st->bad_now, tot, m, carry, n_octets);  // bad_now: of k_bin, an earlier kernel
    }
}

static __global__ __launch_bounds__(SCAN_THREADS) void k_scan_down(const int32_t* counts, int64_t C,
                                                            const unsigned long long* __restrict__ block_sums,
                                                            int32_t* __restrict__ start,
                                                            int32_t* __restrict__ nonempty,
                                                            int32_t* clear) {
    __shared__ unsigned long long sh[SCAN_THREADS / WAVE];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int32_t v[SCAN_ITEMS];
    unsigned long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        int64_t c = base + i;
        v[i] = c < C ? counts[c] : 0;
        s += pack_cell(v[i]);
    }
    // clear = counts: the counts are read once, here, and left zero for the next binning
    if (clear) {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            if (base + i < C) clear[base + i] = 0;
    }
    unsigned long long total;
    unsigned long long run = block_sums[blockIdx.x] + block_excl_scan(s, sh, total);
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        int64_t c = base + i;
        if (c < C) {
            start[c] = (int32_t)(uint32_t)(run & 0xffffffffull);
            if (nonempty && v[i] > 0) nonempty[(uint32_t)(run >> 32)] = (int32_t)c;
        }
        run += pack_cell(v[i]);
    }
}

// Provisional placement: selection position a goes to slot start[key] + slots[a] of its
// cell segment (atomic order).  The slot holds a, not the point index, so k_canon can
// recover the key and break ties between repeated selections.  With reset = slots, each
// entry is set to -1 once read (the hash build reuses the array, cleared, for its bucket
// representatives).
static __global__ __launch_bounds__(256) void k_scatter(const int32_t* __restrict__ keys, const int32_t* slots,
                                                 int64_t n_sel, const int32_t* __restrict__ start,
                                                 int32_t* __restrict__ perm_tmp, int32_t* reset) {
    const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= n_sel) return;
    const int key = keys[a];
    const int slot = key < 0 ? 0 : slots[a];
    if (reset) reset[a] = -1;
    if (key < 0) return;
    perm_tmp[start[key] + slot] = (int32_t)a;
}

// Cells with more points than this keep the provisional (atomic) order instead of the
// O(n^2) rank: their neighbour sets are unaffected, only the order inside the cell.
constexpr int CANON_RANK_LIMIT = 1024;

// Output-major: one thread per sorted slot k of the binned points.  The final position of
// the point in slot k is its cell's start plus its rank in the cell segment by (original
// index, selection position) ascending (canonical = 1: the SerialUpdate insertion order,
// and repeated selections of one point get distinct consecutive slots), or k itself
// (canonical = 0: the order of the reference's ParallelUpdate, nondeterministic inside a
// cell; neighbour sets are the same).  A wavefront's stores land inside the cell segments
// of its 64 slots, so the permutation, the cell per sorted position and the cell-sorted
// coordinate planes (plane d at coords + d * cap) are written in whole lines.
// Slot k's canonical position pos, its selection position a, point p, cell key and the first
// slot s of the cell segment.
struct CanonSlot {
    int pos, key, s;
    int32_t a, p;
};
__device__ __forceinline__ CanonSlot canon_slot(const int32_t* __restrict__ keys, int64_t sel_first,
                                                const int32_t* __restrict__ sel_list,
                                                const int32_t* __restrict__ start,
                                                const int32_t* __restrict__ perm_tmp, int64_t k, int canonical) {
    CanonSlot c;
    c.a = perm_tmp[k];
    c.key = keys[c.a];
    c.p = (int32_t)sel_point(c.a, sel_first, sel_list);
    c.s = start[c.key];
    const int e = start[c.key + 1];
    c.pos = (int)k;
    if (canonical && e - c.s <= CANON_RANK_LIMIT) {
        int rank = 0;
        if (!sel_list) {
            // original index = sel_first + selection position: rank by position
            for (int q = c.s; q < e; ++q) rank += perm_tmp[q] < c.a;
        } else {
            for (int q = c.s; q < e; ++q) {
                const int32_t aq = perm_tmp[q];
                const int32_t pq = sel_list[aq];
                rank += (pq < c.p) || (pq == c.p && aq < c.a);
            }
        }
        c.pos = c.s + rank;
    }
    return c;
}

template <int D, class TC>
__global__ __launch_bounds__(256) void k_canon(const int32_t* __restrict__ keys, int64_t sel_first,
                                               const int32_t* __restrict__ sel_list, const DevStatus* st,
                                               const int32_t* __restrict__ start,
                                               const int32_t* __restrict__ perm_tmp,
                                               const TC* __restrict__ y, int32_t* __restrict__ sorted_idx,
                                               TC* __restrict__ coords, int64_t cap, int canonical,
                                               int32_t* __restrict__ sorted_keys) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= st->n_binned) return;
    const CanonSlot c = canon_slot(keys, sel_first, sel_list, start, perm_tmp, k, canonical);
    sorted_idx[c.pos] = c.p;
    sorted_keys[c.pos] = c.key;
#pragma unroll
    for (int d = 0; d < D; ++d) coords[(int64_t)d * cap + c.pos] = y[(int64_t)D * c.p + d];
}

// The whole scan of up to SCAN_ONE_MAX counts, which it leaves zero, in one workgroup: what
// k_scan_reduce, k_scan_top and k_scan_down do in three launches of 3 to 6 us, most of it the launch
// (1900 cells 10 us and two gaps, here 5; 15,000 cells 12 us, here 7; the time grows by the 64 rows
// of cells that a wavefront takes, so the chip's three passes win beyond).
constexpr int BUILD_THREADS = 1024;
constexpr int SCAN_ONE_ITEMS = 16;
constexpr int SCAN_ONE_MAX = BUILD_THREADS * SCAN_ONE_ITEMS;

// Inclusive sums over the wavefront's lanes (DPP row shifts and broadcasts).
__device__ __forceinline__ int wave_incl_scan_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// Exclusive sums of a workgroup's C counts, count(c), into put(c, first, rank among the non-empty,
// count); returns the packed sum and sets the largest count.  A wavefront takes consecutive rows of
// 64 cells, so that its loads and stores are whole lines.
template <class Count, class Put>
__device__ __forceinline__ unsigned long long scan_one(int C, unsigned long long* sh, int* sh_max, int& max_count,
                                                       Count&& count, Put&& put) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x >> 6;
    const int rows = (C + BUILD_THREADS - 1) / BUILD_THREADS;  // of each wavefront, at most SCAN_ONE_ITEMS
    const int c0 = w * rows * WAVE + lane;
    int v[SCAN_ONE_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; ++i) v[i] = i < rows && c0 + i * WAVE < C ? count(c0 + i * WAVE) : 0;
    unsigned long long s = 0;
    int mx = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; ++i) {
        s += pack_cell(v[i]);
        mx = max(mx, v[i]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, WAVE);
        mx = max(mx, __shfl_xor(mx, o, WAVE));
    }
    if (lane == 0) {
        sh[w] = s;
        sh_max[w] = mx;
    }
    __syncthreads();
    unsigned long long before = 0, total = 0;
    max_count = 0;
#pragma unroll
    for (int i = 0; i < BUILD_THREADS / WAVE; ++i) {
        before += i < w ? sh[i] : 0ull;
        total += sh[i];
        max_count = max(max_count, sh_max[i]);
    }
    int first = (int)(uint32_t)(before & 0xffffffffull), rank = (int)(uint32_t)(before >> 32);
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; ++i) {
        if (i >= rows) break;
        const int incl = wave_incl_scan_dpp(v[i]);
        const unsigned long long some = __ballot(v[i] > 0);
        const int r = rank + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(some >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)some, 0));
        if (c0 + i * WAVE < C) put(c0 + i * WAVE, first + incl - v[i], r, v[i]);
        first += __builtin_amdgcn_readlane(incl, WAVE - 1);
        rank += __popcll(some);
    }
    return total;
}

static __global__ __launch_bounds__(BUILD_THREADS) void k_scan_one(int32_t* __restrict__ counts, int C,
                                                            int32_t* __restrict__ start,
                                                            int32_t* __restrict__ nonempty, DevStatus* st,
                                                            StatusMailbox* mb, unsigned long long seq) {
    __shared__ unsigned long long sh[BUILD_THREADS / WAVE];
    __shared__ int sh_max[BUILD_THREADS / WAVE];
    int max_count;
    const unsigned long long sum = scan_one(
        C, sh, sh_max, max_count, [&](int c) { return counts[c]; },
        [&](int c, int first, int rank, int n) {
            start[c] = first;
            counts[c] = 0;
            if (n > 0) nonempty[rank] = c;
        });
    if (threadIdx.x == 0) {
        start[C] = (int32_t)(uint32_t)(sum & 0xffffffffull);
        publish_status(st, mb, seq, st->bad_now, sum & 0xffffffffull, max_count, sum);
    }
}

// A whole binning (k_bin, the scan, k_scatter and k_canon, in that order below) of up to
// BUILD_SMALL_POINTS points in up to BUILD_SMALL_CELLS cells in one workgroup, the histogram and the
// provisional placement in LDS: the launches cost more than their work there.  2000 points in 2D:
// 24 us in seven kernels and the gaps between them become 9 us; 3375 points in 3D 14.5 us.  One
// compute unit's loads and stores bound it: of 15,600 points the four kernels take 19 us.
constexpr int BUILD_ITEMS = 4;
constexpr int BUILD_SMALL_POINTS = BUILD_THREADS * BUILD_ITEMS;
constexpr int BUILD_SMALL_CELLS = 11 * 1024;  // 64 KB of LDS
// Ranking every point among those of its cell takes a compute unit too long where cells are crowded.
// From a fullest cell of this many points on, the selection is placed in its order, 64 points at a
// time (4096 points, 30 / 250 / 1000 a cell: ranked 22 / 86 / 291 us, placed in order 22 us from 64 on,
// 23 / 19; the kernels of larger clouds 23 / 46 / 109).
constexpr int BUILD_CROWDED = 64;

template <int D, class TC, class TCELL>
__global__ __launch_bounds__(BUILD_THREADS) void k_build_small(Geom g, const TC* __restrict__ y, int64_t sel_first,
                                                               const int32_t* __restrict__ sel_list, int n_sel,
                                                               int32_t* __restrict__ start,
                                                               int32_t* __restrict__ nonempty,
                                                               int32_t* __restrict__ sorted_idx,
                                                               int32_t* __restrict__ sorted_keys,
                                                               TC* __restrict__ coords, int64_t cap, int canonical,
                                                               DevStatus* st, StatusMailbox* mb,
                                                               unsigned long long seq) {
    __shared__ int s_cell[BUILD_SMALL_CELLS + 1];  // counts, then starts
    __shared__ int s_perm[BUILD_SMALL_POINTS];
    __shared__ unsigned long long sh[BUILD_THREADS / WAVE];
    __shared__ int sh_max[BUILD_THREADS / WAVE];
    __shared__ int s_bad;
    __shared__ int s_descends;  // the selection is not in the order of the points
    const int C = g.ncells;
    for (int c = threadIdx.x; c < C; c += BUILD_THREADS) s_cell[c] = 0;
    if (threadIdx.x == 0) {
        s_bad = INT32_MAX;
        s_descends = 0;
    }
    __syncthreads();
    int key[BUILD_ITEMS], slot[BUILD_ITEMS];
    int32_t p[BUILD_ITEMS];
#pragma unroll
    for (int i = 0; i < BUILD_ITEMS; ++i) {
        const int a = (int)threadIdx.x + i * BUILD_THREADS;
        key[i] = -1;
        if (a < n_sel) {
            p[i] = (int32_t)sel_point(a, sel_first, sel_list);
            if (sel_list && a > 0 && sel_list[a - 1] > p[i]) s_descends = 1;
            bool ok;
            const int k = point_key<D, TC, TCELL>(g, y, p[i], ok);
            if (ok) {
                key[i] = k;
                slot[i] = atomicAdd(&s_cell[k], 1);
            } else {
                atomicMin(&s_bad, a);
            }
        }
    }
    __syncthreads();
    int max_count;
    const unsigned long long sum = scan_one(
        C, sh, sh_max, max_count, [&](int c) { return s_cell[c]; },
        [&](int c, int first, int rank, int n) {
            s_cell[c] = first;
            start[c] = first;
            if (n > 0) nonempty[rank] = c;
        });
    if (threadIdx.x == 0) {
        s_cell[C] = start[C] = (int32_t)(uint32_t)(sum & 0xffffffffull);
        publish_status(st, mb, seq, s_bad == INT32_MAX ? ~0ull : (unsigned long long)s_bad, sum & 0xffffffffull,
                       max_count, sum);
    }
    __syncthreads();
    auto place = [&](int i, int pos) {
        sorted_idx[pos] = p[i];
        sorted_keys[pos] = key[i];
#pragma unroll
        for (int d = 0; d < D; ++d) coords[(int64_t)d * cap + pos] = y[(int64_t)D * p[i] + d];
    };
    if (canonical && max_count >= BUILD_CROWDED && !s_descends) {  // the same for the whole workgroup
#pragma unroll
        for (int i = 0; i < BUILD_ITEMS; ++i) {
            // among the wavefront's points: those of its cell, and those of them before it
            int before = 0, n_same = 0;
            for (unsigned long long left = __ballot(key[i] >= 0); left;) {
                const int k = __builtin_amdgcn_readlane(key[i], __builtin_ctzll(left));
                const unsigned long long same = __ballot(key[i] == k);
                if (key[i] == k) {
                    before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)same, 0));
                    n_same = __popcll(same);
                }
                left &= ~same;
            }
            // the wavefronts in turn: s_cell[c] is the next free slot of cell c
            for (int t = 0; t < BUILD_THREADS / WAVE; ++t) {
                if (i * BUILD_THREADS + t * WAVE >= n_sel) break;
                if ((int)threadIdx.x / WAVE == t && key[i] >= 0) {
                    const int next = s_cell[key[i]];
                    if (before == 0) s_cell[key[i]] = next + n_same;
                    place(i, next + before);
                }
                __syncthreads();
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < BUILD_ITEMS; ++i)
            if (key[i] >= 0) s_perm[s_cell[key[i]] + slot[i]] = (int)threadIdx.x + i * BUILD_THREADS;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < BUILD_ITEMS; ++i) {
            if (key[i] < 0) continue;
            const int a = (int)threadIdx.x + i * BUILD_THREADS, b = s_cell[key[i]], e = s_cell[key[i] + 1];
            int pos = b + slot[i];
            if (canonical && e - b <= CANON_RANK_LIMIT) {
                pos = b;
                for (int q = b; q < e; ++q) {
                    const int aq = s_perm[q];
                    if (!sel_list) {
                        pos += aq < a;
                    } else {
                        const int32_t pq = sel_list[aq];
                        pos += (pq < p[i]) || (pq == p[i] && aq < a);
                    }
                }
            }
            place(i, pos);
        }
    }
}

// k_canon for a SpatialHashingCellList, which also records the bucket data the cell kernel
// needs (the reference's collision flags, src/cell_lists/spatial_hashing.jl:84-116, computed
// once per binning instead of per push): the point in the segment's first provisional slot s
// gives the bucket's cell (written by slot s itself), and a point whose cell differs from it
// marks the bucket as mixed (bucket_mixed[key] = epoch; every writer stores the same value).
// Slot s also names its selection position a as the bucket's representative: rep[a] = key
// (rep holds -1 elsewhere).
template <int D, class TC, class TCELL>
__global__ __launch_bounds__(256) void k_canon_hash(const int32_t* __restrict__ keys, int64_t sel_first,
                                                    const int32_t* __restrict__ sel_list, const DevStatus* st,
                                                    const int32_t* __restrict__ start,
                                                    const int32_t* __restrict__ perm_tmp,
                                                    const TC* __restrict__ y, int32_t* __restrict__ sorted_idx,
                                                    TC* __restrict__ coords, int64_t cap, int canonical, Geom g,
                                                    int32_t* __restrict__ bucket_cell,
                                                    int32_t* __restrict__ bucket_mixed, int epoch,
                                                    int32_t* __restrict__ rep) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= st->n_binned) return;
    const CanonSlot c = canon_slot(keys, sel_first, sel_list, start, perm_tmp, k, canonical);
    TC x[D], xs[D];
    const int64_t ps = sel_point(perm_tmp[c.s], sel_first, sel_list);
#pragma unroll
    for (int d = 0; d < D; ++d) {
        x[d] = y[(int64_t)D * c.p + d];
        xs[d] = y[(int64_t)D * ps + d];
    }
    sorted_idx[c.pos] = c.p;
#pragma unroll
    for (int d = 0; d < D; ++d) coords[(int64_t)d * cap + c.pos] = x[d];
    int64_t ck[3], cs[3];
    bool ok;
    hash_cell<D, TC, TCELL>(g, x, ck, ok);
    hash_cell<D, TC, TCELL>(g, xs, cs, ok);
    if (k == c.s) {
#pragma unroll
        for (int d = 0; d < 3; ++d) bucket_cell[3 * (int64_t)c.key + d] = (int32_t)cs[d];
        rep[c.a] = c.key;  // the bucket's representative selection position (for k_order_work)
    }
    bool same = true;
#pragma unroll
    for (int d = 0; d < D; ++d) same = same && ck[d] == cs[d];
    if (!same) bucket_mixed[c.key] = epoch;
}

// SpatialHashingCellList work order: overwrites the non-empty bucket list with the buckets in
// the order of their representatives' selection positions (rep[a] >= 0, from k_canon_hash),
// roughly: a workgroup compacts ORDER_ITEMS positions per thread in order and appends them with
// one atomic, so the order across workgroups is their completion order.  Buckets sit at hash
// positions, so bucket order scatters spatially adjacent work items over the XCDs; the
// selection order follows the input's order, which is spatially coherent in every benchmark
// (cell-sorted clouds), and keeps a neighbourhood's buckets in one XCD's L2.  Every work item
// writes only its own queries' results, so results do not depend on the order.
constexpr int ORDER_THREADS = 1024, ORDER_ITEMS = 4;
static __global__ __launch_bounds__(ORDER_THREADS) void k_order_work(const int32_t* __restrict__ rep, int64_t n_sel,
                                                                      DevStatus* st,
                                                                      int32_t* __restrict__ nonempty) {
    __shared__ int s_wave[ORDER_THREADS / WAVE];
    __shared__ int s_base;
    const int64_t a0 = ((int64_t)blockIdx.x * ORDER_THREADS + threadIdx.x) * ORDER_ITEMS;
    int key[ORDER_ITEMS];
    int n = 0;
#pragma unroll
    for (int i = 0; i < ORDER_ITEMS; ++i) {
        const int64_t a = a0 + i;
        key[i] = a < n_sel ? rep[a] : -1;
        n += key[i] >= 0;
    }
    // exclusive scan of n over the workgroup
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    int inc = n;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const int t = __shfl_up(inc, o, WAVE);
        if (lane >= o) inc += t;
    }
    if (lane == WAVE - 1) s_wave[wv] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < ORDER_THREADS / WAVE; ++w) {
            const int v = s_wave[w];
            s_wave[w] = tot;
            tot += v;
        }
        s_base = tot > 0 ? atomicAdd(&st->n_ordered, tot) : 0;
    }
    __syncthreads();
    int pos = s_base + s_wave[wv] + inc - n;
#pragma unroll
    for (int i = 0; i < ORDER_ITEMS; ++i)
        if (key[i] >= 0) nonempty[pos++] = key[i];
}

// Re-gathers the sorted coordinate planes from y (update-free coordinate refresh).
template <int D, class TC>
__global__ __launch_bounds__(256) void k_regather(const int32_t* __restrict__ sorted_idx, DevStatus* st,
                                                  const TC* __restrict__ y, TC* __restrict__ coords,
                                                  int64_t cap) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) st->moved = 1;
    if (k >= st->n_binned) return;
    const int64_t p = sorted_idx[k];
#pragma unroll
    for (int d = 0; d < D; ++d) coords[(int64_t)d * cap + k] = y[(int64_t)D * p + d];
}

// Synthetic per-step displacement U[-a, a] of every coordinate, a pure function of
// (seed, step, index): SplitMix64 of a counter, top 53 bits.  The step counter lives on
// the device so a captured graph advances it on every replay (the perturbation of
// benchmarks/update.jl:28-49, made replayable).
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

template <class T>
__global__ __launch_bounds__(256) void k_displace(T* __restrict__ x, int64_t n, T a, unsigned long long seed,
                                                  const int64_t* __restrict__ step) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned long long key = splitmix64(seed ^ splitmix64((unsigned long long)*step));
    const double u = (double)(splitmix64(key + (unsigned long long)i) >> 11) * (1.0 / 9007199254740992.0);
    x[i] += (T)((2.0 * u - 1.0) * (double)a);
}

static __global__ void k_step_increment(int64_t* step) { *step += 1; }

}  // namespace pn
