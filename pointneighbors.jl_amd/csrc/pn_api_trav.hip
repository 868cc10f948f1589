// C-ABI traversal entry points: neighbour counts, index sums and CSR neighbour lists.
#include "pn_host.h"
#include "pn_fill.h"
extern "C" {

int pn_count_neighbors(pn_grid_t grid, int queries, int32_t* counts, int accumulate) {
    if (!grid) return fail(PN_ERR_ARGUMENT, "grid is NULL");
    if (!counts) return fail(PN_ERR_ARGUMENT, "counts is NULL");
    pn::CountF f;
    f.out = counts;
    f.accumulate = accumulate;
    return launch_traverse(*grid, queries, f);
}

int pn_sum_neighbor_indices(pn_grid_t grid, int queries, int64_t* sums, int index_base, int accumulate) {
    if (!grid) return fail(PN_ERR_ARGUMENT, "grid is NULL");
    if (!sums) return fail(PN_ERR_ARGUMENT, "sums is NULL");
    pn::IndexSumF f;
    f.out = sums;
    f.accumulate = accumulate;
    f.base = index_base;
    return launch_traverse(*grid, queries, f);
}

// Whether k_fill_sorted can make the lists of the queries: a 3D FullGridCellList without a box or a
// batch, with enough points to fill the chip (r = 3 spacings, k_cells and sort / k_fill_sorted, us:
// 27,000 points 55 / 62, 125,000 points 90 / 86, F64 126 / 101).
static bool fill_sorted_possible(const pn_grid& g, const BinSet& Q) {
    if (g.nd != 3 || g.algorithm != 0 || g.geom.hash || g.geom.periodic || g.geom.table) return false;
    return g.grid.n_sel >= 100000 && Q.n_sel >= g.grid.n_sel;
}

// Whether it makes them, st being the grid's status with n_ordered what k_list_counts found: its fullest
// cell bounds a cell's candidates by what the kernel sorts in registers.  It shares a cell's sorted
// candidates among the cell's queries, so it needs many of them: from 14 points a cell on (us, a million
// points F32: 7.5 a cell 294 / 315, 10 a cell 310 / 347; 216,000 points with 14 a cell 120 / 104; whole
// builds 500,000 points with 12.5 a cell 286 / 305, F64 360 / 356, 16 a cell 376 / 328, 462 / 391; 2D with
// 16 a cell 196 / 203).  It gathers the candidates in the order of the original indices, which has to
// be near the order of the cells: more than four in ten of the points follow each other in both (a
// lattice at 2.4 spacings six; whole builds 500,000 points in no order 16 a cell 415 / 438, F64 503 / 614,
// 30 a cell 567 / 694, 734 / 1036).
static bool fill_sorted_applies(const pn::DevStatus& st) {
    if (st.n_binned < 100000 || st.n_binned / 14 < st.n_nonempty) return false;
    return 27 * (int64_t)st.max_count <= pn::FILL_CAP && 10 * st.n_ordered > 4 * pn::FILL_SAMPLES;
}

// Whether work is being captured on the stream (or may be: an implicit capture refuses the query).
static bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return status != hipStreamCaptureStatusNone;
}

int pn_csr_count(pn_grid_t grid, int queries, int64_t n_rows, int32_t* row_ptr, int32_t max_neighbors,
                 int64_t* nnz, int64_t* max_row) {
    if (!grid) return fail(PN_ERR_ARGUMENT, "grid is NULL");
    if (!row_ptr) return fail(PN_ERR_ARGUMENT, "row_ptr is NULL");
    pn_grid& g = *grid;
    const BinSet* Q = query_set(g, queries);
    if (!Q) return fail(PN_ERR_NOT_INITIALIZED, "the neighborhood search is not initialized");
    if (n_rows < Q->n_src) return fail(PN_ERR_ARGUMENT, "n_rows is smaller than the number of query points");
    if (n_rows > INT32_MAX - 1) return fail(PN_ERR_ARGUMENT, "too many rows");
    int rc;
    // the fill keeps the positions of the grid's points there once the counts are summed
    const int64_t n_counts = std::max(n_rows, std::max<int64_t>(g.grid.n_src, 1));
    if ((rc = g.csr_counts.ensure((size_t)n_counts * 4, g.stream))) return rc;
    if ((rc = g.csr_status.ensure(2 * sizeof(pn::DevStatus), g.stream))) return rc;
    if (!g.csr_host_status)
        PN_HIP(hipHostMalloc((void**)&g.csr_host_status, 2 * sizeof(pn::DevStatus), hipHostMallocDefault));
    auto* st = g.csr_status.as<pn::DevStatus>();
    // the grid's own status from the device: the host's copy is that of an earlier binning where a
    // captured one has been replayed
    g.csr_grid_known = fill_sorted_possible(g, *Q);
    g.csr_grid_seq = g.grid.mail_seq;
    const dim3 fill_blocks(blocks_for(std::min<int64_t>(n_rows, 1 << 20), 256));
    if (g.csr_grid_known) {  // fewer rows than samples (points selected repeatedly) count as no order
        hipLaunchKernelGGL(pn::k_list_status, dim3(1), dim3(1), 0, g.stream, g.grid.status.as<pn::DevStatus>(), st);
        PN_CHECK_LAUNCH();
        hipLaunchKernelGGL(pn::k_list_counts, fill_blocks, dim3(256), 0, g.stream, g.csr_counts.as<int32_t>(), n_rows,
                           g.grid.sorted_idx.as<int32_t>(), st);
    } else {
        hipLaunchKernelGGL(pn::k_reset_status, dim3(1), dim3(1), 0, g.stream, st);
        PN_CHECK_LAUNCH();
        hipLaunchKernelGGL(pn::k_fill_i32, fill_blocks, dim3(256), 0, g.stream, g.csr_counts.as<int32_t>(), n_rows, 0);
    }
    PN_CHECK_LAUNCH();
    pn::CountF f;
    f.out = g.csr_counts.as<int32_t>();
    f.accumulate = 0;
    // lists are mostly made of undeformed lattices, whose ties the cell kernel counts faster (128^3 at
    // r = 3 spacings F32 267 us, runs 400); other clouds' counts lose by it (1 M points at 2.4 spacings
    // 116 us, runs 90)
    if ((rc = launch_traverse(g, queries, f, false))) return rc;
    if ((rc = g.csr_scan.run(g.csr_counts.as<int32_t>(), n_rows, row_ptr, nullptr, st, g.stream))) return rc;
    PN_HIP(hipMemcpyAsync(g.csr_host_status, st, (g.csr_grid_known ? 2 : 1) * sizeof(pn::DevStatus),
                          hipMemcpyDeviceToHost, g.stream));
    PN_HIP(hipStreamSynchronize(g.stream));
    const pn::DevStatus hs = *g.csr_host_status;
    if (nnz) *nnz = (int64_t)hs.total64;
    if (max_row) *max_row = hs.max_count;
    if (hs.total64 > (unsigned long long)INT32_MAX)
        return fail(PN_ERR_UNSUPPORTED, "more than 2^31 - 1 neighbor pairs do not fit int32 row pointers");
    if (max_neighbors > 0 && hs.max_count > max_neighbors)
        return fail(PN_ERR_LIST_FULL, "cell list is full. Use a larger `max_points_per_cell`.");
    return PN_OK;
}

int pn_csr_fill(pn_grid_t grid, int queries, int64_t n_rows, const int32_t* row_ptr, int32_t* col_idx,
                int index_base) {
    if (!grid) return fail(PN_ERR_ARGUMENT, "grid is NULL");
    if (!row_ptr) return fail(PN_ERR_ARGUMENT, "row_ptr is NULL");
    pn_grid& g = *grid;
    const BinSet* Q = query_set(g, queries);
    if (!Q) return fail(PN_ERR_NOT_INITIALIZED, "the neighborhood search is not initialized");
    if (n_rows < Q->n_src) return fail(PN_ERR_ARGUMENT, "n_rows is smaller than the number of query points");
    if (g.csr_host_status && g.csr_host_status->max_count > pn::SORT_CAP)
        return fail(PN_ERR_UNSUPPORTED, "neighbor lists longer than 4096 entries are not supported");
    // by the grid's status at pn_csr_count; a captured fill may be replayed over another binning
    if (g.csr_grid_known && g.csr_grid_seq == g.grid.mail_seq && fill_sorted_possible(g, *Q) &&
        fill_sorted_applies(g.csr_host_status[1]) && (size_t)g.grid.n_src * 4 <= g.csr_counts.bytes &&
        !capturing(g.stream)) {
        const int max_count = g.csr_host_status[1].max_count;
        auto* inv = g.csr_counts.as<int32_t>();
        hipLaunchKernelGGL(pn::k_invert, dim3(blocks_for(g.grid.n_sel, 256)), dim3(256), 0, g.stream,
                           g.grid.sorted_idx.as<int32_t>(), g.grid.status.as<pn::DevStatus>(), inv);
        PN_CHECK_LAUNCH();
        const int64_t nwork = Q->stats_known ? Q->stats.n_nonempty : std::min<int64_t>(g.geom.ncells, Q->n_sel);
        const int nblocks = (int)std::min<int64_t>(round_up8(std::max<int64_t>(nwork, 1)), g.persist_blocks);
        // at least a cell's candidates; the network sorts 64 times a power of two keys
        int n_keys = 4 * pn::WAVE;
        while (n_keys < 27 * max_count) n_keys *= 2;
        const pn::FillArgs a{inv, row_ptr, col_idx, index_base};
        g.last_traversal = PN_TRAVERSAL_SORTED_FILL;
        LaunchTimer timer(g);  // brackets the one traversal kernel launched below
        return dispatch_trav(g, [&](auto dc, auto tcv, auto trv) -> int {
            if constexpr (decltype(dc)::value == 3) {
                using TC = decltype(tcv);
                using TR = decltype(trv);
                const TR r = (TR)g.radius;
                hipLaunchKernelGGL((pn::k_fill_sorted<3, TC, TR>), dim3(nblocks), dim3(pn::WAVE),
                                   n_keys * sizeof(int), g.stream, g.geom, Q->view(), g.grid.view(), r * r, a, n_keys,
                                   nblocks);
                PN_CHECK_LAUNCH();
            }
            return PN_OK;
        });
    }
    pn::FillF f;
    f.row_ptr = row_ptr;
    f.col = col_idx;
    f.base = index_base;
    f.row_end = 0;
    int rc = launch_traverse(g, queries, f);
    if (rc) return rc;
    if (n_rows == 0) return PN_OK;
    // persistent grids; the LDS sort only runs when some row is longer than 512 entries
    {
        const int nblocks = (int)std::min<int64_t>(round_up8(n_rows), 65536);
        hipLaunchKernelGGL(pn::k_sort_rows, dim3(nblocks), dim3(pn::WAVE), 0, g.stream, row_ptr, n_rows, col_idx,
                           nblocks);
        PN_CHECK_LAUNCH();
    }
    if (!g.csr_host_status || g.csr_host_status->max_count > pn::SORT_REGS_MAX) {
        const int nb_lds = (int)std::min<int64_t>(n_rows, 4096);
        hipLaunchKernelGGL(pn::k_sort_rows_lds, dim3(nb_lds), dim3(pn::WAVE), 0, g.stream, row_ptr, n_rows, col_idx,
                           nb_lds);
        PN_CHECK_LAUNCH();
    }
    return PN_OK;
}

}  // extern "C"
