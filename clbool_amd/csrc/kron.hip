// kron.hip -- DCSR Kronecker product C = A (x) B.
//
// dcsr::kronecker_product (src/dcsr/dcsr_kronecker_product.cpp:6-65) with
// count_nnz_per_row / calculate_kronecker_product (dcsr_kronecker.cl:38-98):
// output row r = ia * b_nzr + ib has |A_ia| * |B_ib| entries, row id
// a_row * b_nrows + b_row and columns a_col * b_ncols + b_col (already in
// ascending order).  Output rows are A-row-major, so row (ia, ib) starts at
// a_rpt[ia] * b_nnz + |A_ia| * b_rpt[ib]: the row pointer is a closed form,
// no scan.  The reference finds each output's row by a binary search per
// nonzero; here the work is cut into tiles of B nonzeros (one workgroup per
// tile and group of A rows): a partition pass finds each tile's first B row, the
// tile's slice of b_rpt is staged in LDS, and each thread places its B nonzero once
// per column of the A row -- consecutive threads write consecutive columns.
// Sizes are checked in 64 bits: the reference computes nnz, nzr and the
// shape as wrapping uint32 products (:10-13), which this library reports as
// an error instead.
#include "clb_internal.hpp"

#include "device_utils.hpp"

namespace clb {

constexpr u32 KRON_WG = 256, KRON_ITEMS = 4, KRON_TILE = KRON_WG * KRON_ITEMS;
// A group of A rows shares the search of a tile's rows.  R-MAT 65536 x 16 and
// an automaton of 64 states and 200 moves (764 MB) / of 30 and 40: 251 / 95 us
// with a group per A row; about 6 A nonzeros to a group 220 / 67, 10 229 / 62,
// 16 235 / 62 (later pieces of a line are stored further apart).
constexpr u32 KRON_MIN_GRID = 1u << 12, KRON_GROUP = 8;

__global__ void k_kron_rows(const u32 *__restrict__ a_rpt, const u32 *__restrict__ b_rpt,
                            const u32 *__restrict__ a_rows, const u32 *__restrict__ b_rows, u32 c_nzr, u32 b_nzr,
                            u32 b_nnz, u32 b_nrows, u32 c_nnz, u32 *__restrict__ c_rpt, u32 *__restrict__ c_rows) {
    const u32 r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r == 0) c_rpt[c_nzr] = c_nnz;
    if (r >= c_nzr) return;
    const u32 ia = r / b_nzr, ib = r % b_nzr;
    c_rpt[r] = a_rpt[ia] * b_nnz + (a_rpt[ia + 1] - a_rpt[ia]) * b_rpt[ib];
    c_rows[r] = a_rows[ia] * b_nrows + b_rows[ib];
}

// first[t] = the B row holding B nonzero t * KRON_TILE.
__global__ void k_kron_tiles(const u32 *__restrict__ b_rpt, u32 b_nzr, u32 ntiles, u32 *__restrict__ first) {
    const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    const u32 e = t * KRON_TILE;
    u32 lo = 0, hi = b_nzr;  // last row with b_rpt[row] <= e
    while (hi - lo > 1) {
        const u32 mid = lo + (hi - lo) / 2;
        if (b_rpt[mid] <= e) lo = mid;
        else hi = mid;
    }
    first[t] = lo;
}

// Workgroup (tile, group): B nonzeros [tile * KRON_TILE, +KRON_TILE) times the
// A rows [group * per, +per).  Stores bound it, in pieces of a B row's length:
// 3.6 TB/s of a fill's 6.9 at 191 million nonzeros.  Stores of 16 bytes from
// positions found by a search each, and from a tile put together in LDS, were
// slower (336 and 417 us against 225 for the kernel alone): what they add to
// the chain of a workgroup costs more than whole lines save.
__global__ __launch_bounds__(KRON_WG) void k_kron_fill(const u32 *__restrict__ first, u32 ntiles, u32 per, u32 a_nzr,
                                                       const u32 *__restrict__ a_rpt, const u32 *__restrict__ a_cols,
                                                       const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_cols,
                                                       u32 b_nzr, u32 b_nnz, u32 b_ncols, u32 *__restrict__ c_cols) {
    __shared__ u32 srpt[KRON_TILE + 1];
    const u32 tile = blockIdx.x % ntiles, ia0 = blockIdx.x / ntiles * per;
    const u32 ia1 = a_nzr - ia0 < per ? a_nzr : ia0 + per;
    const u32 e0 = tile * KRON_TILE;
    const u32 e1 = b_nnz - e0 < KRON_TILE ? b_nnz : e0 + KRON_TILE;
    const u32 ib0 = first[tile];
    u32 a0 = a_rpt[ia0], a1 = a_rpt[ia0 + 1];  // needed last: on their way meanwhile
    // the tile's rows start at ib0 and number at most KRON_TILE (each holds a
    // nonzero); srpt[j] = b_rpt[ib0 + j], the end row clamped to b_nzr
    const u32 nr = b_nzr - ib0 < KRON_TILE ? b_nzr - ib0 : KRON_TILE;
    for (u32 j = threadIdx.x; j <= nr; j += KRON_WG) srpt[j] = b_rpt[ib0 + j];
    __syncthreads();
    auto row_of = [&](u32 e) {  // last j with srpt[j] <= e
        u32 lo = 0, hi = nr;
        while (hi - lo > 1) {
            const u32 mid = (lo + hi) >> 1;
            if (srpt[mid] <= e) lo = mid;
            else hi = mid;
        }
        return lo;
    };
    if (per == 1) {  // nothing to share: each item's stores behind its own search
        const u32 alen = a1 - a0, abase = a0 * b_nnz;
#pragma unroll
        for (u32 i = 0; i < KRON_ITEMS; ++i) {
            const u32 e = e0 + i * KRON_WG + threadIdx.x;
            if (e >= e1) break;
            const u32 j = row_of(e), rs = srpt[j], blen = srpt[j + 1] - rs, bc = b_cols[e];
            u32 *out = c_cols + abase + alen * rs + (e - rs);
            for (u32 ka = 0; ka < alen; ++ka) out[ka * blen] = a_cols[a0 + ka] * b_ncols + bc;
        }
        return;
    }
    u32 rs[KRON_ITEMS], blen[KRON_ITEMS], bc[KRON_ITEMS];
#pragma unroll
    for (u32 i = 0; i < KRON_ITEMS; ++i) {
        const u32 e = e0 + i * KRON_WG + threadIdx.x, j = row_of(e);
        rs[i] = srpt[j];
        blen[i] = srpt[j + 1] - rs[i];
        bc[i] = e < e1 ? b_cols[e] : 0u;
    }
    for (u32 ia = ia0; ia < ia1; ++ia) {
        const u32 next = ia + 1 < ia1 ? a_rpt[ia + 2] : 0u;
        const u32 alen = a1 - a0, abase = a0 * b_nnz;
#pragma unroll
        for (u32 i = 0; i < KRON_ITEMS; ++i) {
            const u32 e = e0 + i * KRON_WG + threadIdx.x;
            u32 *out = c_cols + abase + alen * rs[i] + (e - rs[i]);
            if (e < e1)
                for (u32 ka = 0; ka < alen; ++ka) out[ka * blen[i]] = a_cols[a0 + ka] * b_ncols + bc[i];
        }
        a0 = a1;
        a1 = next;
    }
}

}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_dcsr_kronecker(clb_controls ctl, const clb_dcsr *a, const clb_dcsr *b, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        const u64 c_nnz = (u64)a->nnz * b->nnz;
        const u64 c_nzr = (u64)a->nzr * b->nzr;
        const u64 c_nrows = (u64)a->nrows * b->nrows;
        const u64 c_ncols = (u64)a->ncols * b->ncols;
        if (c_nrows > 0xFFFFFFFFull || c_ncols > 0xFFFFFFFFull)
            raise(INVALID_VALUE, "kronecker product shape exceeds uint32 indices");
        clb_dcsr r{};
        r.nrows = (u32)c_nrows;
        r.ncols = (u32)c_ncols;
        if (c_nnz == 0) {  // :15-18
            *out = r;
            return;
        }
        if (c_nnz > 0xFFFFFFFFull) raise(INVALID_VALUE, "kronecker product has more than 2^32-1 nonzeros");
        try {
            r.rpt = buffer_new(ctl, 4ull * (c_nzr + 1));
            r.rows = buffer_new(ctl, 4ull * c_nzr);
            r.cols = buffer_new(ctl, 4ull * c_nnz);
            k_kron_rows<<<div_up(c_nzr + 1, 256), 256, 0, ctl->stream>>>(u32p(a->rpt), u32p(b->rpt), u32p(a->rows),
                                                                         u32p(b->rows), (u32)c_nzr, b->nzr, b->nnz,
                                                                         b->nrows, (u32)c_nnz, u32p(r.rpt),
                                                                         u32p(r.rows));
            CLB_LAUNCHED("count_nnz_per_row");
            const u32 ntiles = div_up(b->nnz, KRON_TILE);
            DevArray<u32> first(ctl, ntiles);
            k_kron_tiles<<<div_up(ntiles, 256), 256, 0, ctl->stream>>>(u32p(b->rpt), b->nzr, ntiles, first.ptr);
            CLB_LAUNCHED("kron_tiles");
            // whole A rows to a workgroup: about KRON_GROUP of A's nonzeros,
            // but no fewer than KRON_MIN_GRID workgroups
            u64 per = ((u64)KRON_GROUP * a->nzr + a->nnz / 2) / a->nnz;
            const u64 most = (u64)ntiles * a->nzr / KRON_MIN_GRID;
            if (per > most) per = most;
            if (per < 1) per = 1;
            // and no more than 2^23 (2^31 threads)
            while (ntiles * (((u64)a->nzr + per - 1) / per) > (1u << 23)) per *= 2;
            const u64 groups = ((u64)a->nzr + per - 1) / per;
            k_kron_fill<<<(u32)(ntiles * groups), KRON_WG, 0, ctl->stream>>>(
                first.ptr, ntiles, (u32)per, a->nzr, u32p(a->rpt), u32p(a->cols), u32p(b->rpt), u32p(b->cols), b->nzr,
                b->nnz, b->ncols, u32p(r.cols));
            CLB_LAUNCHED("calculate_kronecker_product");
            sync(ctl);
        } catch (...) {
            settle(ctl);
            clb_dcsr_release(&r);
            throw;
        }
        r.nnz = (u32)c_nnz;
        r.nzr = (u32)c_nzr;
        *out = r;
    });
}

}  // extern "C"
