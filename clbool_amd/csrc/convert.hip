// convert.hip -- format conversions between COO, CSR and DCSR.
//
// Restates src/common/matrices_conversions.cpp: coo_to_dcsr_shallow (:78-91,
// rows
// compressed by counting row starts per tile, cols shared), dcsr_to_coo_shallow /
// _deep (:43-76), dcsr_to_csr (:247-271, cols shared, nnz checked) and
// csr_to_dcsr (:211-244, empty rows dropped, cols shared).
#include "device_utils.hpp"
#include "expand.hpp"
#include "sort.hpp"

namespace clb {

// Rows of a COO matrix -> the DCSR row pointer and rows
// (prepare_array_for_rows_positions, prepare_positions.cl:29-44, and
// set_positions_rows, set_positions.cl:89-113).  A row starts where rows[i]
// differs from rows[i - 1].  The starts are counted per tile of RP_TILE
// entries, the tiles' counts are scanned, and a second pass places each start
// by its rank in the tile.  Both passes read the rows once, 16 bytes per lane;
// nothing of the size of nnz is written or scanned (flags and their scan over
// 16.1 million entries took 195 us).
constexpr u32 RP_WG = 256, RP_ROUNDS = 4, RP_TILE = RP_WG * RP_ROUNDS * 4;

// The flags (bit k: entry i + k starts a row) of the four entries at i.
__device__ __forceinline__ u32 row_start_bits(const u32 *__restrict__ rows, u32 n, u64 i, u32 (&v)[4]) {
    u32 prev = i && i < n ? rows[i - 1] : 0u;
    if (i + 4 <= n) {
        const uint4 x = *reinterpret_cast<const uint4 *>(rows + i);  // i is a multiple of 4
        v[0] = x.x;
        v[1] = x.y;
        v[2] = x.z;
        v[3] = x.w;
    } else {
#pragma unroll
        for (u32 k = 0; k < 4; ++k) v[k] = i + k < n ? rows[i + k] : 0u;
    }
    u32 f = 0;
#pragma unroll
    for (u32 k = 0; k < 4; ++k) {
        if (i + k < n && (i + k == 0 || v[k] != prev)) f |= 1u << k;
        prev = v[k];
    }
    return f;
}

__global__ __launch_bounds__(RP_WG) void k_row_starts_count(const u32 *__restrict__ rows, u32 n,
                                                            u32 *__restrict__ counts) {
    __shared__ u32 red[RP_WG / dev::WAVE + 1];
    const u64 base = (u64)blockIdx.x * RP_TILE;
    u32 c = 0;
#pragma unroll
    for (u32 q = 0; q < RP_ROUNDS; ++q) {
        u32 v[4];
        c += (u32)__popc(row_start_bits(rows, n, base + (q * RP_WG + threadIdx.x) * 4, v));
    }
    const u32 t = dev::block_sum<u32, RP_WG>(c, red);
    if (threadIdx.x == 0) counts[blockIdx.x] = t;
}

__global__ __launch_bounds__(RP_WG) void k_row_starts_place(const u32 *__restrict__ rows, u32 n,
                                                            const u32 *__restrict__ offs,
                                                            const u32 *__restrict__ total, u32 *__restrict__ rpt,
                                                            u32 *__restrict__ crows) {
    __shared__ u32 red[RP_WG / dev::WAVE + 1];
    const u64 base = (u64)blockIdx.x * RP_TILE;
    u32 at = offs[blockIdx.x];
    for (u32 q = 0; q < RP_ROUNDS; ++q) {
        const u64 i = base + (q * RP_WG + threadIdx.x) * 4;
        u32 v[4];
        const u32 f = row_start_bits(rows, n, i, v);
        u32 all;
        u32 p = at + dev::block_excl_scan<u32, RP_WG>((u32)__popc(f), red, all);
#pragma unroll
        for (u32 k = 0; k < 4; ++k)
            if ((f >> k) & 1u) {
                rpt[p] = (u32)i + k;
                crows[p] = v[k];
                ++p;
            }
        at += all;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) rpt[*total] = n;
}

void rows_to_dcsr(clb_controls_s *ctl, const u32 *rows, u32 nnz, clb_buffer_s **rpt_out, clb_buffer_s **rows_out,
                  u32 *nzr_out) {
    const u32 tiles = div_up(nnz, RP_TILE);
    DevArray<u32> offs(ctl, (u64)tiles + 1);  // [tiles]: the number of rows
    k_row_starts_count<<<tiles, RP_WG, 0, ctl->stream>>>(rows, nnz, offs.ptr);
    CLB_LAUNCHED("prepare_array_for_rows_positions");
    exclusive_scan_u32(ctl, offs.ptr, offs.ptr, tiles, offs.ptr + tiles);
    u32 nzr = 0;
    readback(ctl, &nzr, offs.ptr + tiles, 4);
    clb_buffer_s *rpt = buffer_new(ctl, 4ull * (nzr + 1ull));
    clb_buffer_s *cr = nullptr;
    try {
        cr = buffer_new(ctl, 4ull * (nzr ? nzr : 1));
        k_row_starts_place<<<tiles, RP_WG, 0, ctl->stream>>>(rows, nnz, offs.ptr, offs.ptr + tiles, u32p(rpt),
                                                             u32p(cr));
        CLB_LAUNCHED("set_positions_rows");
        sync(ctl);
    } catch (...) {
        buffer_release(rpt);
        buffer_release(cr);
        throw;
    }
    *rpt_out = rpt;
    *rows_out = cr;
    *nzr_out = nzr;
}

// dscr_to_coo (dscr_to_coo.cl:8-23)
struct RowOfNonzero {
    u32 *out;
    __device__ __forceinline__ void operator()(u32 e, u32, u32 id) const { out[e] = id; }
};

void dcsr_expand_rows(clb_controls_s *ctl, const u32 *rpt, const u32 *rows, u32 nzr, u32 nnz, u32 *out_rows) {
    expand_rows(ctl, Expand<RowOfNonzero>{rpt, rows, 0, nzr, 0, nnz, {out_rows}});
}

// dcsr_to_csr_set_size (conversions.cl:8-18)
__global__ void k_dcsr_row_sizes(const u32 *__restrict__ rpt, const u32 *__restrict__ rows, u32 nzr, u32 nrows,
                                 u32 *__restrict__ csr_rpt) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nzr && rows[i] <= nrows) csr_rpt[rows[i]] = rpt[i + 1] - rpt[i];
}

// prepare_for_shift_empty_rows (prepare_positions.cl:69-84)
__global__ void k_nonempty_flags(const u32 *__restrict__ rpt, u32 n, u32 *__restrict__ flags) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flags[i] = rpt[i] != rpt[i + 1];
    if (i == n) flags[n] = 0;
}

// set_positions_pointers_and_rows_csr (set_positions.cl:69-85)
__global__ void k_csr_set_positions(const u32 *__restrict__ rpt, const u32 *__restrict__ pos, u32 nrows,
                                    u32 *__restrict__ c_rpt, u32 *__restrict__ c_rows) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) c_rpt[pos[nrows]] = rpt[nrows];
    if (i < nrows && pos[i] != pos[i + 1]) {
        c_rpt[pos[i]] = rpt[i];
        c_rows[pos[i]] = i;
    }
}

}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_coo_to_dcsr_shallow(clb_controls ctl, const clb_coo *a, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        clb_dcsr r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz != 0) {
            rows_to_dcsr(ctl, u32p(a->rows), a->nnz, &r.rpt, &r.rows, &r.nzr);
            buffer_retain(a->cols);  // shallow: the columns are shared
            r.cols = a->cols;
            r.nnz = a->nnz;
        }
        *out = r;
    });
}

static void dcsr_to_coo(clb_controls ctl, const clb_dcsr *a, clb_coo *out, bool deep) {
    clb_coo r{};
    r.nrows = a->nrows;
    r.ncols = a->ncols;
    if (a->nnz != 0) {
        r.rows = buffer_new(ctl, 4ull * a->nnz);
        try {
            dcsr_expand_rows(ctl, u32p(a->rpt), u32p(a->rows), a->nzr, a->nnz, u32p(r.rows));
            if (deep) {
                r.cols = buffer_new(ctl, 4ull * a->nnz);
                CLB_HIP(hipMemcpyAsync(r.cols->ptr, a->cols->ptr, 4ull * a->nnz, hipMemcpyDeviceToDevice,
                                       ctl->stream),
                        COPY_BUFFER_ERROR);
            } else {
                buffer_retain(a->cols);
                r.cols = a->cols;
            }
            sync(ctl);
        } catch (...) {
            settle(ctl);
            clb_coo_release(&r);
            throw;
        }
        r.nnz = a->nnz;
    }
    *out = r;
}

clb_status clb_dcsr_to_coo_shallow(clb_controls ctl, const clb_dcsr *a, clb_coo *out) {
    return run_guarded(ctl, [&] { dcsr_to_coo(ctl, a, out, false); });
}

clb_status clb_dcsr_to_coo_deep(clb_controls ctl, const clb_dcsr *a, clb_coo *out) {
    return run_guarded(ctl, [&] { dcsr_to_coo(ctl, a, out, true); });
}

clb_status clb_dcsr_to_csr(clb_controls ctl, const clb_dcsr *a, clb_csr *out) {
    return run_guarded(ctl, [&] {
        clb_csr r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz == 0) {  // :248-250
            *out = r;
            return;
        }
        const u64 n1 = (u64)a->nrows + 1;
        r.rpt = buffer_new(ctl, 4ull * n1);
        try {
            fill_u32(ctl, u32p(r.rpt), n1, 0);
            k_dcsr_row_sizes<<<div_up(a->nzr, 256), 256, 0, ctl->stream>>>(u32p(a->rpt), u32p(a->rows), a->nzr,
                                                                             a->nrows, u32p(r.rpt));
            CLB_LAUNCHED("dcsr_to_csr_set_size");
            DevArray<u32> tot(ctl, 1);
            exclusive_scan_u32(ctl, u32p(r.rpt), u32p(r.rpt), n1, tot.ptr);
            u32 c_nnz = 0;
            readback(ctl, &c_nnz, tot.ptr, 4);
            // :268
            if (c_nnz != a->nnz) raise(INVALID_VALUE, "nnz in dcsr and csr matrices should be equal!");
        } catch (...) {
            settle(ctl);
            buffer_release(r.rpt);
            throw;
        }
        buffer_retain(a->cols);
        r.cols = a->cols;
        r.nnz = a->nnz;
        *out = r;
    });
}

clb_status clb_csr_to_dcsr(clb_controls ctl, const clb_csr *a, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        clb_dcsr r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz == 0) {  // :212-214
            *out = r;
            return;
        }
        const u64 n1 = (u64)a->nrows + 1;
        DevArray<u32> pos(ctl, n1);
        k_nonempty_flags<<<div_up(n1, 256), 256, 0, ctl->stream>>>(u32p(a->rpt), a->nrows, pos.ptr);
        CLB_LAUNCHED("prepare_for_shift_empty_rows");
        DevArray<u32> tot(ctl, 1);
        exclusive_scan_u32(ctl, pos.ptr, pos.ptr, n1, tot.ptr);
        u32 nzr = 0;
        readback(ctl, &nzr, tot.ptr, 4);
        r.rpt = buffer_new(ctl, 4ull * (nzr + 1ull));
        try {
            r.rows = buffer_new(ctl, 4ull * (nzr ? nzr : 1));
            k_csr_set_positions<<<div_up(n1, 256), 256, 0, ctl->stream>>>(u32p(a->rpt), pos.ptr, a->nrows,
                                                                           u32p(r.rpt), u32p(r.rows));
            CLB_LAUNCHED("set_positions_pointers_and_rows_csr");
            sync(ctl);
        } catch (...) {
            clb_dcsr_release(&r);
            throw;
        }
        buffer_retain(a->cols);
        r.cols = a->cols;
        r.nnz = a->nnz;
        r.nzr = nzr;
        *out = r;
    });
}

}  // extern "C"
