// addition.hip -- boolean matrix addition (union) by merge path.
//
// coo::matrix_addition (src/coo/coo_matrix_addition.cpp:32-73) merges two
// sorted (row, col) lists with merge_path.cl:182-261 and then drops
// duplicates (reduce_duplicates2, matrix_coo.cpp:117-170).  Here the pairs
// are 64-bit keys row << 32 | col, and every tile of the merge is deduplicated
// where it was merged, in LDS.
//
// csr::matrix_addition (src/csr/csr_addition.cpp:26-168) bins rows by length
// and merges each row in a workgroup.  Because CSR rows with sorted columns
// are already one globally sorted key list, the same flat merge handles it
// with no per-row load imbalance; the CSR row pointer is rebuilt by one
// lower-bound search per row.  The DCSR union (the X += T step of a closure)
// reuses the same engine.
#include "device_utils.hpp"
#include "expand.hpp"
#include "sort.hpp"

namespace clb {

// Merge of two ascending key lists, in tiles of MG_TILE outputs.  A first
// pass finds where every tile boundary cuts A (merge_path.cl:38-90: the
// number of A elements among the first d outputs, A first on ties), one
// thread per boundary.  Each workgroup then loads its tile's pieces of A and B
// into LDS with coalesced loads, every thread merges MG_ITEMS consecutive
// outputs from LDS (its own merge-path search within the tile), and the tile
// is written back with coalesced stores.
constexpr int MG_WG = 256, MG_ITEMS = 8, MG_TILE = MG_WG * MG_ITEMS;

__global__ void k_merge_partition(const u64 *__restrict__ A, u64 na, const u64 *__restrict__ B, u64 nb, u64 ntiles,
                                  u64 *__restrict__ split) {
    const u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (t > ntiles) return;
    const u64 total = na + nb;
    const u64 d = t * MG_TILE < total ? t * MG_TILE : total;
    u64 lo = d > nb ? d - nb : 0, hi = d < na ? d : na;
    while (lo < hi) {
        const u64 mid = (lo + hi) >> 1;
        if (A[mid] <= B[d - 1 - mid]) lo = mid + 1;
        else hi = mid;
    }
    split[t] = lo;
}

// Merges elements [a0, a1) of A and the tile's share of B into s[0, n) (LDS).
__device__ __forceinline__ void merge_tile(const u64 *__restrict__ A, const u64 *__restrict__ B, u64 a0, u64 b0,
                                           u32 la, u32 n, u64 *s) {
    const u32 lb = n - la;
    for (u32 t = threadIdx.x; t < n; t += MG_WG) s[t] = t < la ? A[a0 + t] : B[b0 + (t - la)];
    __syncthreads();
    if (la && lb) {  // uniform
        const u32 k0 = threadIdx.x * MG_ITEMS;
        u64 v[MG_ITEMS];
        if (k0 < n) {
            u32 lo = k0 > lb ? k0 - lb : 0, hi = k0 < la ? k0 : la;
            while (lo < hi) {
                const u32 mid = (lo + hi) >> 1;
                if (s[mid] <= s[la + k0 - 1 - mid]) lo = mid + 1;
                else hi = mid;
            }
            u32 i = lo, j = k0 - lo;
#pragma unroll
            for (int k = 0; k < MG_ITEMS; ++k) {
                const bool take_a = i < la && (j >= lb || s[i] <= s[la + j]);
                v[k] = s[take_a ? i : (j < lb ? la + j : n - 1)];  // n - 1: past the tile, never stored
                i += take_a;
                j += !take_a;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MG_ITEMS; ++k)
            if (k0 + k < n) s[k0 + k] = v[k];
        __syncthreads();
    }
}

// The tile of a merge of A and B that workgroup blockIdx.x takes.
struct MergeTile {
    u64 d0, a0, b0;
    u32 la, n;
    __device__ __forceinline__ MergeTile(u64 na, u64 nb, const u64 *__restrict__ split) {
        const u64 total = na + nb;
        d0 = (u64)blockIdx.x * MG_TILE;
        const u64 d1 = d0 + MG_TILE < total ? d0 + MG_TILE : total;
        a0 = split[blockIdx.x];
        b0 = d0 - a0;
        la = (u32)(split[blockIdx.x + 1] - a0);
        n = (u32)(d1 - d0);
    }
};

__global__ __launch_bounds__(MG_WG) void k_merge_tiles(const u64 *__restrict__ A, u64 na, const u64 *__restrict__ B,
                                                       u64 nb, const u64 *__restrict__ split,
                                                       u64 *__restrict__ out) {
    __shared__ u64 s[MG_TILE];
    const MergeTile t(na, nb, split);
    merge_tile(A, B, t.a0, t.b0, t.la, t.n, s);
    for (u32 o = threadIdx.x; o < t.n; o += MG_WG) out[t.d0 + o] = s[o];
}

// Union of two ascending key lists: the merge of each tile stays in LDS and is
// done twice, once to count its distinct keys and row starts and, once the
// counts are scanned, to place them.  Against writing the merged list and
// deduplicating it in two passes of its own this reads the lists once more
// instead of writing 8 bytes per key and reading them three times: 20.2
// million keys took 69 + 36 + 60 us and four scan launches, now 58 + 70 and two.
//
// The lists may hold the rows of several matrices, matrix x in rows
// [x * n, (x + 1) * n) (n = 0: one matrix).  The first tile that holds or
// follows matrix x's place notes how many of its keys come before it.
struct UnionBound {
    u32 tile, kept, starts, pad;
};

// bit 0: key s[o] is kept (differs from the one before it), bit 1: it starts a row
__device__ __forceinline__ u32 union_flags(const u64 *s, u32 o, bool first, u64 prev) {
    const u64 k = s[o], p = o ? s[o - 1] : prev;
    if (o == 0 && first) return 3u;
    return k == p ? 0u : ((k >> 32) != (p >> 32) ? 3u : 1u);
}

__device__ __forceinline__ u64 key_before(const u64 *__restrict__ A, const u64 *__restrict__ B, const MergeTile &t) {
    const u64 x = t.a0 ? A[t.a0 - 1] : 0ull, y = t.b0 ? B[t.b0 - 1] : 0ull;
    return x > y ? x : y;
}

// counts[tile] = kept keys | row starts << 32
__global__ __launch_bounds__(MG_WG) void k_union_count(const u64 *__restrict__ A, u64 na, const u64 *__restrict__ B,
                                                       u64 nb, const u64 *__restrict__ split, u32 n, u32 nmat,
                                                       u64 *__restrict__ counts, UnionBound *__restrict__ bounds) {
    __shared__ u64 s[MG_TILE];
    __shared__ u32 red[MG_WG / dev::WAVE + 1];
    const MergeTile t(na, nb, split);
    merge_tile(A, B, t.a0, t.b0, t.la, t.n, s);
    const u64 prev = key_before(A, B, t);
    u32 fl = 0;  // item q's flags at bits 2q
#pragma unroll
    for (int q = 0; q < MG_ITEMS; ++q) {
        const u32 o = q * MG_WG + threadIdx.x;
        if (o < t.n) fl |= union_flags(s, o, t.d0 == 0, prev) << (2 * q);
    }
    // at most 2048 of either per tile: both sums in one word
    const u32 c = (u32)__popc(fl & 0x5555u) | ((u32)__popc(fl & 0xAAAAu) << 16);
    const u32 sum = dev::block_sum<u32, MG_WG>(c, red);
    if (threadIdx.x == 0) counts[blockIdx.x] = (u64)(sum & 0xFFFFu) | ((u64)(sum >> 16) << 32);
    if (n) {
        // matrices that begin in this tile, or after the key before it
        const u32 x0 = t.d0 ? (u32)(prev >> 32) / n + 1u : 0u;
        const u32 x1 = (u32)(s[t.n - 1] >> 32) / n;
        for (u32 x = x0; x <= x1 && x < nmat; ++x) {  // uniform
            const u64 lim = (u64)((u64)x * n) << 32;
            u32 below = 0;
#pragma unroll
            for (int q = 0; q < MG_ITEMS; ++q) {
                const u32 o = q * MG_WG + threadIdx.x;
                if (o < t.n && s[o] < lim) {
                    below += (fl >> (2 * q)) & 1u;
                    below += ((fl >> (2 * q + 1)) & 1u) << 16;
                }
            }
            const u32 b = dev::block_sum<u32, MG_WG>(below, red);
            if (threadIdx.x == 0) bounds[x] = UnionBound{blockIdx.x, b & 0xFFFFu, b >> 16, 0u};
        }
    }
}

// out[2x], out[2x + 1] = kept keys and row starts before matrix x; bounds that
// no tile noted (tile == ~0) lie after the last key.  x = nmat: the totals.
__global__ void k_union_bounds(const UnionBound *__restrict__ bounds, u32 nmat, const u64 *__restrict__ offs,
                               const u64 *__restrict__ total, u32 *__restrict__ out) {
    const u32 x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x > nmat) return;
    u64 v = *total;
    if (x < nmat && bounds[x].tile != 0xFFFFFFFFu)
        v = offs[bounds[x].tile] + bounds[x].kept + ((u64)bounds[x].starts << 32);
    out[2 * x] = (u32)v;
    out[2 * x + 1] = (u32)(v >> 32);
}

// Where the union goes.  DCSR of one matrix: cols[p] = column of the p-th
// kept key; rows[q], rpt[q] = row and p of the q-th row start.  Pairs: rows[p]
// instead.  Several matrices: one DCSR each (cols == nullptr: not written).
struct UnionDcsr {
    u32 *cols, *rows, *rpt;
    u32 kept0, starts0, kept1, starts1;  // its first key's and row's ranks, and its end's
};

template <int KIND>  // 0: pairs, 1: one DCSR, 2: several
__global__ __launch_bounds__(MG_WG) void k_union_place(const u64 *__restrict__ A, u64 na, const u64 *__restrict__ B,
                                                       u64 nb, const u64 *__restrict__ split, u32 n,
                                                       const u64 *__restrict__ offs, UnionDcsr one,
                                                       const UnionDcsr *__restrict__ many, u32 nmat) {
    constexpr u32 NW = MG_WG / dev::WAVE;
    __shared__ u64 s[MG_TILE];
    __shared__ u32 wcnt[MG_ITEMS][NW];
    const MergeTile t(na, nb, split);
    merge_tile(A, B, t.a0, t.b0, t.la, t.n, s);
    const u64 prev = key_before(A, B, t);
    const u32 w = dev::wave_id();
    u32 fl = 0;
    u64 bk[MG_ITEMS], bs[MG_ITEMS];
#pragma unroll
    for (int q = 0; q < MG_ITEMS; ++q) {
        const u32 o = q * MG_WG + threadIdx.x;
        const u32 f = o < t.n ? union_flags(s, o, t.d0 == 0, prev) : 0u;
        fl |= f << (2 * q);
        bk[q] = __ballot(f & 1u);
        bs[q] = __ballot(f >> 1);
        if (dev::lane() == 0) wcnt[q][w] = (u32)__popcll(bk[q]) | ((u32)__popcll(bs[q]) << 16);
    }
    __syncthreads();
    const u64 off = offs[blockIdx.x];
    u32 p0 = (u32)off, q0 = (u32)(off >> 32);
    const u32 xa = KIND == 2 ? (u32)(s[0] >> 32) / n : 0u;
    const bool same = KIND != 2 || (u32)(s[t.n - 1] >> 32) / n == xa;  // uniform
    const UnionDcsr ua = KIND == 2 ? many[xa] : one;
#pragma unroll
    for (int q = 0; q < MG_ITEMS; ++q) {
        u32 before = 0, all = 0;
#pragma unroll
        for (u32 v = 0; v < NW; ++v) {
            const u32 c = wcnt[q][v];
            before += v < w ? c : 0u;
            all += c;
        }
        if ((fl >> (2 * q)) & 1u) {
            const u64 k = s[q * MG_WG + threadIdx.x];
            const u32 p = p0 + (before & 0xFFFFu) + dev::lanes_below(bk[q]);
            const u32 row = (u32)(k >> 32);
            if (KIND == 0) {
                one.cols[p] = (u32)k;
                one.rows[p] = row;
            } else {
                const u32 x = same ? xa : row / n;
                const UnionDcsr u = same ? ua : many[x];
                if (KIND == 1 || u.cols) {
                    u.cols[p - u.kept0] = (u32)k;
                    if ((fl >> (2 * q + 1)) & 1u) {
                        const u32 z = q0 + (before >> 16) + dev::lanes_below(bs[q]) - u.starts0;
                        u.rows[z] = KIND == 2 ? row - x * n : row;
                        u.rpt[z] = p - u.kept0;
                    }
                }
            }
        }
        p0 += all & 0xFFFFu;
        q0 += all >> 16;
    }
    if (blockIdx.x == 0) {
        if (KIND == 1 && threadIdx.x == 0) one.rpt[one.starts1 - one.starts0] = one.kept1 - one.kept0;
        if (KIND == 2)
            for (u32 x = threadIdx.x; x < nmat; x += MG_WG)
                if (many[x].cols) many[x].rpt[many[x].starts1 - many[x].starts0] = many[x].kept1 - many[x].kept0;
    }
}

// CSR row pointer of sorted rows: rpt[r] = lower_bound(rows, r), r <= nrows.
__global__ void k_rows_lower_bound(const u32 *__restrict__ rows, u32 m, u32 nrows, u32 *__restrict__ rpt) {
    const u32 r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nrows) return;
    u32 lo = 0, hi = m;
    while (lo < hi) {
        const u32 mid = lo + (hi - lo) / 2;
        if (rows[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    rpt[r] = lo;
}

// Tile boundaries of a merge.
static u32 merge_split(clb_controls_s *ctl, const u64 *a, u64 na, const u64 *b, u64 nb, DevArray<u64> &split) {
    const u64 tiles = (na + nb + MG_TILE - 1) / MG_TILE;
    if (tiles >= 0xFFFFFFFFull) raise(INVALID_VALUE, "merge larger than the grid allows");
    split.reset(ctl, tiles + 1);
    k_merge_partition<<<div_up(tiles + 1, 64), 64, 0, ctl->stream>>>(a, na, b, nb, tiles, split.ptr);
    CLB_LAUNCHED("merge_partition");
    return (u32)tiles;
}

void merge_keys(clb_controls_s *ctl, const u64 *a, u64 na, const u64 *b, u64 nb, u64 *out) {
    if (na + nb == 0) return;
    DevArray<u64> split;
    const u32 tiles = merge_split(ctl, a, na, b, nb, split);
    k_merge_tiles<<<tiles, MG_WG, 0, ctl->stream>>>(a, na, b, nb, split.ptr, out);
    CLB_LAUNCHED("merge");
}

// The counting half of a union, shared by its forms: split and offs (kept |
// starts << 32 before each tile, offs[tiles]: the totals).
struct UnionCounts {
    DevArray<u64> split, offs;
    u32 tiles = 0;
};
static void union_count(clb_controls_s *ctl, const u64 *a, u64 na, const u64 *b, u64 nb, u32 n, u32 nmat,
                        UnionBound *bounds, UnionCounts &c) {
    if (na + nb >= 0xFFFFFFFFull) raise(INVALID_VALUE, "more keys than uint32 indices allow");
    c.tiles = merge_split(ctl, a, na, b, nb, c.split);
    c.offs.reset(ctl, (u64)c.tiles + 1);
    k_union_count<<<c.tiles, MG_WG, 0, ctl->stream>>>(a, na, b, nb, c.split.ptr, n, nmat, c.offs.ptr, bounds);
    CLB_LAUNCHED("union_count");
    exclusive_scan_u64(ctl, c.offs.ptr, c.offs.ptr, c.tiles, c.offs.ptr + c.tiles);
}

// Union of two sorted key lists -> (rows, cols) buffers.
static u32 union_keys(clb_controls_s *ctl, const u64 *ka, u64 na, const u64 *kb, u64 nb, clb_buffer_s **rows,
                      clb_buffer_s **cols) {
    *rows = *cols = nullptr;
    if (na + nb == 0) {
        *rows = buffer_new(ctl, 4);
        *cols = buffer_new(ctl, 4);
        return 0;
    }
    UnionCounts c;
    union_count(ctl, ka, na, kb, nb, 0, 0, nullptr, c);
    u64 total = 0;
    readback(ctl, &total, c.offs.ptr + c.tiles, 8);
    const u32 m = (u32)total;
    *rows = buffer_new(ctl, 4ull * m);
    try {
        *cols = buffer_new(ctl, 4ull * m);
        k_union_place<0><<<c.tiles, MG_WG, 0, ctl->stream>>>(ka, na, kb, nb, c.split.ptr, 0, c.offs.ptr,
                                                             UnionDcsr{u32p(*cols), u32p(*rows), nullptr, 0, 0, 0, 0},
                                                             nullptr, 0);
        CLB_LAUNCHED("union_place");
    } catch (...) {
        buffer_release(*rows);
        buffer_release(*cols);
        *rows = *cols = nullptr;
        throw;
    }
    return m;
}

// Union of two sorted key lists -> a canonical DCSR (out.nrows/ncols are kept).
static void union_keys_to_dcsr(clb_controls_s *ctl, const u64 *ka, u64 na, const u64 *kb, u64 nb, clb_dcsr &out) {
    UnionCounts c;
    union_count(ctl, ka, na, kb, nb, 0, 0, nullptr, c);
    u64 total = 0;
    readback(ctl, &total, c.offs.ptr + c.tiles, 8);
    const u32 m = (u32)total, nzr = (u32)(total >> 32);
    clb_dcsr r{};
    r.nrows = out.nrows;
    r.ncols = out.ncols;
    try {
        r.cols = buffer_new(ctl, 4ull * m);
        r.rows = buffer_new(ctl, 4ull * nzr);
        r.rpt = buffer_new(ctl, 4ull * (nzr + 1ull));
        k_union_place<1><<<c.tiles, MG_WG, 0, ctl->stream>>>(
            ka, na, kb, nb, c.split.ptr, 0, c.offs.ptr,
            UnionDcsr{u32p(r.cols), u32p(r.rows), u32p(r.rpt), 0, 0, m, nzr}, nullptr, 0);
        CLB_LAUNCHED("union_place");
        sync(ctl);
    } catch (...) {
        clb_dcsr_release(&r);
        throw;
    }
    r.nnz = m;
    r.nzr = nzr;
    out = r;
}

void union_keys_to_matrices(clb_controls_s *ctl, const u64 *ka, u64 na, const u64 *kb, u64 nb, u32 n,
                            std::vector<clb_dcsr> &mats) {
    const u32 nmat = (u32)mats.size();
    UnionCounts c;
    DevArray<UnionBound> bounds(ctl, nmat);
    fill_u32(ctl, reinterpret_cast<u32 *>(bounds.ptr), 4ull * nmat, 0xFFFFFFFFu);
    union_count(ctl, ka, na, kb, nb, n, nmat, bounds.ptr, c);
    DevArray<u32> ends(ctl, 2ull * (nmat + 1));
    k_union_bounds<<<div_up(nmat + 1, 64), 64, 0, ctl->stream>>>(bounds.ptr, nmat, c.offs.ptr, c.offs.ptr + c.tiles,
                                                                 ends.ptr);
    CLB_LAUNCHED("union_bounds");
    std::vector<u32> e(2ull * (nmat + 1));
    readback(ctl, e.data(), ends.ptr, 4ull * e.size());
    std::vector<UnionDcsr> dst(nmat);
    std::vector<clb_dcsr> r(nmat);
    DevArray<UnionDcsr> table(ctl, nmat);
    bool any = false;
    try {
        for (u32 x = 0; x < nmat; ++x) {
            UnionDcsr &u = dst[x];
            u = UnionDcsr{nullptr, nullptr, nullptr, e[2 * x], e[2 * x + 1], e[2 * x + 2], e[2 * x + 3]};
            const u32 m = u.kept1 - u.kept0, nzr = u.starts1 - u.starts0;
            if (m == mats[x].nnz) continue;  // unions only add: equal size means unchanged
            r[x].nrows = r[x].ncols = n;
            r[x].cols = buffer_new(ctl, 4ull * m);
            r[x].rows = buffer_new(ctl, 4ull * nzr);
            r[x].rpt = buffer_new(ctl, 4ull * (nzr + 1ull));
            r[x].nnz = m;
            r[x].nzr = nzr;
            u.cols = u32p(r[x].cols);
            u.rows = u32p(r[x].rows);
            u.rpt = u32p(r[x].rpt);
            any = true;
        }
        if (any) {
            CLB_HIP(hipMemcpyAsync(table.ptr, dst.data(), nmat * sizeof(UnionDcsr), hipMemcpyHostToDevice,
                                   ctl->stream),
                    WRITE_BUFFER_ERROR);
            k_union_place<2><<<c.tiles, MG_WG, 0, ctl->stream>>>(ka, na, kb, nb, c.split.ptr, n, c.offs.ptr,
                                                                 UnionDcsr{}, table.ptr, nmat);
            CLB_LAUNCHED("union_place");
            sync(ctl);
        }
    } catch (...) {
        for (auto &m : r) clb_dcsr_release(&m);
        throw;
    }
    for (u32 x = 0; x < nmat; ++x)
        if (r[x].cols) mats[x] = r[x];
}

static void check_same_shape(u32 ar, u32 ac, u32 br, u32 bc) {
    // coo_matrix_addition.cpp:36-41, csr_addition.cpp:28-33
    if (ar != br || ac != bc) {
        std::string s = "Invalid matrixes size! a: " + std::to_string(ar) + " x " + std::to_string(ac) +
                        ", b: " + std::to_string(br) + " x " + std::to_string(bc);
        raise(INVALID_ARGUMENT, s);
    }
}

static clb_buffer_s *copy_buffer(clb_controls_s *ctl, const clb_buffer_s *src, u64 bytes) {
    clb_buffer_s *b = buffer_new(ctl, bytes);
    hipError_t e = hipMemcpyAsync(b->ptr, src->ptr, bytes, hipMemcpyDeviceToDevice, ctl->stream);
    if (e != hipSuccess) {
        buffer_release(b);
        check_hip(e, COPY_BUFFER_ERROR, "copy buffer");
    }
    return b;
}

}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_coo_addition(clb_controls ctl, const clb_coo *a, const clb_coo *b, clb_coo *out) {
    return run_guarded(ctl, [&] {
        check_same_shape(a->nrows, a->ncols, b->nrows, b->ncols);
        clb_coo r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz == 0 && b->nnz == 0) {  // :43-46
            *out = r;
            return;
        }
        if (a->nnz == 0 || b->nnz == 0) {  // :48-64: a copy of the filled operand
            const clb_coo *f = a->nnz ? a : b;
            r.rows = copy_buffer(ctl, f->rows, 4ull * f->nnz);
            try {
                r.cols = copy_buffer(ctl, f->cols, 4ull * f->nnz);
                sync(ctl);
            } catch (...) {
                settle(ctl);
                clb_coo_release(&r);
                throw;
            }
            r.nnz = f->nnz;
            *out = r;
            return;
        }
        DevArray<u64> ka(ctl, a->nnz), kb(ctl, b->nnz);
        pack_pairs(ctl, u32p(a->rows), u32p(a->cols), a->nnz, ka.ptr);
        pack_pairs(ctl, u32p(b->rows), u32p(b->cols), b->nnz, kb.ptr);
        r.nnz = union_keys(ctl, ka.ptr, a->nnz, kb.ptr, b->nnz, &r.rows, &r.cols);
        sync(ctl);
        *out = r;
    });
}

clb_status clb_csr_addition(clb_controls ctl, const clb_csr *a, const clb_csr *b, clb_csr *out) {
    return run_guarded(ctl, [&] {
        check_same_shape(a->nrows, a->ncols, b->nrows, b->ncols);
        clb_csr r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz == 0 && b->nnz == 0) {  // :35-38
            *out = r;
            return;
        }
        if (a->nnz == 0 || b->nnz == 0) {  // :40-55
            const clb_csr *f = a->nnz ? a : b;
            r.rpt = copy_buffer(ctl, f->rpt, 4ull * (f->nrows + 1ull));
            try {
                r.cols = copy_buffer(ctl, f->cols, 4ull * f->nnz);
                sync(ctl);
            } catch (...) {
                settle(ctl);
                clb_csr_release(&r);
                throw;
            }
            r.nnz = f->nnz;
            *out = r;
            return;
        }
        // the rows [0, nrows) hold rpt[nrows] entries; like the reference's
        // per-row kernels (csr_addition.cl), only those are merged
        u32 na = 0, nb = 0;
        readback(ctl, &na, u32p(a->rpt) + a->nrows, 4);
        readback(ctl, &nb, u32p(b->rpt) + b->nrows, 4);
        na = na < a->nnz ? na : a->nnz;
        nb = nb < b->nnz ? nb : b->nnz;
        DevArray<u64> ka(ctl, na ? na : 1), kb(ctl, nb ? nb : 1);
        expand_rows_two(
            ctl, Expand<KeyOfNonzero>{u32p(a->rpt), nullptr, 0, a->nrows, 0, na, {u32p(a->cols), 0, 0, ka.ptr}},
            Expand<KeyOfNonzero>{u32p(b->rpt), nullptr, 0, b->nrows, 0, nb, {u32p(b->cols), 0, 0, kb.ptr}});
        clb_buffer_s *rows = nullptr;
        const u32 m = union_keys(ctl, ka.ptr, na, kb.ptr, nb, &rows, &r.cols);
        try {
            r.rpt = buffer_new(ctl, 4ull * (a->nrows + 1ull));
            k_rows_lower_bound<<<div_up(a->nrows + 1ull, 256), 256, 0, ctl->stream>>>(u32p(rows), m, a->nrows,
                                                                                     u32p(r.rpt));
            CLB_LAUNCHED("rows_lower_bound");
            sync(ctl);
        } catch (...) {
            settle(ctl);
            buffer_release(rows);
            clb_csr_release(&r);
            throw;
        }
        buffer_release(rows);
        r.nnz = m;
        *out = r;
    });
}

clb_status clb_dcsr_addition(clb_controls ctl, const clb_dcsr *a, const clb_dcsr *b, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        check_same_shape(a->nrows, a->ncols, b->nrows, b->ncols);
        clb_dcsr r{};
        r.nrows = a->nrows;
        r.ncols = a->ncols;
        if (a->nnz == 0 && b->nnz == 0) {
            *out = r;
            return;
        }
        if (a->nnz == 0 || b->nnz == 0) {
            const clb_dcsr *f = a->nnz ? a : b;
            try {
                r.rpt = copy_buffer(ctl, f->rpt, 4ull * (f->nzr + 1ull));
                r.rows = copy_buffer(ctl, f->rows, 4ull * f->nzr);
                r.cols = copy_buffer(ctl, f->cols, 4ull * f->nnz);
                sync(ctl);
            } catch (...) {
                settle(ctl);
                clb_dcsr_release(&r);
                throw;
            }
            r.nnz = f->nnz;
            r.nzr = f->nzr;
            *out = r;
            return;
        }
        DevArray<u64> ka(ctl, a->nnz), kb(ctl, b->nnz);
        expand_rows_two(
            ctl, Expand<KeyOfNonzero>{u32p(a->rpt), u32p(a->rows), 0, a->nzr, 0, a->nnz, {u32p(a->cols), 0, 0, ka.ptr}},
            Expand<KeyOfNonzero>{u32p(b->rpt), u32p(b->rows), 0, b->nzr, 0, b->nnz, {u32p(b->cols), 0, 0, kb.ptr}});
        union_keys_to_dcsr(ctl, ka.ptr, a->nnz, kb.ptr, b->nnz, r);
        *out = r;
    });
}

}  // extern "C"
